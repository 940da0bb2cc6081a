// Common pieces of the registered per-thread systems.
//
// A system is a struct with the compile-time sizes of the reference's
// ProblemSolver template (SD, NCP, NSP, NISP, NE, NA, NIA; see
// SourceCodes/SingleSystem_PerThread_Interface.cuh:117) and the six user
// callbacks of the reference, as static member templates with the reference's
// argument lists (Tutorials_SingleSystem_PerThread/T1_Reference/
// Reference_SystemDefinition.cuh:5-76):
//   OdeFunction, EventFunction, ActionAfterEventDetection,
//   ActionAfterSuccessfulTimeStep, Initialization, Finalization.
// Systems that support the discrete adjoint also provide
//   OdeVJP(tid, NT, lam, X, T, cPAR, sPAR, sPARi, ACC, ACCi, gX, gP)
// setting gX = (dF/dX)^T lam and gP = (dF/dcPAR)^T lam.
// Systems whose right-hand side contains terms of the time (and the control
// parameters) alone may name them, so that the solver evaluates them once and
// reuses them (a step's end is the next step's start; with a fixed step and a
// time common to a wavefront, its lanes evaluate different times at once; with
// few instances, several lanes make one's steps and evaluate a stage's terms each):
//   NTT                                       number of such terms
//   TT_TIME_ONLY                              true when no parameter enters them
//   TimeTerms(T, cPAR, tt)                    evaluates them
//   OdeFunctionTT(tid, NT, F, X, T, tt, ...)  the right-hand side, given them
//   OdeVJPTT(tid, NT, lam, X, T, tt, ...)     its vector-Jacobian product (with
//                                             TT_TIME_ONLY and HAS_VJP only)
// with OdeFunction and OdeVJP the same functions over terms evaluated at T.
// Per-block systems take (sid, uid) for (tid, NT) and the system parameters for
// cPAR, with the argument lists of their OdeFunction and OdeVJP.
// Such a system leaves T, the time domain and the parameters in its terms
// alone after Initialization, and its callbacks change only what they are
// given for the instance (several lanes may make the same steps of one).
// Every callback is MPGOS_HD so the same definition serves the gfx950 kernels
// and the host oracle; elementary functions come from mpgos::math so both
// sides evaluate identical bits.
#pragma once

#include <type_traits>

#include "../mpgos_math.h"

namespace mpgos {
namespace systems {

// Callbacks that do nothing, for systems without events or accessories.
struct NoCallbacks {
    template <class P> MPGOS_HD static void EventFunction(int, int, P*, P, P, P*, P*, P*, P*, int*, P*, int*) {}
    template <class P> MPGOS_HD static void ActionAfterEventDetection(int, int, int, int&, P&, P&, P*, P*, P*, P*, int*, P*, int*) {}
    template <class P> MPGOS_HD static void ActionAfterSuccessfulTimeStep(int, int, int&, P&, P&, P*, P*, P*, P*, int*, P*, int*) {}
    template <class P> MPGOS_HD static void Initialization(int, int, int&, P&, P&, P*, P*, P*, P*, int*, P*, int*) {}
    template <class P> MPGOS_HD static void Finalization(int, int, int&, P&, P&, P*, P*, P*, P*, int*, P*, int*) {}
};

// The same for per-block systems (callback argument lists in pb_ring.h).
struct PBNoCallbacks {
#define MPGOS_PB_ARGS P*, P*, P*, int*, P*, int*, P*, int*
    template <class P> MPGOS_HD static void EventFunction(int, int, P*, P, P, P*, P*, MPGOS_PB_ARGS) {}
    template <class P> MPGOS_HD static void ActionAfterEventDetection(int, int, int, int&, P&, P&, P*, P*, MPGOS_PB_ARGS) {}
    template <class P> MPGOS_HD static void ActionAfterSuccessfulTimeStep(int, int, int&, P&, P&, P*, P*, MPGOS_PB_ARGS) {}
    template <class P> MPGOS_HD static void Finalization(int, int, int&, P&, P&, P*, P*, MPGOS_PB_ARGS) {}
#undef MPGOS_PB_ARGS
};

// Whether a system leaves ActionAfterSuccessfulTimeStep to Base (NoCallbacks or
// PBNoCallbacks).
template <class Sys, class Base> constexpr bool no_step_action()
{
    if constexpr (std::is_base_of<Base, Sys>::value)
        return &Sys::template ActionAfterSuccessfulTimeStep<double> == &Base::template ActionAfterSuccessfulTimeStep<double>;
    else return false;
}

// Number of time terms of a system (0 for systems that name none), and whether
// they depend on the time alone.
template <class Sys, class = void> struct TimeTermsOf {
    static constexpr int n = 0;
    static constexpr bool timeOnly = false;
};
template <class Sys> struct TimeTermsOf<Sys, decltype((void)Sys::NTT)> {
    static constexpr int n = Sys::NTT;
    static constexpr bool timeOnly = Sys::TT_TIME_ONLY;
};

} // namespace systems
} // namespace mpgos
