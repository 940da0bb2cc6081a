// Registry of the systems compiled into libmpgos.so.  Each system's kernels
// are instantiated in its own translation unit (sys_<name>.hip) so the build
// parallelises; the C ABI (capi.hip) selects a factory by name.
#pragma once

#include "pb_engine.h"
#include "pt_engine.h"

#define MPGOS_PT_FACTORY(NAME, SYS)                                                   \
    ::mpgos::pt::SolverBase* make_pt_##NAME(int precision)                            \
    {                                                                                 \
        switch (precision) {                                                          \
        case MPGOS_DOUBLE: return new ::mpgos::pt::Solver<SYS, double, false>();      \
        case MPGOS_FLOAT: return new ::mpgos::pt::Solver<SYS, float, false>();        \
        case MPGOS_FLOAT_KAHAN: return new ::mpgos::pt::Solver<SYS, float, true>();   \
        default: return nullptr;                                                      \
        }                                                                             \
    }

#define MPGOS_PB_FACTORY(NAME, SYS)                                                   \
    ::mpgos::pb::SolverBase* make_pb_##NAME(int precision)                            \
    {                                                                                 \
        switch (precision) {                                                          \
        case MPGOS_DOUBLE: return new ::mpgos::pb::Solver<SYS, double>();             \
        case MPGOS_FLOAT: return new ::mpgos::pb::Solver<SYS, float>();               \
        case MPGOS_FLOAT_KAHAN: return new ::mpgos::pb::Solver<SYS, float, true>();   \
        default: return nullptr;                                                      \
        }                                                                             \
    }

// The kernels of a per-thread system that are held to few registers:
// MPGOS_PT_NARROW_KERNELS in an object of their own (sys_narrow_<name>.hip),
// declared with MPGOS_PT_NARROW_EXTERN where the factory stands.
#define MPGOS_PT_NARROW(EXTERN, SYS)                                                                                          \
    EXTERN template auto narrow_kernel<SYS, double, false>(int, int, int) -> void (*)(Args<SYS, double, double>);              \
    EXTERN template auto narrow_kernel<SYS, float, false>(int, int, int) -> void (*)(Args<SYS, float, float>);                 \
    EXTERN template auto narrow_kernel<SYS, float, true>(int, int, int) -> void (*)(Args<SYS, float, double>);
#define MPGOS_PT_NARROW_KERNELS(SYS) MPGOS_PT_NARROW(, SYS)
#define MPGOS_PT_NARROW_EXTERN(SYS) MPGOS_PT_NARROW(extern, SYS)

// The lane-per-pair kernels of a per-block system: MPGOS_PB_LANE_KERNELS in an
// object of their own (sys_lane_pb_<name>.hip, default flags), declared with
// MPGOS_PB_LANE_EXTERN where the factory stands.
#define MPGOS_PB_LANE(EXTERN, SYS)                                                                                      \
    EXTERN template void launch_lane<SYS, double, false>(int, bool, int, int, size_t, hipStream_t, const Args<SYS, double>&); \
    EXTERN template void launch_lane<SYS, float, false>(int, bool, int, int, size_t, hipStream_t, const Args<SYS, float>&);   \
    EXTERN template void launch_lane<SYS, float, true>(int, bool, int, int, size_t, hipStream_t, const Args<SYS, float, double>&); \
    EXTERN template void launch_lane_record<SYS>(int, bool, int, int, size_t, hipStream_t, const Args<SYS, double>&);         \
    EXTERN template void launch_lane_reverse<SYS>(int, int, int, size_t, hipStream_t, const Args<SYS, double>&, const AdjArgs<SYS>&);
#define MPGOS_PB_LANE_KERNELS(SYS) MPGOS_PB_LANE(, SYS)
#define MPGOS_PB_LANE_EXTERN(SYS) MPGOS_PB_LANE(extern, SYS)

namespace mpgos {
namespace pb {
struct Registration {
    const char* name;
    SolverBase* (*make)(int precision);
};
SolverBase* make_pb_ring_duffing(int precision);
SolverBase* make_pb_ring_dw(int precision);
SolverBase* make_pb_pb_linear(int precision);
SolverBase* make_pb_ring_duffing_q(int precision);
} // namespace pb

namespace pt {

struct Registration {
    const char* name;
    SolverBase* (*make)(int precision);
};

SolverBase* make_pt_duffing(int precision);
SolverBase* make_pt_duffing_q(int precision);
SolverBase* make_pt_duffing_eps(int precision);
SolverBase* make_pt_duffing_dw(int precision);
SolverBase* make_pt_relief_valve(int precision);
SolverBase* make_pt_keller_miksis(int precision);
SolverBase* make_pt_keller_miksis_max(int precision);
SolverBase* make_pt_lorenz(int precision);
SolverBase* make_pt_affine2(int precision);

} // namespace pt
} // namespace mpgos
