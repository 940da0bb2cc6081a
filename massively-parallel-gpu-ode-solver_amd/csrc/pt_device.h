// Per-thread solver for gfx950: one lane integrates one instance.
//
// Semantics follow the reference kernel SingleSystem_PerThread
// (SourceCodes/SingleSystem_PerThread_Solver.cuh:11-437) step for step:
// prologue (loads, Initialization, first event evaluation, first dense store),
// the loop  clip-to-end -> stepper -> controller -> event step control ->
// [accept: t,x update, ActionAfterSuccessfulTimeStep, event detection and
// ActionAfterEventDetection, event re-evaluation, dense output, termination],
// then Finalization and write-back.  The numerics are
//   RK4     SingleSystem_PerThread_ExplicitRungeKutta_Steppers.cuh:6-117
//   RKCK45  SingleSystem_PerThread_ExplicitRungeKutta_Steppers.cuh:121-290
//   controllers  SingleSystem_PerThread_ExplicitRungeKutta_ErrorControllers.cuh:5-86
//   event step control  SingleSystem_PerThread_EventHandling.cuh:5-45
//   dense output  SingleSystem_PerThread_DenseOutput.cuh:5-58
// with every multiply-add of the stage combinations written as an explicit
// fused multiply-add (the form a contracting compiler gives the reference's
// expressions) and the rest compiled with -ffp-contract=off, so the FP64 result
// is reproducible bit for bit by the host oracle.
//
// Design for MI355X (not present in the reference):
//  * instance state lives in VGPRs; SoA HBM layout (index tid + c*NT) keeps
//    every load/store of a wavefront contiguous;
//  * tolerances and solver options arrive by value in the kernel argument
//    block, so they sit in SGPRs; shared parameters are staged in LDS when
//    PreferSharedMemory is on (the reference default);
//  * device printf is replaced by per-instance status bits and counters;
//  * a persistent form pulls instances from a device work queue and refills
//    lanes whose instance finished, found with a wavefront ballot;
//  * FLOAT_KAHAN mode: FP32 state and stages, compensated accumulation of
//    time and state, FP64 error norm, controller and event step control.
#pragma once

#include <hip/hip_runtime.h>
#include <cstddef>
#include <type_traits>

#include "mpgos_math.h"
#include "mpgos.h"
#include "systems/system_base.h"

namespace mpgos {
namespace pt {

using systems::TimeTermsOf;

constexpr int kMaxBlock = 512;
constexpr int kMaxWaves = kMaxBlock / 64;

template <int N> struct Pos { static constexpr int value = N > 0 ? N : 1; };

// Kernel argument block.  CP is the precision of the step-size control.
template <class Sys, class P, class CP>
struct Args {
    static constexpr int SD = Sys::SD;
    static constexpr int NE = Sys::NE;
    // SoA buffers (reference layout)
    P* TD; P* X; P* T; P* cPAR; P* sPAR; int* sPARi; P* ACC; int* ACCi;
    int* DOidx; P* DOt; P* DOx;
    // per-instance outputs
    long long* nacc; long long* nrej; int* status; int* nev; P* evlog; int* evlogidx;
    unsigned int* queue;      // persistent form: [0] = next list entry past the solo ones; [1] = suspended count
                              // of a slice; [2] = next solo entry
    // time-sliced solve: the instances to work on are list[0, listLen) (the
    // identity 0..nActive-1 when list is null); with slice > 0 an instance
    // that has attempted `slice` steps in this launch is suspended (in the
    // relaunch form's last launch, listOut null, it stops there with
    // MPGOS_STATUS_STEP_BUDGET instead): its lane
    // state goes to its record saved[id * W .. id * W + W) (W 32-bit words,
    // 16-byte aligned), phase[id] = 1, and its id is appended to listOut
    // (count in queue[1]); phase[id] = 2 once finished
    const int* list; int* listOut; uint32_t* saved; int* phase;
    int listLen, slice;
    const unsigned* listLenDev;   // relaunch form: the list length is the previous launch's count (device)
    unsigned* outCount;           // relaunch form: count of this launch's suspended instances (else queue[1])
    float* sortKey;               // sorted form's pilot launch: estimated remaining attempted steps of each
                                  // suspended instance, at its slot of listOut
    int NT, nActive, NDO, evcap, preferShared;
    int doFreq;
    int roundSteps;           // persistent form: attempted steps between compactions
    int octets;               // sorted form's last launch: workgroups [0, octets) give an instance 8 lanes
    int solo;                 // persistent form: list entries [0, solo) run one per workgroup (workgroups [0, solo))
    CP dt0, dtmax, dtmin, grow, shrink;
    P doMinDt;
    CP rtol[Pos<SD>::value], atol[Pos<SD>::value];
    P etol[Pos<NE>::value];
    int edir[Pos<NE>::value];
};

// The kernel's argument block read afresh from the kernel-argument segment,
// through a pointer the compiler cannot see through.  Used on the rare paths
// (finishing or suspending an instance, dense-output and event-log stores):
// the fields they read are then loaded where they are used instead of being
// held in SGPRs, and spilled to VGPR lanes, across the whole step loop.  Valid
// only in kernels whose argument block begins with the Args: solve_kernel and
// the adjoint kernels (whose AdjArgs start with it, asserted there).
template <class A>
__device__ __forceinline__ const A& kernel_args()
{
    typedef __attribute__((address_space(4))) const A* KP;
    KP p = (KP)__builtin_amdgcn_kernarg_segment_ptr();
    asm volatile("" : "+s"(p));
    return *(const A*)p;
}

// The same for bodies with run_common_time, where the compiler joins control
// flow so that the pointer reaches the statement above in vector registers,
// which it cannot copy back: hidden there and read back explicitly.
template <class A>
__device__ __forceinline__ const A& kernel_args_joined()
{
    typedef __attribute__((address_space(4))) const A* KP;
    const uint64_t b = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
    uint32_t lo = (uint32_t)b, hi = (uint32_t)(b >> 32);
    asm volatile("" : "+v"(lo), "+v"(hi));
    lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)lo);
    hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)hi);
    return *(const A*)(KP)(((uint64_t)hi << 32) | lo);
}

// Value that lane `src` of the wavefront holds, in scalar registers.
__device__ __forceinline__ float lane_value(float v, int src)
{
    return __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, v), src));
}
__device__ __forceinline__ double lane_value(double v, int src)
{
    const uint64_t b = math::bits(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)b, src);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(b >> 32), src);
    return math::from_bits(((uint64_t)hi << 32) | lo);
}

// t advanced by h as often as the lane's place in the wavefront says: lane l
// of a full wavefront l / 2 times (l / 3 times in the compensated form), one
// rounded addition after the other as the step loop makes them.  The lanes
// still to advance are always the highest ones, so every addition runs under
// an execution mask two (three) lanes shorter than the last: two instructions
// per step instead of a loop's compare, select and branch.
__device__ __forceinline__ void advance_by_lane(double& t, double&, double h)
{
    uint64_t save;
    asm volatile("s_mov_b64 %1, exec\n"
                 "s_mov_b64 exec, -1\n"
                 ".rept 31\n"
                 "s_lshl_b64 exec, exec, 2\n"
                 "v_add_f64 %0, %0, %2\n"
                 ".endr\n"
                 "s_mov_b64 exec, %1"
                 : "+v"(t), "=&s"(save) : "v"(h) : "scc");
}
__device__ __forceinline__ void advance_by_lane(float& t, float&, float h)
{
    uint64_t save;
    asm volatile("s_mov_b64 %1, exec\n"
                 "s_mov_b64 exec, -1\n"
                 ".rept 31\n"
                 "s_lshl_b64 exec, exec, 2\n"
                 "v_add_f32 %0, %0, %2\n"
                 ".endr\n"
                 "s_mov_b64 exec, %1"
                 : "+v"(t), "=&s"(save) : "v"(h) : "scc");
}
// Kahan form: y = h - c, s = t + y, c = (s - t) - y, t = s
__device__ __forceinline__ void advance_by_lane_kahan(float& t, float& c, float h)
{
    uint64_t save;
    float y, d;
    asm volatile("s_mov_b64 %2, exec\n"
                 "s_mov_b64 exec, -1\n"
                 ".rept 21\n"
                 "s_lshl_b64 exec, exec, 3\n"
                 "v_sub_f32 %3, %5, %1\n"
                 "v_add_f32 %4, %0, %3\n"
                 "v_sub_f32 %1, %4, %0\n"
                 "v_sub_f32 %1, %1, %3\n"
                 "v_mov_b32 %0, %4\n"
                 ".endr\n"
                 "s_mov_b64 exec, %2"
                 : "+v"(t), "+v"(c), "=&s"(save), "=&v"(y), "=&v"(d) : "v"(h) : "scc");
}

// ---- several lanes per instance
// With fewer instances than keep the card busy, GROUP (4 or 8) neighbouring
// lanes hold one instance: all of them make its steps, on the same values, and
// the time terms of a Cash-Karp step's six stages, whose times are known when
// the step starts, are evaluated one stage per lane (two with 4 lanes) and
// exchanged within the group, in one or two evaluations per step instead of
// five.  The values are those that a single lane would compute.  A lone
// wavefront is bound by the instructions of its step; the step of a double-well
// Duffing oscillator has 455 FP64 instructions with one lane and 345 with 8.
// 20000 uneven Duffing instances 116 -> 67 ms, 10007 Cash-Karp adjoints 3.76 ->
// 2.82 ms, 4000 double wells 127 -> 92 us.
template <int GROUP> __host__ __device__ constexpr int group_evals() { return GROUP > 1 ? (6 + GROUP - 1) / GROUP : 1; }

// Word that lane J of the lane's group of GROUP holds.
template <int GROUP, int J>
__device__ __forceinline__ int group_word(int v)
{
    constexpr int j = J & 3, quad = j | j << 2 | j << 4 | j << 6;
    int q = __builtin_amdgcn_update_dpp(0, v, quad, 0xf, 0xf, true);            // lane j of each 4 lanes
    if (GROUP == 8)                                                             // the other 4 take it mirrored
        q = __builtin_amdgcn_update_dpp(q, q, 0x141, 0xf, J < 4 ? 0xa : 0x5, false);
    return q;
}
template <int GROUP, int J> __device__ __forceinline__ float group_value(float v)
{
    return __builtin_bit_cast(float, group_word<GROUP, J>(__builtin_bit_cast(int, v)));
}
template <int GROUP, int J> __device__ __forceinline__ double group_value(double v)
{
    const uint64_t b = math::bits(v);
    const uint32_t lo = (uint32_t)group_word<GROUP, J>((int)(uint32_t)b), hi = (uint32_t)group_word<GROUP, J>((int)(uint32_t)(b >> 32));
    return math::from_bits(((uint64_t)hi << 32) | lo);
}
// The node c of the stage whose terms the lane evaluates in evaluation e: its
// time is fma(h, c, t), as in the stepper (t itself for c = 0, t + h for c = 1).
template <int GROUP, class P>
__device__ __forceinline__ P stage_node(int e)
{
    const int j = e * GROUP + (int)(threadIdx.x & (GROUP - 1));
    P c = P(7.0 / 8.0);
    c = j == 0 ? P(0) : c;
    c = j == 1 ? P(1.0 / 5.0) : c;
    c = j == 2 ? P(3.0 / 10.0) : c;
    c = j == 3 ? P(3.0 / 5.0) : c;
    return j == 4 ? P(1) : c;
}

// wavefronts per SIMD from which a kernel is short of registers (128 and 64)
constexpr int kNarrowWaves = 4;

// Whether a kernel for WPE wavefronts per SIMD has the way for usual steps beside
// the general one (Lane::step).  With 64 registers and compensated steps the two
// together spill far more than the general way does: 65536 Lorenz instances
// 53 us without the short way, 92 us with it; 65536 in the other forms and other
// systems 1.1 to 1.4 times as long with it.  In the others it pays in most (FP64
// without it: 0.9 to 1.4 times as long with 64 registers, to 1.5 times with 128).
template <bool KAHAN, int WPE>
constexpr bool short_way() { return !(KAHAN && WPE >= 2 * kNarrowWaves); }

// What a step reads of the argument block.  The control limits and tolerances
// are put into vector registers once, before the step loop: in scalar registers
// they and the step's constants exceed the 102 there are, and the compiler
// reloads them from memory or rebuilds constants inside the loop (a lone
// wavefront pays for every such instruction and waits for every load).  Kernels
// that are held to few registers (wide = false) leave them to the compiler: there
// they and what they push out are spilled at every step (64 registers, 65536
// Duffing oscillators: 0.75 ms so, 1.04 ms with them pinned).
template <class Sys, class P, class CP>
struct StepArgs {
    static constexpr int SD = Sys::SD, NE = Sys::NE;
    CP dt0, dtmin, dtmax, grow, shrink;
    CP least;                   // steps above it, and tolerances as they should be: the short way through step()
    CP rtol[SD], atol[SD];
    P etol[Pos<NE>::value];
    int edir[Pos<NE>::value];
    int NT, NDO, doFreq;
    P node[2];                  // several lanes per instance: stage_node of this lane

    template <class T> static __device__ __forceinline__ T in_register(T v)
    {
        asm volatile("" : "+v"(v));
        return v;
    }
    __device__ __forceinline__ StepArgs(const Args<Sys, P, CP>& a, bool adaptive, bool wide = true)
    {
        auto pin = [&](auto v) { return wide ? in_register(v) : v; };
        dt0 = a.dt0; NT = a.NT; NDO = a.NDO; doFreq = a.doFreq;
        if (adaptive) {
            dtmin = pin(a.dtmin); dtmax = pin(a.dtmax); grow = pin(a.grow); shrink = pin(a.shrink);
            CP l = a.dtmin * CP(1.01);
#pragma unroll
            for (int i = 0; i < NE; i++)
                if (!(a.etol[i] >= P(0))) l = CP(__builtin_huge_val());
            // the maximum in step() drops a NaN tolerance, which no error is
            // below (a NaN rtol alone leaves tol = atol)
#pragma unroll
            for (int i = 0; i < SD; i++)
                if (a.atol[i] != a.atol[i]) l = CP(__builtin_huge_val());
            least = pin(l);
#pragma unroll
            for (int i = 0; i < SD; i++) { rtol[i] = pin(a.rtol[i]); atol[i] = pin(a.atol[i]); }
        } else {
            dtmin = a.dtmin;
        }
#pragma unroll
        for (int i = 0; i < NE; i++) {
            etol[i] = pin(a.etol[i]);
            edir[i] = a.edir[i];
        }
    }
    template <int GROUP> __device__ __forceinline__ void set_nodes()
    {
#pragma unroll
        for (int e = 0; e < group_evals<GROUP>(); e++) node[e] = in_register(stage_node<GROUP, P>(e));
    }
};

template <class Sys, class P, bool KAHAN, int ALG>
struct Lane {
    using CP = typename std::conditional<KAHAN, double, P>::type;
    using A = Args<Sys, P, CP>;
    using C = StepArgs<Sys, P, CP>;
    using Sys_t = Sys;
    static constexpr bool kKahan = KAHAN;
    static constexpr int SD = Sys::SD, NCP = Sys::NCP, NE = Sys::NE, NA = Sys::NA, NIA = Sys::NIA;
    static constexpr int NTT = TimeTermsOf<Sys>::n;
    // fixed steps whose time terms a wavefront can share (run_common_time)
    static constexpr bool kCommonTime = ALG == MPGOS_RK4 && NE == 0 && TimeTermsOf<Sys>::timeOnly;

    P TD[2];
    P X[SD];
    P Xc[KAHAN ? SD : 1];                 // Kahan compensation of the state
    P cPAR[Pos<NCP>::value];
    P ACC[Pos<NA>::value];
    int ACCi[Pos<NIA>::value];
    P EF[Pos<NE>::value];
    P t;
    P tc;                                 // Kahan compensation of the time
    CP dt, newDt;
    P doT;
    int doIdx, skipped, term, udt;
    int nacc, nrej, status, nev;
    int tid;
    int left;                             // time-sliced solve: attempted steps left in this launch

    // whole lane state to and from HBM (time-sliced solve), bit for bit
    // one 16-byte aligned record per instance (rare: once per slice), moved
    // with 16-byte accesses from one base address per lane
    static constexpr int kSavedWords = (int)((sizeof(Lane) / 4 + 3) & ~(size_t)3);
    __device__ __forceinline__ void save(const A& a) const
    {
        uint32_t w[kSavedWords] = {};
        __builtin_memcpy(w, this, sizeof(Lane));
        uint4* dst = reinterpret_cast<uint4*>(a.saved + (size_t)tid * kSavedWords);
#pragma unroll
        for (int i = 0; i < kSavedWords / 4; i++) dst[i] = make_uint4(w[4 * i], w[4 * i + 1], w[4 * i + 2], w[4 * i + 3]);
    }
    __device__ __forceinline__ void restore(const A& a, int id)
    {
        uint32_t w[kSavedWords];
        const uint4* src = reinterpret_cast<const uint4*>(a.saved + (size_t)id * kSavedWords);
#pragma unroll
        for (int i = 0; i < kSavedWords / 4; i++) {
            const uint4 v = src[i];
            w[4 * i] = v.x; w[4 * i + 1] = v.y; w[4 * i + 2] = v.z; w[4 * i + 3] = v.w;
        }
        __builtin_memcpy(this, w, sizeof(Lane));
    }
    // the instance's first launch initialises it, later launches resume it
    __device__ __forceinline__ void begin(const A& a, int id, P* sPAR, int* sPARi)
    {
        if (a.phase[id] == 1) restore(a, id);
        else load(a, id, sPAR, sPARi);
        left = a.slice;
    }
    // after a step: true when the lane is to be released (finished, or its
    // slice budget spent); release() then finishes or suspends it
    __device__ __forceinline__ bool stop() { return term || --left <= 0; }
    __device__ __forceinline__ void release(const A& a, P* sPAR, int* sPARi)
    {
        if (term) {
            finish(a, sPAR, sPARi);
            a.phase[tid] = 2;
            return;
        }
        if (!a.listOut) {   // the relaunch form's last launch: no later launch resumes the instance
            status |= MPGOS_STATUS_STEP_BUDGET;
            finish(a, sPAR, sPARi);
            a.phase[tid] = 2;
            return;
        }
        save(a);
        a.phase[tid] = 1;
        const unsigned slot = atomicAdd(a.outCount ? a.outCount : &a.queue[1], 1u);
        a.listOut[slot] = tid;
        if (a.sortKey) {
            // remaining attempts at the rate so far: attempts * (TD1 - t) / (t - TD0)
            const double done = (double)t - (double)TD[0], rest = (double)TD[1] - (double)t;
            const double att = (double)(nacc + nrej);
            a.sortKey[slot] = done > 0.0 ? (float)__builtin_fmin(att * rest / done, 3.0e38) : 3.0e38f;
        }
    }

    // ------------------------------------------------------------ load / prologue
    // a lane without an instance that accompanies its wavefront
    __device__ __forceinline__ void idle()
    {
        tid = 0;
        TD[0] = TD[1] = P(0);
#pragma unroll
        for (int i = 0; i < SD; i++) { X[i] = P(0); if (KAHAN) Xc[i] = P(0); }
#pragma unroll
        for (int i = 0; i < NCP; i++) cPAR[i] = P(0);
        t = tc = doT = P(0);
        dt = newDt = CP(0);
        doIdx = 0x7fffffff;     // no dense output
        skipped = udt = nacc = nrej = status = nev = 0;
        term = 1;
    }
    __device__ __forceinline__ void load(const A& a, int id, P* sPAR, int* sPARi)
    {
        tid = id;
        const int NT = a.NT;
#pragma unroll
        for (int i = 0; i < 2; i++) TD[i] = a.TD[tid + i * NT];
#pragma unroll
        for (int i = 0; i < SD; i++) { X[i] = a.X[tid + i * NT]; if (KAHAN) Xc[i] = P(0); }
#pragma unroll
        for (int i = 0; i < NCP; i++) cPAR[i] = a.cPAR[tid + i * NT];
#pragma unroll
        for (int i = 0; i < NA; i++) ACC[i] = a.ACC[tid + i * NT];
#pragma unroll
        for (int i = 0; i < NIA; i++) ACCi[i] = a.ACCi[tid + i * NT];
        t = a.T[tid];
        tc = P(0);
        dt = a.dt0;
        newDt = a.dt0;
        doIdx = a.DOidx[tid];
        skipped = 0;
        term = 0;
        udt = 0;
        nacc = 0; nrej = 0; status = 0; nev = 0;
        doT = P(0);

        // PT-SOL:148-193
        P dtP = (P)dt;
        Sys::template Initialization<P>(tid, NT, doIdx, t, dtP, TD, X, cPAR, sPAR, sPARi, ACC, ACCi);
        dt = (CP)dtP;
        if (NE > 0)
            Sys::template EventFunction<P>(tid, NT, EF, t, dtP, TD, X, cPAR, sPAR, sPARi, ACC, ACCi);
        if (a.NDO > 0 && doIdx < a.NDO) store_dense(a);
    }

    __device__ __forceinline__ void store_dense(const A& a)
    {
        // PT-DO:5-37 (store branch)
        const int NT = a.NT;
        a.DOt[tid + doIdx * NT] = t;
        int k = tid + doIdx * NT * SD;
#pragma unroll
        for (int i = 0; i < SD; i++) { a.DOx[k] = X[i]; k += NT; }
        doIdx++;
        skipped = 0;
        doT = mpgos_fmin(t + a.doMinDt, TD[1]);
    }

    // min and max of values that are results of arithmetic (never signalling
    // NaNs): the instruction itself, where the builtin first canonicalises each
    // operand whose origin it does not see (a v_max per operand).  _abs: of the
    // magnitudes.
#define MPGOS_MINMAX(name, ins)                                                                                                  \
    static __device__ __forceinline__ double name(double x, double y)                                                           \
    { double r; asm(ins "_f64 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y)); return r; }                                              \
    static __device__ __forceinline__ float name(float x, float y)                                                              \
    { float r; asm(ins "_f32 %0, %1, %2" : "=v"(r) : "v"(x), "v"(y)); return r; }
    MPGOS_MINMAX(lane_min, "v_min")
    MPGOS_MINMAX(lane_max, "v_max")
#undef MPGOS_MINMAX
    static __device__ __forceinline__ double lane_max_abs(double x, double y)
    { double r; asm("v_max_f64 %0, |%1|, |%2|" : "=v"(r) : "v"(x), "v"(y)); return r; }
    static __device__ __forceinline__ float lane_max_abs(float x, float y)
    { float r; asm("v_max_f32 %0, |%1|, |%2|" : "=v"(r) : "v"(x), "v"(y)); return r; }

    static __device__ __forceinline__ double mpgos_fmin(double x, double y) { return __builtin_fmin(x, y); }
    static __device__ __forceinline__ float mpgos_fmin(float x, float y) { return __builtin_fminf(x, y); }
    static __device__ __forceinline__ double mpgos_fmax(double x, double y) { return __builtin_fmax(x, y); }
    static __device__ __forceinline__ float mpgos_fmax(float x, float y) { return __builtin_fmaxf(x, y); }

    // ------------------------------------------------------------ steppers
    // terms of the right-hand side that depend on the time (and parameters)
    __device__ __forceinline__ void time_terms(P T, P* tt)
    {
        if constexpr (NTT > 0) Sys::template TimeTerms<P>(T, cPAR, tt);
    }
    // right-hand side at (Y, T) with the time terms tt at T
    __device__ __forceinline__ void ode(int NT, P* F, P* Y, P T, const P* tt, P* sPAR, int* sPARi)
    {
        if constexpr (NTT > 0) Sys::template OdeFunctionTT<P>(tid, NT, F, Y, T, tt, cPAR, sPAR, sPARi, ACC, ACCi);
        else Sys::template OdeFunction<P>(tid, NT, F, Y, T, cPAR, sPAR, sPARi, ACC, ACCi);
    }

    // RK4: PT-STP:6-117, with the time terms at t, t + h/2 and t + h.  Returns
    // next state in `nx`; in Kahan mode `inc` gets the increment
    // dt/6 (k1 + 2k2 + 2k3 + k4).
    __device__ __forceinline__ void rk4(const C& a, P h, P* nx, P* inc, P* sPAR, int* sPARi, const P* tt1, const P* ttm,
                                        const P* tt4)
    {
        using math::fma;
        P Xs[SD], k[SD];
        const P dTp2 = P(0.5) * h;
        const P dTp6 = P(1.0 / 6.0) * h;
        ode(a.NT, nx, X, t, tt1, sPAR, sPARi);
        P T = t + dTp2;
#pragma unroll
        for (int i = 0; i < SD; i++) Xs[i] = fma(nx[i], dTp2, X[i]);
        ode(a.NT, k, Xs, T, ttm, sPAR, sPARi);
#pragma unroll
        for (int i = 0; i < SD; i++) { nx[i] = fma(P(2.0), k[i], nx[i]); Xs[i] = fma(k[i], dTp2, X[i]); }
        ode(a.NT, k, Xs, T, ttm, sPAR, sPARi);
        T = t + h;
#pragma unroll
        for (int i = 0; i < SD; i++) { nx[i] = fma(P(2.0), k[i], nx[i]); Xs[i] = fma(k[i], h, X[i]); }
        ode(a.NT, k, Xs, T, tt4, sPAR, sPARi);
#pragma unroll
        for (int i = 0; i < SD; i++) {
            const P s = nx[i] + k[i];
            if (KAHAN) { inc[i] = dTp6 * s; nx[i] = X[i] + inc[i]; }
            else nx[i] = fma(dTp6, s, X[i]);
        }
    }

    // RKCK45: PT-STP:121-290.  err[] in control precision.  tt: the time terms
    // at t; tt5 receives those at t + h.
    template <int GROUP>
    __device__ __forceinline__ void rkck45(const C& a, P h, P* nx, P* inc, CP* err, P* sPAR, int* sPARi, const P* tt, P* tt5)
    {
        using math::fma;
        P Xs[SD], k1[SD], k2[SD], k3[SD], k4[SD], k5[SD], k6[SD];
        P ts[Pos<NTT>::value];
        P all[group_evals<GROUP>()][Pos<NTT>::value];
        if constexpr (GROUP > 1) {
#pragma unroll
            for (int e = 0; e < group_evals<GROUP>(); e++) time_terms(fma(h, a.node[e], t), all[e]);
        }
        // the time terms of stage J, at T
        auto terms = [&](auto J, P T, P* r) {
            if constexpr (GROUP > 1) {
#pragma unroll
                for (int i = 0; i < NTT; i++) r[i] = group_value<GROUP, J.value % GROUP>(all[J.value / GROUP][i]);
            } else {
                time_terms(T, r);
            }
        };
        if constexpr (GROUP > 1) {
            terms(std::integral_constant<int, 0>{}, t, ts);
            ode(a.NT, k1, X, t, ts, sPAR, sPARi);
        } else {
            ode(a.NT, k1, X, t, tt, sPAR, sPARi);
        }

        P T = fma(h, P(1.0 / 5.0), t);
#pragma unroll
        for (int i = 0; i < SD; i++) Xs[i] = fma(h, P(1.0 / 5.0) * k1[i], X[i]);
        terms(std::integral_constant<int, 1>{}, T, ts);
        ode(a.NT, k2, Xs, T, ts, sPAR, sPARi);

        T = fma(h, P(3.0 / 10.0), t);
#pragma unroll
        for (int i = 0; i < SD; i++) {
            P s = P(3.0 / 40.0) * k1[i];
            s = fma(P(9.0 / 40.0), k2[i], s);
            Xs[i] = fma(h, s, X[i]);
        }
        terms(std::integral_constant<int, 2>{}, T, ts);
        ode(a.NT, k3, Xs, T, ts, sPAR, sPARi);

        T = fma(h, P(3.0 / 5.0), t);
#pragma unroll
        for (int i = 0; i < SD; i++) {
            P s = P(3.0 / 10.0) * k1[i];
            s = fma(P(-9.0 / 10.0), k2[i], s);
            s = fma(P(6.0 / 5.0), k3[i], s);
            Xs[i] = fma(h, s, X[i]);
        }
        terms(std::integral_constant<int, 3>{}, T, ts);
        ode(a.NT, k4, Xs, T, ts, sPAR, sPARi);

        T = t + h;
#pragma unroll
        for (int i = 0; i < SD; i++) {
            P s = P(-11.0 / 54.0) * k1[i];
            s = fma(P(5.0 / 2.0), k2[i], s);
            s = fma(P(-70.0 / 27.0), k3[i], s);
            s = fma(P(35.0 / 27.0), k4[i], s);
            Xs[i] = fma(h, s, X[i]);
        }
        terms(std::integral_constant<int, 4>{}, T, tt5);
        ode(a.NT, k5, Xs, T, tt5, sPAR, sPARi);

        T = fma(h, P(7.0 / 8.0), t);
#pragma unroll
        for (int i = 0; i < SD; i++) {
            P s = P(1631.0 / 55296.0) * k1[i];
            s = fma(P(175.0 / 512.0), k2[i], s);
            s = fma(P(575.0 / 13824.0), k3[i], s);
            s = fma(P(44275.0 / 110592.0), k4[i], s);
            s = fma(P(253.0 / 4096.0), k5[i], s);
            Xs[i] = fma(h, s, X[i]);
        }
        terms(std::integral_constant<int, 5>{}, T, ts);
        ode(a.NT, k6, Xs, T, ts, sPAR, sPARi);

#pragma unroll
        for (int i = 0; i < SD; i++) {
            P s = P(37.0 / 378.0) * k1[i];
            s = fma(P(250.0 / 621.0), k3[i], s);
            s = fma(P(125.0 / 594.0), k4[i], s);
            s = fma(P(512.0 / 1771.0), k6[i], s);
            if (KAHAN) { inc[i] = h * s; nx[i] = X[i] + inc[i]; }
            else nx[i] = fma(h, s, X[i]);

            if (KAHAN) {
                // FP64 error norm over the FP32 stages
                double e = (37.0 / 378.0 - 2825.0 / 27648.0) * (double)k1[i];
                e = math::fma(250.0 / 621.0 - 18575.0 / 48384.0, (double)k3[i], e);
                e = math::fma(125.0 / 594.0 - 13525.0 / 55296.0, (double)k4[i], e);
                e = math::fma(0.0 - 277.0 / 14336.0, (double)k5[i], e);
                e = math::fma(512.0 / 1771.0 - 1.0 / 4.0, (double)k6[i], e);
                err[i] = math::fma((double)h, math::fabs(e), 1e-18);
            } else {
                P e = P(37.0 / 378.0 - 2825.0 / 27648.0) * k1[i];
                e = fma(P(250.0 / 621.0 - 18575.0 / 48384.0), k3[i], e);
                e = fma(P(125.0 / 594.0 - 13525.0 / 55296.0), k4[i], e);
                e = fma(P(0.0 - 277.0 / 14336.0), k5[i], e);
                e = fma(P(512.0 / 1771.0 - 1.0 / 4.0), k6[i], e);
                if (std::is_same<P, double>::value) err[i] = (CP)math::fma((double)h, (double)math::fabs(e), 1e-18);
                else err[i] = (CP)((double)(h * math::fabs(e)) + 1e-18);   // float*float, then + double literal
            }
        }
    }

    // ------------------------------------------------------------ controllers
    __device__ __forceinline__ void next_step_size(const C& a, CP fac)
    {
        fac = lane_min(fac, a.grow);
        fac = lane_max(fac, a.shrink);
        newDt = dt * fac;
        newDt = lane_min(newDt, a.dtmax);
        newDt = lane_max(newDt, a.dtmin);
    }

    // PT-CTL:23-86, every case of it.  ok: every err_i < tol_i; root: ctrl_root(R, ok).
    __device__ __forceinline__ void control_rkck45(const C& a, const P* nx, const CP* err, bool ok, CP root, int& update)
    {
        bool fin = true;
#pragma unroll
        for (int i = 0; i < SD; i++) fin = fin && math::isfinite(nx[i]) && math::isfinite(err[i]);
        CP fac = CP(0.9) * root;
        fin = fin && math::isfinite(fac);
        const bool smallest = dt < a.dtmin * CP(1.01);
        if (__builtin_amdgcn_ballot_w64(!fin || smallest) != 0) {
            if (!fin) {
                fac = a.shrink;
                ok = false;
                if (smallest) { term = 1; status |= MPGOS_STATUS_NONFINITE_MIN_STEP; }
            } else if (smallest) {
                ok = true;
                status |= MPGOS_STATUS_MIN_STEP_REACHED;
            }
        }
        update = ok ? 1 : 0;
        next_step_size(a, fac);
    }

    // PT-EVT:5-45
    __device__ __forceinline__ void event_control(const C& a, const P* EFn, int& update)
    {
        CP evDt = dt;
        int corrected = 0;
        if (update == 1 && term == 0) {
#pragma unroll
            for (int i = 0; i < NE; i++) {
                const P tol = a.etol[i];
                if ((EF[i] > tol && EFn[i] < -tol && a.edir[i] <= 0) ||
                    (EF[i] < -tol && EFn[i] > tol && a.edir[i] >= 0)) {
                    evDt = mpgos_fmin(evDt, (-(CP)EF[i] / ((CP)EFn[i] - (CP)EF[i])) * dt);
                    corrected = 1;
                }
            }
        }
        if (corrected == 1) {
            if (evDt < a.dtmin) status |= MPGOS_STATUS_EVENT_OMITTED;
            else { newDt = evDt; update = 0; }
        }
    }

    // ------------------------------------------------------------ one attempted step
    // One iteration of the loop at PT-SOL:197-394; returns whether the instance
    // has ended, `accepted` whether the step was.  DENSE = false compiles the
    // dense-output bookkeeping out (the adjoint's re-steps, which run with
    // NDO = 0), so that the step has no branch on it.  CARRY: tt holds the time
    // terms at t (time_terms(t, tt) before the first step); else they are
    // evaluated anew.  GROUP: several lanes per instance (RKCK45, no CARRY).
    // SHORT: see short_way.
    template <bool DENSE = true, bool CARRY = false, int GROUP = 1, bool SHORT = true>
    __device__ __forceinline__ bool step(const C& a, P* sPAR, int* sPARi, bool& accepted, P* tt = nullptr)
    {
        const int NT = a.NT;
        int update = 1;
        bool stop;
        dt = newDt;
        CP remaining;
        if (KAHAN) remaining = (CP)TD[1] - ((CP)t - (CP)tc);
        else remaining = (CP)(TD[1] - t);
        const bool endReached = dt > remaining;
        if (endReached) dt = remaining;

        const P h = (P)dt;
        P nx[SD], inc[KAHAN ? SD : 1];
        P tt1[Pos<NTT>::value], ttm[Pos<NTT>::value], ttEnd[Pos<NTT>::value];
        if constexpr (CARRY) {
#pragma unroll
            for (int i = 0; i < NTT; i++) tt1[i] = tt[i];
        } else if constexpr (GROUP == 1) {
            time_terms(t, tt1);
        }
        P EFn[Pos<NE>::value];
        P dtP = h;
        if constexpr (ALG == MPGOS_RK4) {
            time_terms(t + P(0.5) * h, ttm);
            time_terms(t + h, ttEnd);
            rk4(a, h, nx, inc, sPAR, sPARi, tt1, ttm, ttEnd);
            // PT-CTL:5-20, by selection: a branch here costs every step of a lone
            // wavefront (persistent form, 256 to 200000 Lorenz instances: 0.93
            // times the speed)
            bool fin = true;
#pragma unroll
            for (int i = 0; i < SD; i++) fin = fin && math::isfinite(nx[i]);
            term = fin ? term : 1;
            status |= fin ? 0 : MPGOS_STATUS_NONFINITE_RK4;
            newDt = a.dt0;
            if (NE > 0) Sys::template EventFunction<P>(tid, NT, EFn, t + h, dtP, TD, nx, cPAR, sPAR, sPARi, ACC, ACCi);
            accepted = settle<CARRY>(a, h, dtP, nx, inc, EFn, update, sPAR, sPARi, tt, ttEnd);
            stop = term != 0;
        } else {
            CP err[SD], tol[SD];
            rkck45<GROUP>(a, h, nx, inc, err, sPAR, sPARi, tt1, ttEnd);
            if (NE > 0) Sys::template EventFunction<P>(tid, NT, EFn, t + h, dtP, TD, nx, cPAR, sPAR, sPARi, ACC, ACCi);
            // Nearly always every lane of the wavefront has an accepted, finite
            // step above the smallest size with no event near: u < 0 in one
            // comparison and one branch per wavefront, and no execution mask.
            // Each u >= 0 (or NaN) sends the wavefront the general way, which
            // decides every case as the reference does.  A comparison whose
            // result a scalar instruction or branch waits for costs a lone
            // wavefront 20 cycles, a branch 10 to 20 more, a vector
            // instruction 4; so the tests are folded into arithmetic:
            //   err_i < tol_i           <=>  err_i - tol_i < 0
            //   no event near           <=   |EF| tolerance - (EFn with the sign of EF) <= 0
            //   everything finite       <=>  adding 0 * value leaves u as it is
            // Whole Solves against one masked way for all cases: 256 relief
            // valves 520 -> 325 us, 50001 Lorenz instances 2660 -> 2140 us,
            // 262144 in the sorted form 3.22 -> 2.93 ms, 20000 Duffing instances
            // with events 129 -> 116 ms, Cash-Karp adjoint of 10007 4.50 -> 3.76 ms.
            if constexpr (!SHORT) {
                CP R = CP(1e30);
                bool ok = true;
#pragma unroll
                for (int i = 0; i < SD; i++) {
                    tol[i] = mpgos_fmax(a.rtol[i] * mpgos_fmax(math::fabs((CP)nx[i]), math::fabs((CP)X[i])), a.atol[i]);
                    ok = ok && err[i] < tol[i];
                    R = mpgos_fmin(R, tol[i] / err[i]);
                }
                control_rkck45(a, nx, err, ok, math::ctrl_root(R, ok), update);
                accepted = settle<CARRY>(a, h, dtP, nx, inc, EFn, update, sPAR, sPARi, tt, ttEnd);
                stop = term != 0;
            } else {
                CP R = CP(1e30), u = a.least - dt;
#pragma unroll
                for (int i = 0; i < SD; i++) {
                    tol[i] = lane_max(a.rtol[i] * lane_max_abs((CP)nx[i], (CP)X[i]), a.atol[i]);
                    u = lane_max(u, err[i] - tol[i]);
                    R = lane_min(R, tol[i] / err[i]);
                }
#pragma unroll
                for (int i = 0; i < NE; i++) u = lane_max(u, (CP)(a.etol[i] - math::flip_sign(EFn[i], EF[i])));
#pragma unroll
                for (int i = 0; i < SD; i++) u = math::fma((CP)nx[i], CP(0), math::fma(err[i], CP(0), u));
                const uint64_t unusual = __builtin_amdgcn_ballot_w64(!(u < CP(0)));
                const CP regular = math::ctrl_root_regular(R);
                if (__builtin_expect(unusual == 0, 1)) {
                    next_step_size(a, CP(0.9) * regular);
#pragma unroll
                    for (int i = 0; i < NTT; i++) if (CARRY) tt[i] = ttEnd[i];
                    accept(a, h, dtP, nx, inc, EFn, false, sPAR, sPARi);
                    accepted = true;
                    stop = false;
                } else {
                    bool ok = true;
#pragma unroll
                    for (int i = 0; i < SD; i++) ok = ok && err[i] < tol[i];
                    CP root = regular;
                    if (__builtin_amdgcn_ballot_w64(!(R >= CP(0x1p-100))) != 0) root = math::ctrl_root(R, true);
                    if (__builtin_amdgcn_ballot_w64(!ok) != 0) {
                        const CP fourth = math::ctrl_root(R, false);
                        root = ok ? root : fourth;
                    }
                    control_rkck45(a, nx, err, ok, root, update);
                    accepted = settle<CARRY>(a, h, dtP, nx, inc, EFn, update, sPAR, sPARi, tt, ttEnd);
                    stop = term != 0;
                }
            }
        }
        if (DENSE && __builtin_expect(a.NDO > 0, 0)) {
            if (accepted) dense_output(a, endReached);
        }
        return stop || (accepted && (endReached || udt == 1));
    }

    // After the controller: event step control, then the accepted or rejected step.
    template <bool CARRY>
    __device__ __forceinline__ bool settle(const C& a, P h, P& dtP, const P* nx, const P* inc, P* EFn, int update, P* sPAR,
                                           int* sPARi, P* tt, const P* ttEnd)
    {
        if (NE > 0) event_control(a, EFn, update);
        if constexpr (CARRY) {
            // t + h becomes t when the step is accepted
#pragma unroll
            for (int i = 0; i < NTT; i++) tt[i] = update == 1 ? ttEnd[i] : tt[i];
        }
        if (update == 1) accept(a, h, dtP, nx, inc, EFn, true, sPAR, sPARi);
        else nrej++;
        return update == 1;
    }

    // The accepted part of the loop body (PT-SOL:323-394): t and x take the
    // step's values, then the user's action and event detection (dense output and
    // termination follow).
    __device__ __forceinline__ void accept(const C& a, P h, P& dtP, const P* nx, const P* inc, P* EFn, bool near, P* sPAR, int* sPARi)
    {
        const int NT = a.NT;
        if (KAHAN) {
            // compensated t += h and x += inc
            P y = h - tc; P s = t + y; tc = (s - t) - y; t = s;
#pragma unroll
            for (int i = 0; i < SD; i++) { P yi = inc[i] - Xc[i]; P si = X[i] + yi; Xc[i] = (si - X[i]) - yi; X[i] = si; }
        } else {
            t += h;
#pragma unroll
            for (int i = 0; i < SD; i++) X[i] = nx[i];
        }
        Sys::template ActionAfterSuccessfulTimeStep<P>(tid, NT, udt, t, dtP, TD, X, cPAR, sPAR, sPARi, ACC, ACCi);
        if (NE > 0) {
            if (near) {
#pragma unroll
                for (int i = 0; i < NE; i++) {
                    const P tol = a.etol[i];
                    if ((EF[i] > tol && math::fabs(EFn[i]) < tol && a.edir[i] <= 0) ||
                        (EF[i] < -tol && math::fabs(EFn[i]) < tol && a.edir[i] >= 0)) {
                        const A& c = kernel_args<A>();   // rare path: fields loaded here
                        if (nev < c.evcap) {
                            const long long base = (long long)nev * (SD + 1);
                            c.evlog[tid + base * NT] = t;
#pragma unroll
                            for (int j = 0; j < SD; j++) c.evlog[tid + (base + 1 + j) * NT] = X[j];
                            c.evlogidx[tid + (long long)nev * NT] = i;
                        }
                        nev++;
                        Sys::template ActionAfterEventDetection<P>(tid, NT, i, udt, t, dtP, TD, X, cPAR, sPAR, sPARi, ACC, ACCi);
                    }
                }
            }
            Sys::template EventFunction<P>(tid, NT, EFn, t, dtP, TD, X, cPAR, sPAR, sPARi, ACC, ACCi);
#pragma unroll
            for (int i = 0; i < NE; i++) EF[i] = EFn[i];
        }
        dt = (CP)dtP;   // a callback may have changed dT; it reaches Finalization (PT-SOL:398-410)
        nacc++;
    }

    // PT-DO:40-58 then PT-DO:5-37
    __device__ __forceinline__ void dense_output(const C& a, bool endReached)
    {
        int upd;
        if (doIdx < a.NDO && doT < t && skipped >= a.doFreq - 1) upd = 1;
        else upd = 0;
        if (doIdx < a.NDO && (endReached || udt == 1)) upd = 1;
        if (upd) {
            if constexpr (kCommonTime) store_dense(kernel_args_joined<A>());
            else store_dense(kernel_args<A>());
        } else {
            skipped++;
        }
    }

    // ------------------------------------------------------------ common time
    // Fixed steps of a whole wavefront whose instances share their time.  The
    // time terms (cos t of a forced oscillator: a third to a half of the
    // step's instructions) are then the same in every lane, and the next steps'
    // times are known: each lane evaluates the terms of another time (start
    // and middle of the next 31 steps; start, middle and end of the next 21
    // in the compensated form, whose next start is not t + h), and the steps
    // read them with v_readlane.  One evaluation serves 31 steps instead of
    // three per step; the values are those that every lane would have
    // computed, so the results do not change.  Forced Duffing oscillators, RK4,
    // 16384 instances x 64000 steps (one wavefront per compute unit, bound by the
    // instructions of a step): 158 -> 49 vector instructions per step, 20.9 ->
    // 7.1 ms; 65536 instances recording adjoint checkpoints: 10.9 -> 4.4 ms.
    //
    // Called by every lane of the wavefront, lanes without an instance with term
    // set.  Returns when an instance ends or fewer than a block of steps remain
    // before the end of the time domain, or at once when the lanes' times or
    // ends differ; the caller's ordinary loop does the rest.  `every` > 0:
    // calls at(until) after every `every` accepted steps, the first after
    // `until`.
    template <bool DENSE, class F>
    __device__ __forceinline__ void run_common_time(const C& a, P* sPAR, int* sPARi, int every, int& until, F&& at)
    {
        constexpr int PTS = KAHAN ? 3 : 2, BLK = KAHAN ? 21 : 31;
        const uint64_t live = __ballot(term == 0);
        if (live == 0) return;
        const int first = __builtin_ctzll(live);
        P t0 = lane_value(t, first), c0 = lane_value(tc, first);
        const P end = lane_value(TD[1], first);
        const bool same = math::bits(t) == math::bits(t0) && math::bits(TD[1]) == math::bits(end) && math::bits(tc) == math::bits(c0);
        if (!__all(term != 0 || same) || !(a.dt0 > CP(0))) return;
        const P h = (P)a.dt0;
        const int kind = (int)(__lane_id() % PTS);
        const bool mine = term == 0;    // the others step along on zeros, storing nothing
        for (;;) {
            P tv = t0, cv = c0;
            if constexpr (KAHAN) advance_by_lane_kahan(tv, cv, h);
            else advance_by_lane(tv, cv, h);
            // no step of the block may be clipped to the end: t grows, so the
            // last one decides
            const P tl = lane_value(tv, PTS * (BLK - 1)), cl = lane_value(cv, PTS * (BLK - 1));
            CP remaining;
            if (KAHAN) remaining = (CP)end - ((CP)tl - (CP)cl);
            else remaining = (CP)(end - tl);
            if (__any(a.dt0 > remaining)) return;
            const P T = kind == 0 ? tv : (kind == 1 ? tv + P(0.5) * h : tv + h);
            P tt[Pos<NTT>::value];
            time_terms(T, tt);
            for (int j = 0; j < BLK;) {
                int n = BLK - j;
                if (every > 0 && until < n) n = until;
                const Lane before = *this;
                P tt1[Pos<NTT>::value], ttm[Pos<NTT>::value], tt4[Pos<NTT>::value];
#pragma unroll
                for (int i = 0; i < NTT; i++) tt1[i] = lane_value(tt[i], PTS * j);
                P zero = P(0);          // becomes NaN at the first non-finite state
                int ended = 0;          // the user ended the integration
                auto one = [&](int m) {
#pragma unroll
                    for (int i = 0; i < NTT; i++) {
                        if (KAHAN) tt1[i] = lane_value(tt[i], PTS * m);
                        ttm[i] = lane_value(tt[i], PTS * m + 1);
                        tt4[i] = lane_value(tt[i], PTS * m + 2);
                    }
                    P nx[SD], inc[KAHAN ? SD : 1], EFn[1], dtP = h;
                    rk4(a, h, nx, inc, sPAR, sPARi, tt1, ttm, tt4);
                    // an instance that has ended stores no more points
                    const bool open = !DENSE || (zero == P(0) && ended == 0);
#pragma unroll
                    for (int i = 0; i < SD; i++) zero = math::fma(nx[i], P(0), zero);
                    accept(a, h, dtP, nx, inc, EFn, false, sPAR, sPARi);
                    if (DENSE && open) dense_output(a, false);
                    ended |= udt;
#pragma unroll
                    for (int i = 0; i < NTT; i++) tt1[i] = tt4[i];
                };
                int m = j;
                for (; m + 4 <= j + n; m += 4) { one(m); one(m + 1); one(m + 2); one(m + 3); }
                for (; m < j + n; m++) one(m);
                // an instance ended on the way: the ordinary loop makes these
                // steps again (the dense output up to its end is stored again)
                if (__any(mine && (zero != P(0) || ended != 0))) {
                    *this = before;
                    return;
                }
                j += n;
                if (every > 0) {
                    until -= n;
                    if (until == 0) { until = every; at(); }
                }
            }
            t0 = lane_value(tv, PTS * BLK);
            c0 = lane_value(cv, PTS * BLK);
        }
    }

    // ------------------------------------------------------------ epilogue
    __device__ __forceinline__ void finish(const A& a, P* sPAR, int* sPARi)
    {
        const int NT = a.NT;
        P dtP = (P)dt;
        Sys::template Finalization<P>(tid, NT, doIdx, t, dtP, TD, X, cPAR, sPAR, sPARi, ACC, ACCi);
#pragma unroll
        for (int i = 0; i < 2; i++) a.TD[tid + i * NT] = TD[i];
#pragma unroll
        for (int i = 0; i < SD; i++) a.X[tid + i * NT] = X[i];
#pragma unroll
        for (int i = 0; i < NCP; i++) a.cPAR[tid + i * NT] = cPAR[i];
#pragma unroll
        for (int i = 0; i < NA; i++) a.ACC[tid + i * NT] = ACC[i];
#pragma unroll
        for (int i = 0; i < NIA; i++) a.ACCi[tid + i * NT] = ACCi[i];
        a.T[tid] = t;
        a.DOidx[tid] = doIdx;
        a.nacc[tid] = nacc;
        a.nrej[tid] = nrej;
        a.status[tid] = status;
        a.nev[tid] = nev;
    }
};

// Words of the lane state that an instantiation never uses (Kahan terms
// without Kahan, accessories, event values and the slice budget of systems or
// forms that have none): the persistent form does not move them between
// lanes, so they hold no registers.
template <class L_t, bool SLICED>
__host__ __device__ constexpr bool lane_word_live(int w)
{
    using Sys = typename L_t::Sys_t;
    const int b = 4 * w;
    auto in = [&](size_t off, size_t bytes) { return (size_t)b >= off && (size_t)b < off + bytes; };
    if (!L_t::kKahan && (in(offsetof(L_t, Xc), sizeof(L_t::Xc)) || in(offsetof(L_t, tc), sizeof(L_t::tc)))) return false;
    if (Sys::NA == 0 && in(offsetof(L_t, ACC), sizeof(L_t::ACC))) return false;
    if (Sys::NIA == 0 && in(offsetof(L_t, ACCi), sizeof(L_t::ACCi))) return false;
    if (Sys::NE == 0 && in(offsetof(L_t, EF), sizeof(L_t::EF))) return false;
    if (!SLICED && in(offsetof(L_t, left), sizeof(L_t::left))) return false;
    return true;
}

// Stage shared parameters into LDS (PT-SOL:67-88) or point at global memory.
template <class Sys, class P, class CP>
__device__ __forceinline__ void stage_shared(const Args<Sys, P, CP>& a, P*& sPAR, int*& sPARi)
{
    constexpr int NSP = Sys::NSP, NISP = Sys::NISP;
    extern __shared__ __align__(16) unsigned char mpgos_dyn_lds[];
    if (a.preferShared && (NSP + NISP) > 0) {
        P* lp = reinterpret_cast<P*>(mpgos_dyn_lds);
        int* li = reinterpret_cast<int*>(lp + NSP);
        for (int i = threadIdx.x; i < NSP; i += blockDim.x) lp[i] = a.sPAR[i];
        for (int i = threadIdx.x; i < NISP; i += blockDim.x) li[i] = a.sPARi[i];
        __syncthreads();
        sPAR = lp;
        sPARi = li;
    } else {
        sPAR = a.sPAR;
        sPARi = a.sPARi;
    }
}

// Reference form: lane = instance, whole integration in one launch.  GROUP: that
// many lanes per instance (whole wavefronts; its first lane stores).  Instances
// list[first + ...) in the order of the lanes of workgroups `block0` and later.
template <class Sys, class P, bool KAHAN, int ALG, bool SLICED = false, int GROUP = 1, int WPE = 1>
__device__ __forceinline__ void plain_body(const Args<Sys, P, typename Lane<Sys, P, KAHAN, ALG>::CP>& a, int block0 = 0, int first = 0)
{
    P* sPAR; int* sPARi;
    stage_shared(a, sPAR, sPARi);
    const int i = first + (int)(threadIdx.x / GROUP) + ((int)blockIdx.x - block0) * (int)(blockDim.x / GROUP);
    const int n = (SLICED && a.listLenDev) ? (int)*a.listLenDev : a.listLen;
    using L_t = Lane<Sys, P, KAHAN, ALG>;
    L_t L;
    typename L_t::C c(a, ALG == MPGOS_RKCK45, WPE < kNarrowWaves);
    if constexpr (GROUP > 1) c.template set_nodes<GROUP>();
    const bool stores = GROUP == 1 || threadIdx.x % GROUP == 0;
    const int id = i < n ? (a.list ? a.list[i] : i) : 0;
    constexpr bool COMMON = !SLICED && L_t::kCommonTime;
    // a step's end is the next one's start (in the compensated form it is not t + h)
    constexpr bool CARRY = L_t::NTT > 0 && !KAHAN && GROUP == 1;
    P tt[Pos<L_t::NTT>::value];
    if constexpr (COMMON) {
        if (i < n) L.load(a, id, sPAR, sPARi);
        else L.idle();
        // whole wavefronts only (the lanes of a wavefront work together)
        if ((blockDim.x & 63) == 0) {
            int until = 0;
            if (a.NDO > 0) L.template run_common_time<true>(c, sPAR, sPARi, 0, until, [] {});
            else L.template run_common_time<false>(c, sPAR, sPARi, 0, until, [] {});
        }
    }
    if (i < n) {
        if constexpr (SLICED) {
            // the loop only steps; finishing or suspending follows it, so
            // the step loop keeps the plain form's registers
            L.begin(a, id, sPAR, sPARi);
            if (CARRY) L.time_terms(L.t, tt);
            // the budget is the same for every lane
            int left = a.slice;
            bool ended, accepted;
            do ended = L.template step<true, CARRY, GROUP, short_way<KAHAN, WPE>()>(c, sPAR, sPARi, accepted, tt);
            while (!ended && --left > 0);
            if (ended) L.term = 1;
            if (stores) L.release(kernel_args<typename L_t::A>(), sPAR, sPARi);
        } else {
            if constexpr (!COMMON) L.load(a, id, sPAR, sPARi);
            if (CARRY) L.time_terms(L.t, tt);
            bool ended = L.term != 0, accepted;
            while (!ended) ended = L.template step<true, CARRY, GROUP, short_way<KAHAN, WPE>()>(c, sPAR, sPARi, accepted, tt);
            if (!stores) return;
            if constexpr (COMMON) L.finish(kernel_args_joined<typename L_t::A>(), sPAR, sPARi);
            else L.finish(kernel_args<typename L_t::A>(), sPAR, sPARi);
        }
    }
}

// Sorted form's long launch: the first a.octets workgroups give their instances
// (the longest ones) 8 lanes each.
template <class Sys, class P, bool KAHAN, int ALG>
__device__ __forceinline__ void mixed_body(const Args<Sys, P, typename Lane<Sys, P, KAHAN, ALG>::CP>& a)
{
    if ((int)blockIdx.x < a.octets) {
        // before the others that share its SIMD: it decides when the launch ends
        __builtin_amdgcn_s_setprio(2);
        plain_body<Sys, P, KAHAN, ALG, true, 8>(a);
    } else {
        plain_body<Sys, P, KAHAN, ALG, true>(a, a.octets, a.octets * (int)(blockDim.x / 8));
    }
}

// Persistent form with lane compaction.  Lanes pull instances from a device
// work queue; every `roundSteps` attempted steps the workgroup
//   1. counts its live lanes (wavefront ballots, prefix over waves in LDS),
//   2. reserves as many fresh instances as it has idle lanes (one atomic per
//      workgroup) and starts them in the idle lanes where they are (no state
//      moves while the queue lasts),
//   3. once nothing new arrives, packs the live instances into the lowest
//      lanes through LDS -- only when that empties at least one wave, so the
//      waves above the packed range have nothing to do and sleep at the
//      barrier instead of issuing instructions for idle lanes.
// Every instance's arithmetic is independent of the lane that runs it, so the
// results are bit-identical to the plain form.  The workgroup leaves the loop
// together once the queue is drained and no lane is live (block-uniform test).
template <class Sys, class P, bool KAHAN, int ALG, bool SLICED = false, int WPE = 1>
__device__ __forceinline__ void persistent_body(const Args<Sys, P, typename Lane<Sys, P, KAHAN, ALG>::CP>& a)
{
    using L_t = Lane<Sys, P, KAHAN, ALG>;
    constexpr int NW = (int)(sizeof(L_t) / 4);       // lane state in 32-bit words
    constexpr int CW = 4;                             // words moved per LDS pass
    constexpr int NCH = (NW + CW - 1) / CW;
    P* sPAR; int* sPARi;
    stage_shared(a, sPAR, sPARi);

    extern __shared__ __align__(16) unsigned char mpgos_dyn_lds[];
    const size_t sharedBytes = ((size_t)Sys::NSP * sizeof(P) + (size_t)Sys::NISP * sizeof(int) + 15) & ~(size_t)15;
    unsigned* ctl = reinterpret_cast<unsigned*>(mpgos_dyn_lds + sharedBytes);   // [0..15] wave counts, [16] base, [17] fresh, [18] drained
    unsigned* xch = ctl + 32;                                                  // CW * blockDim.x words

    const int B = blockDim.x;
    const int tid = threadIdx.x;
    const int wave = tid >> 6;
    const int nwaves = (B + 63) >> 6;
    const unsigned lane = __lane_id();

    L_t L;
    const typename L_t::C c(a, ALG == MPGOS_RKCK45, WPE < kNarrowWaves);
    bool busy = false;
    const unsigned D = (unsigned)a.solo;
    if (tid == 0) {
        ctl[18] = 0u;
        ctl[20] = blockIdx.x < D ? 1u : 0u;   // solo phase: lane 0 alone runs one of the first D entries
    }
    for (;;) {
        // ---- 1. count live lanes
        const unsigned long long live_mask = __ballot(busy);
        if (lane == 0) ctl[wave] = (unsigned)__popcll(live_mask);
        __syncthreads();
        unsigned before = 0, live = 0, occupied = 0;
        for (int w = 0; w < nwaves; w++) {
            const unsigned c = ctl[w];
            if (w < wave) before += c;
            live += c;
            occupied += c > 0 ? 1u : 0u;
        }
        const unsigned long long below = (1ull << lane) - 1ull;
        const unsigned rank = before + (unsigned)__popcll(live_mask & below);             // among live lanes
        const unsigned idleRank = (unsigned)(wave * 64) - before + (unsigned)__popcll(~live_mask & below);   // among idle lanes
        // ---- 2. reserve fresh instances for the idle lanes
        if (tid == 0) {
            unsigned base = 0, fresh = 0;
            if (ctl[20] && live == 0) {
                const unsigned q = atomicAdd(&a.queue[2], 1u);
                if (q < D) { base = q; fresh = 1u; }
                else ctl[20] = 0u;                  // solo entries taken: a full workgroup from now on
            }
            if (!ctl[20]) {
                const unsigned need = (unsigned)B - live;
                if (!ctl[18] && need > 0) {
                    base = D + atomicAdd(a.queue, need);
                    if (base < (unsigned)a.listLen) fresh = min(need, (unsigned)a.listLen - base);
                    if (base + need >= (unsigned)a.listLen) ctl[18] = 1u;
                }
            }
            ctl[16] = base;
            ctl[17] = fresh;
        }
        __syncthreads();
        const unsigned base = ctl[16], fresh = ctl[17];
        if (live == 0 && fresh == 0) break;           // block-uniform: queue drained, nothing live
        // ---- 3. fresh instances start in the idle lanes where they are; with
        // nothing new, live states are packed into lanes [0, live) when that
        // empties a wave (block-uniform decision)
        if (fresh != 0) {
            if (!busy && idleRank < fresh) {
                const int q = (int)(base + idleRank);
                const int id = a.list ? a.list[q] : q;
                if constexpr (SLICED) L.begin(a, id, sPAR, sPARi);
                else L.load(a, id, sPAR, sPARi);
                busy = true;
            }
        } else if (occupied > (live + 63u) / 64u) {
            // the lane state moves in place, CW words per pass (no second copy of it)
            unsigned char* lw = reinterpret_cast<unsigned char*>(&L);
#pragma unroll
            for (int c = 0; c < NCH; c++) {
                constexpr int last = NW - (NCH - 1) * CW;
                const int nw = c == NCH - 1 ? last : CW;
                bool any = false;
#pragma unroll
                for (int j = 0; j < CW; j++) any = any || (j < nw && lane_word_live<L_t, SLICED>(c * CW + j));
                if (!any) continue;                   // compile-time: a chunk of unused words
                uint32_t w[CW];
                __builtin_memcpy(w, lw + c * CW * 4, nw * 4);
                if (busy) {
#pragma unroll
                    for (int j = 0; j < CW; j++)
                        if (j < nw && lane_word_live<L_t, SLICED>(c * CW + j)) xch[j * B + rank] = w[j];
                }
                __syncthreads();
                if ((unsigned)tid < live) {
#pragma unroll
                    for (int j = 0; j < CW; j++)
                        if (j < nw && lane_word_live<L_t, SLICED>(c * CW + j)) w[j] = xch[j * B + tid];
                    __builtin_memcpy(lw + c * CW * 4, w, nw * 4);
                }
                __syncthreads();
            }
            busy = (unsigned)tid < live;
        }
        // ---- 4. integrate
        for (int m = 0; m < a.roundSteps; m++) {
            if (!__any(busy)) break;
            if (busy) {
                bool accepted;
                const bool ended = L.template step<true, false, 1, short_way<KAHAN, WPE>()>(c, sPAR, sPARi, accepted);
                if (ended) L.term = 1;
                if constexpr (SLICED) {
                    if (L.stop()) {
                        L.release(kernel_args<typename L_t::A>(), sPAR, sPARi);
                        busy = false;
                    }
                } else if (ended) {
                    L.finish(kernel_args<typename L_t::A>(), sPAR, sPARi);
                    busy = false;
                }
            }
        }
    }
}

// LDS bytes of the persistent form beyond the shared parameters.
template <class Sys, class P, bool KAHAN, int ALG>
constexpr size_t persistent_lds_bytes(int block)
{
    return 32 * 4 + (size_t)4 * 4 * block;
}

// Clears the per-instance phases and the per-launch counts of the relaunch
// form (a kernel, so the launch sequence can be captured in a graph).
template <int Unused = 0>
__global__ void reset_relaunch_kernel(int* phase, int n, unsigned* counts, int nc)
{
    const int i = threadIdx.x + blockIdx.x * blockDim.x;
    if (i < n) phase[i] = 0;
    if (i < nc) counts[i] = 0u;
}

// Sorted form: after the pilot launch the suspended instances are ordered by
// their estimated remaining attempted steps, largest first, so that every
// wavefront of the following launch holds instances of similar length (lane
// coherence; the order only schedules, results are bit-identical).  A
// counting sort on 256 buckets of 1/8 octave (float exponent and the top three
// mantissa bits of the estimate): histogram, scan, scatter.
__device__ __forceinline__ int sort_bucket(float key)
{
    const float k = key < 1.0f ? 1.0f : (key > 4.0e9f ? 4.0e9f : key);
    const unsigned b = __float_as_uint(k);
    const int v = ((int)(b >> 23) - 127) * 8 + (int)((b >> 20) & 7u);   // 0 .. 255 for keys in [1, 2^32)
    return 255 - v;                                                       // largest estimates first
}

template <int Unused = 0>
__global__ void sort_histogram_kernel(const float* key, const unsigned* n, unsigned* hist)
{
    __shared__ unsigned h[256];
    for (int j = threadIdx.x; j < 256; j += blockDim.x) h[j] = 0u;
    __syncthreads();
    const unsigned len = *n;
    for (unsigned i = threadIdx.x + blockIdx.x * blockDim.x; i < len; i += gridDim.x * blockDim.x)
        atomicAdd(&h[sort_bucket(key[i])], 1u);
    __syncthreads();
    for (int j = threadIdx.x; j < 256; j += blockDim.x)
        if (h[j]) atomicAdd(&hist[j], h[j]);
}

// exclusive scan of the 256 bucket counts into bucket offsets (one workgroup)
template <int Unused = 0>
__global__ void sort_scan_kernel(unsigned* hist)
{
    if (threadIdx.x == 0) {
        unsigned run = 0u;
        for (int j = 0; j < 256; j++) { const unsigned c = hist[j]; hist[j] = run; run += c; }
    }
}

// one workgroup per 256 list entries: the workgroup counts its entries per
// bucket in LDS, reserves each bucket's range with one global atomic, and
// places its entries with LDS atomics (no global atomics per entry)
template <int Unused = 0>
__global__ void sort_scatter_kernel(const float* key, const int* listIn, const unsigned* n, unsigned* offset, int* listOut)
{
    __shared__ unsigned cnt[256], base[256];
    const unsigned len = *n;
    const unsigned i = threadIdx.x + blockIdx.x * blockDim.x;
    if (blockIdx.x * blockDim.x >= len) return;          // workgroup-uniform
    cnt[threadIdx.x] = 0u;
    __syncthreads();
    const int b = i < len ? sort_bucket(key[i]) : -1;
    if (b >= 0) atomicAdd(&cnt[b], 1u);
    __syncthreads();
    const unsigned c = cnt[threadIdx.x];
    if (c) base[threadIdx.x] = atomicAdd(&offset[threadIdx.x], c);
    cnt[threadIdx.x] = 0u;
    __syncthreads();
    if (b >= 0) listOut[base[b] + atomicAdd(&cnt[b], 1u)] = listIn[i];
}

template <int Unused = 0>
__global__ void zero_kernel(unsigned* p, int n)
{
    const int i = threadIdx.x + blockIdx.x * blockDim.x;
    if (i < n) p[i] = 0u;
}

// Resets the work-queue head on the stream (a kernel, so the sequence can be
// captured in a graph without a memset node).
template <int Unused = 0>
__global__ void reset_queue_kernel(unsigned int* q)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) { q[0] = 0u; q[2] = 0u; }
}

} // namespace pt
} // namespace mpgos
