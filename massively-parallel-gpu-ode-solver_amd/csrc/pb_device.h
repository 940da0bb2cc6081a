// Per-block coupled-systems solver for gfx950: one workgroup integrates SPB
// systems of UPS coupled units, a lane owns one (system, unit) pair.
//
// Semantics follow the reference's per-block kernels
// (SourceCodes/CoupledSystmes_PerBlock_Solver.cuh, single-system form at
// :2214-2888, multi-system masking at :359 and :2532): system scope (time,
// step, system parameters and accessories, dense-output bookkeeping, flags)
// lives in LDS, unit scope in VGPRs; every right-hand-side evaluation is
// followed by the coupling terms
//   F[CouplingIndex[i]] += CouplingStrength[i] * CPF[i] * sum_col M_i(u, col) CPT_col[i]
// (ComputeCouplingValue_SingleSystem, CoupledSystems_PerBlock_ExplicitRungeKutta_Steppers.cuh:2634-2713,
// all four storage forms of the coupling matrix); the step is controlled per
// system by reductions over its units: acceptance = AND over units, ratio =
// min over units of min_i tol_i/err_i, safety factor 0.8
// (CoupledSystems_PerBlock_ExplicitRungeKutta_ErrorControllers.cuh:424-542);
// event step control takes the minimum interpolated step over units
// (CoupledSystems_PerBlock_EventHandling.cuh:215-268); dense output is stored
// only after accepted steps (CoupledSystems_PerBlock_DenseOutput.cuh:312-395).
//
// MI355X design: the reductions are LDS atomics on ordered bit patterns
// (min of non-negative doubles, AND of flags), which are order-independent and
// therefore deterministic; multiply-adds are explicit fma in the contracted
// form of the reference's expressions, so the host oracle reproduces every bit.
//
// Two coupling forms:
//  * lane-per-pair (any storage form and precision, this file): each lane forms
//    its own dot product, coupling matrix from L2 (or LDS), coupling terms
//    double-buffered in LDS (one barrier per stage);
//  * dense contraction (full FP64 matrix, pb_dense.h): the products of all
//    systems of a workgroup on the matrix cores, with the same bits.
#pragma once

#include <hip/hip_runtime.h>

#include <type_traits>

#include "mpgos.h"
#include "mpgos_math.h"

namespace mpgos {
namespace pb {

template <int N> struct Pos { static constexpr int value = N > 0 ? N : 1; };

// Workgroup barrier that orders LDS only: waits for the wave's own LDS
// operations (lgkmcnt) and not for its global loads and stores, which stay in
// flight across the barrier (__syncthreads also drains vmcnt).  For barriers
// whose only purpose is LDS communication; global data exchanged between lanes
// still needs __syncthreads.
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

constexpr int kMaxBlock = 1024;
enum Coupling { kLaneCoupling = 0, kDenseCoupling = 1 };

// CP: precision of the step size, tolerances and controller (FP64 in the
// FLOAT_KAHAN mode, else P).
template <class Sys, class P, class CP = P>
struct Args {
    static constexpr int UD = Sys::UD, NE = Sys::NE;
    // unit scope, index (system * UPS + unit) + component * NU, NU = NS * UPS
    P* X; P* uPAR; P* uACC; int* uACCi;
    // system scope, index system + component * NS
    P* TD; P* T; P* sPAR; P* sACC; int* sACCi; P* strength; int* DOidx; P* DOt;
    P* DOx;                   // unit index + component * NU + k * NU * UD
    // global scope
    P* gPAR; int* gPARi; int* cIndex; P* cMat;
    const P* cTile;           // dense-contraction form: the matrix in column-block pairs per lane
    int ldsPairs;             // dense-contraction form: leading column-block pairs of every tile of cTile held in LDS
    long long* nacc; long long* nrej; int* status;
    int NS, UPS, SPB, nActive, NDO, CBW, CCI, cMatSize, sharedGlobals, sharedMatrix;
    int doFreq;
    CP dt0, dtmax, dtmin, grow, shrink;
    P doMinDt;
    CP rtol[UD], atol[UD];
    P etol[Pos<NE>::value];
    int edir[Pos<NE>::value];
    // record pass of the discrete adjoint (unused otherwise): unit states every
    // recK accepted steps, recX[(k * UD + c) * NU + unit], k < recCkCap; time
    // and size of every accepted step, recT/recH[n * NS + system], n < recStepCap
    P* recX; P* recT; P* recH;
    int recK, recCkCap, recStepCap;
};

// System scope of one system (LDS).  KAHAN: FP32 time with its compensation
// tc, FP64 step sizes, and dtP, the FP32 copy of the step size that the user
// callbacks see (and may change).
template <class Sys, class P, bool KAHAN = false>
struct SysScope {
    using CP = typename std::conditional<KAHAN, double, P>::type;
    P TD[2];
    P t;
    CP dt, newDt;
    P doT;
    P tc, dtP;
    P sPAR[Pos<Sys::NSP>::value];
    P sACC[Pos<Sys::NSA>::value];
    P strength[Pos<Sys::NC>::value];
    unsigned long long ratioBits;     // min over units of tol/err (non-negative double bits)
    unsigned long long eventBits;     // min over units of the interpolated event step
    int sACCi[Pos<Sys::NiSA>::value];
    int DOidx, updDO, skipped;
    int update, isfin, end, term, udt, corrected;
    int nacc, nrej, status;
};

template <class P> __device__ __forceinline__ unsigned long long order_bits(P v);
template <> __device__ __forceinline__ unsigned long long order_bits<double>(double v) { return (unsigned long long)math::bits(v); }
template <> __device__ __forceinline__ unsigned long long order_bits<float>(float v) { return (unsigned long long)math::bits(v); }
template <class P> __device__ __forceinline__ P from_order_bits(unsigned long long b);
template <> __device__ __forceinline__ double from_order_bits<double>(unsigned long long b) { return math::from_bits(b); }
template <> __device__ __forceinline__ float from_order_bits<float>(unsigned long long b) { return math::from_bits32((uint32_t)b); }

template <class P> __device__ __forceinline__ P dmin(P a, P b);
template <> __device__ __forceinline__ double dmin<double>(double a, double b) { return __builtin_fmin(a, b); }
template <> __device__ __forceinline__ float dmin<float>(float a, float b) { return __builtin_fminf(a, b); }
template <class P> __device__ __forceinline__ P dmax(P a, P b);
template <> __device__ __forceinline__ double dmax<double>(double a, double b) { return __builtin_fmax(a, b); }
template <> __device__ __forceinline__ float dmax<float>(float a, float b) { return __builtin_fmaxf(a, b); }

// LDS of the lane-per-pair form: system scopes, two [system][unit][coupling]
// buffers of coupling terms, optional copies of the global parameters and
// coupling matrices.
struct LdsLayout {
    size_t cpt, g, gi, m, total;
};

template <class Sys, class P, bool KAHAN = false>
__host__ __device__ inline LdsLayout lds_layout(int SPB, int UPS, int sharedGlobals, int sharedMatrix, int cMatSize)
{
    constexpr int NCp = Pos<Sys::NC>::value;
    LdsLayout L;
    size_t o = (size_t)SPB * sizeof(SysScope<Sys, P, KAHAN>);
    o = (o + 15) & ~(size_t)15;
    L.cpt = o;
    o += 2 * (size_t)SPB * UPS * NCp * sizeof(P);
    L.g = o;
    if (sharedGlobals) o += (size_t)Sys::NGP * sizeof(P);
    o = (o + 15) & ~(size_t)15;
    L.m = o;
    if (sharedMatrix) o += (size_t)Sys::NC * cMatSize * sizeof(P);
    L.gi = o;
    if (sharedGlobals) o += (size_t)Sys::NiGP * sizeof(int);
    L.total = (o + 15) & ~(size_t)15;
    return L;
}

template <class Sys, class P>
struct Unit {
    static constexpr int UD = Sys::UD, NC = Sys::NC, NE = Sys::NE;

    using GP = const __attribute__((address_space(1))) P*;
    using LP = const __attribute__((address_space(3))) P*;

    // v = fma(M(u, k), CPT_k, v) over the columns k = col .. col + N - 1, in
    // order, the matrix values loaded ahead
    template <int N>
    static __device__ __forceinline__ void dot(GP Mi, LP cpt, int col, int i, int UPS, P& v)
    {
        P m[N];
#pragma unroll
        for (int j = 0; j < N; j++) m[j] = Mi[(size_t)(col + j) * UPS];
#pragma unroll
        for (int j = 0; j < N; j++) v = math::fma(m[j], cpt[(col + j) * NC + i], v);
    }

    // coupling: F[CouplingIndex[i]] += strength_i CPF_i sum_col M_i(u, col) CPT_col[i].
    // GROUPED: full matrices in global memory, the columns in groups (lane_grouped
    // in pb_engine.h says where); else any storage form, one after the other.
    template <bool GROUPED, class A>
    static __device__ __forceinline__ void couple(const A& a, const P* M, const int* cIndex, const P* strength,
                                                  const P* cptSys, int u, const P* CPF, P* F)
    {
        const int UPS = a.UPS;
#pragma unroll
        for (int i = 0; i < NC; i++) {
            P v = P(0);
            if constexpr (GROUPED) {
                const GP Mi = (GP)(M + (size_t)i * UPS * UPS + u);
                const LP cpt = (LP)cptSys;
                // Bound by the latency of the matrix loads (L2 and beyond), so
                // eight are in flight at a time, as global loads (through a
                // generic pointer they count as LDS operations too, and the
                // coupling terms from LDS wait for them: 100 x 128 FP64, RK4,
                // 1.10 -> 0.84 ms).  Against a plain loop over the columns: 46 x 64
                // FP32 622 -> 500 us, 500 x 256 FP32 4.80 -> 3.39 ms, 60 x 300
                // FP64 16.0 -> 6.3 ms, 200 x 1024 FP64 163 -> 68 ms.  The last 1 to
                // 3 columns load the last one again in place of absent ones and
                // skip the product (300 x 7 FP32: 0.46 -> 0.38 ms against a plain
                // loop for all but the eights).
                int col = 0;
                for (; col + 8 <= UPS; col += 8) dot<8>(Mi, cpt, col, i, UPS, v);
                if (col + 4 <= UPS) { dot<4>(Mi, cpt, col, i, UPS, v); col += 4; }
                if (col < UPS) {
                    P m[3], c[3];
#pragma unroll
                    for (int j = 0; j < 3; j++) {
                        const int k = col + j < UPS ? col + j : UPS - 1;
                        m[j] = Mi[(size_t)k * UPS];
                        c[j] = cpt[k * NC + i];
                    }
#pragma unroll
                    for (int j = 0; j < 3; j++) {
                        const P w = math::fma(m[j], c[j], v);
                        v = col + j < UPS ? w : v;
                    }
                }
            } else if (a.CCI == 0 && a.CBW == 0) {
                const P* Mi = M + (size_t)i * UPS * UPS + u;
                for (int col = 0; col < UPS; col++) v = math::fma(Mi[(size_t)col * UPS], cptSys[col * NC + i], v);
            } else if (a.CCI == 0) {
                const int W = 2 * a.CBW + 1;
                const P* Mi = M + (size_t)i * UPS * W + u;
                for (int d = 0; d < W; d++) {
                    int col = u + d - a.CBW;
                    if (col >= UPS) col -= UPS;
                    if (col < 0) col += UPS;
                    v = math::fma(Mi[(size_t)d * UPS], cptSys[col * NC + i], v);
                }
            } else {
                const int W = a.CBW > 0 ? 2 * a.CBW + 1 : UPS;
                const P* Mi = M + (size_t)i * W;
                for (int d = 0; d < W; d++) {
                    int col = u + d - a.CBW;
                    if (col >= UPS) col -= UPS;
                    if (col < 0) col += UPS;
                    v = math::fma(Mi[d], cptSys[col * NC + i], v);
                }
            }
            add(cIndex[i], strength[i] * CPF[i], v, F);
        }
    }

    // F[ci] = fma(sc, v, F[ci]) for a run-time component ci, written as a
    // select per component so that F stays in registers (a conditional store
    // per component is merged by the compiler into one dynamically indexed
    // store, which moves F to scratch memory)
    static __device__ __forceinline__ void add(int ci, P sc, P v, P* F)
    {
#pragma unroll
        for (int c = 0; c < UD; c++) {
            const P f = math::fma(sc, v, F[c]);
            F[c] = c == ci ? f : F[c];
        }
    }
};

// One workgroup = SPB systems: lane t owns unit t % UPS of block system t / UPS,
// so global accesses to unit-scope arrays are coalesced.
//
// KAHAN (P = float): FLOAT_KAHAN mode.  Unit states, stages, right-hand sides
// and coupling terms in FP32; the state and the time are accumulated with Kahan
// compensation (x += dt * sum b_j k_j and t += dt as compensated sums); the
// step size, the error norm (from the FP32 stages in FP64 arithmetic), the
// controller and the event step control in FP64.
//
// A lane's registers decide how many wavefronts a SIMD holds, and these kernels
// sit at the limits (FP32 Cash-Karp of the double-well ring: 128 of the 128 that
// allow four).  Two loops over the lane's kUnits = 1 units keep its values from
// being live where they are not needed; written without them the same kernel has
// 130 registers and three wavefronts: 4000 systems of 10 units 0.26 -> 0.34 ms.
// The right-hand sides' polynomials keep their coefficients out of registers
// (MPGOS_HORNER_IN_REGISTERS) for the same reason: with them in registers 141,
// and a circular matrix of 64 units (FP32, RK4) 0.80 -> 1.50 ms.
template <class Sys, class P, int ALG, bool GROUPED, bool REC = false, bool KAHAN = false>
__device__ void pb_body(const Args<Sys, P, typename SysScope<Sys, P, KAHAN>::CP>& a)
{
    constexpr int UD = Sys::UD, NC = Sys::NC, NUP = Sys::NUP, NSP = Sys::NSP, NGP = Sys::NGP, NiGP = Sys::NiGP;
    constexpr int NUA = Sys::NUA, NiUA = Sys::NiUA, NSA = Sys::NSA, NiSA = Sys::NiSA, NE = Sys::NE;
    constexpr int NCp = Pos<NC>::value, kUnits = 1;
    using S = SysScope<Sys, P, KAHAN>;
    using CP = typename S::CP;
    using U = Unit<Sys, P>;
    using math::fma;

    extern __shared__ __align__(16) unsigned char mpgos_pb_lds[];
    const LdsLayout L = lds_layout<Sys, P, KAHAN>(a.SPB, a.UPS, a.sharedGlobals, a.sharedMatrix, a.cMatSize);
    S* sys = reinterpret_cast<S*>(mpgos_pb_lds);
    P* cptBuf = reinterpret_cast<P*>(mpgos_pb_lds + L.cpt);
    const int cptStride = a.SPB * a.UPS * NCp;

    const int UPS = a.UPS, NS = a.NS, SPB = a.SPB;
    const int tid = threadIdx.x;
    const int lsys = tid / UPS;
    const int u = tid - lsys * UPS;
    const bool lane = lsys < SPB;                              // lane owns a (system, unit) pair
    const bool leader = lane && u == 0;
    const size_t NU = (size_t)NS * UPS;
    const int gsys = blockIdx.x * SPB + lsys;
    const bool exists = lane && gsys < NS;
    const bool active = exists && gsys < a.nActive;
    S* const my = lane ? &sys[lsys] : &sys[0];
    auto gu = [&]() { return (size_t)gsys * UPS + u; };        // unit-scope index, formed where it is used

    // ---- global scope (LDS when SharedGlobalVariables / SharedCouplingMatrices)
    P* gPAR = a.gPAR;
    int* gPARi = a.gPARi;
    const P* M = a.cMat;
    if (a.sharedGlobals) {
        P* lg = reinterpret_cast<P*>(mpgos_pb_lds + L.g);
        int* lgi = reinterpret_cast<int*>(mpgos_pb_lds + L.gi);
        for (int i = tid; i < NGP; i += blockDim.x) lg[i] = a.gPAR[i];
        for (int i = tid; i < NiGP; i += blockDim.x) lgi[i] = a.gPARi[i];
        gPAR = lg;
        gPARi = lgi;
    }
    if (a.sharedMatrix) {
        P* lm = reinterpret_cast<P*>(mpgos_pb_lds + L.m);
        for (int i = tid; i < NC * a.cMatSize; i += blockDim.x) lm[i] = a.cMat[i];
        M = lm;
    }
    int cIndex[NCp];
#pragma unroll
    for (int i = 0; i < NC; i++) cIndex[i] = a.cIndex[i];

    // ---- system scope (PB-SOL:2285-2335)
    if (leader) {
        S& s = sys[lsys];
        if (active) {
            s.TD[0] = a.TD[gsys]; s.TD[1] = a.TD[gsys + NS];
            s.t = a.T[gsys];
            s.dt = a.dt0; s.newDt = a.dt0;
            s.tc = P(0); s.dtP = (P)a.dt0;
            for (int i = 0; i < NSP; i++) s.sPAR[i] = a.sPAR[gsys + i * NS];
            for (int i = 0; i < NSA; i++) s.sACC[i] = a.sACC[gsys + i * NS];
            for (int i = 0; i < NiSA; i++) s.sACCi[i] = a.sACCi[gsys + i * NS];
            for (int i = 0; i < NC; i++) s.strength[i] = a.strength[gsys + i * NS];
            s.DOidx = a.DOidx[gsys];
            s.updDO = 1; s.skipped = 0; s.term = 0; s.udt = 0; s.update = 0; s.doT = P(0);
        } else {
            s.term = 1; s.update = 0; s.updDO = 0;
        }
        s.nacc = 0; s.nrej = 0; s.status = 0;
    }

    // ---- unit scope in registers
    P X[UD], uPAR[Pos<NUP>::value], uACC[Pos<NUA>::value], EF[Pos<NE>::value];
    P Xc[KAHAN ? UD : 1];                 // Kahan compensation of the unit states
    P CPF[NCp];
    int uACCi[Pos<NiUA>::value];
#pragma unroll
    for (int k = 0; k < kUnits; k++) {
        if (exists) {
            const size_t g = gu();
#pragma unroll
            for (int c = 0; c < UD; c++) { X[c] = a.X[g + c * NU]; if (KAHAN) Xc[c] = P(0); }
#pragma unroll
            for (int c = 0; c < NUP; c++) uPAR[c] = a.uPAR[g + c * NU];
#pragma unroll
            for (int c = 0; c < NUA; c++) uACC[c] = a.uACC[g + c * NU];
#pragma unroll
            for (int c = 0; c < NiUA; c++) uACCi[c] = a.uACCi[g + c * NU];
        }
#pragma unroll
        for (int i = 0; i < NC; i++) CPF[i] = P(0);
    }
    __syncthreads();

    // the step size as the user callbacks see it (FP32 copy in the Kahan mode)
    auto udt = [&]() -> P& {
        if constexpr (KAHAN) return my->dtP;
        else return my->dt;
    };
#define MPGOS_PB_USER(TT, DTT) TT, DTT, my->TD, X, uPAR, my->sPAR, gPAR, gPARi, uACC, uACCi, my->sACC, my->sACCi
    // ---- initialisation (PB-SOL:2465-2528)
    if (active) Sys::template Initialization<P>(gsys, u, my->DOidx, MPGOS_PB_USER(my->t, udt()));
    __syncthreads();
    if (NE > 0) {
        if (active) Sys::template EventFunction<P>(gsys, u, EF, MPGOS_PB_USER(my->t, udt()));
        __syncthreads();
    }
    if (a.NDO > 0) {
        // first store (the reference stores unconditionally; skipped once the buffer is full)
        if (active && my->DOidx < a.NDO) {
            const int k = my->DOidx;
#pragma unroll
            for (int c = 0; c < UD; c++) a.DOx[gu() + c * NU + (size_t)k * NU * UD] = X[c];
            if (leader) a.DOt[gsys + (size_t)k * NS] = my->t;
        }
        __syncthreads();
        if (leader && active && my->DOidx < a.NDO) {
            my->DOidx++;
            my->skipped = 0;
            my->doT = dmin<P>(my->t + a.doMinDt, my->TD[1]);
        }
        __syncthreads();
    }

    if (REC && active) {        // checkpoint 0: the initial unit states
#pragma unroll
        for (int c = 0; c < UD; c++) a.recX[(size_t)c * NU + gu()] = X[c];
    }

    int buf = 0;
    // right-hand sides of this lane's pair at (Y, T), then the coupling terms
    auto rhs = [&](P* F, P* Y, const P T) {
        const bool run = lane && my->term == 0;
        P* cpt = cptBuf + (size_t)buf * cptStride;
        if (run)
            Sys::template OdeFunction<P>(gsys, u, F, Y, T, uPAR, my->sPAR, gPAR, gPARi, uACC, uACCi, my->sACC, my->sACCi,
                                         cpt + (size_t)(lsys * UPS + u) * NCp, CPF);
        __syncthreads();
        if (run) U::template couple<GROUPED>(a, M, cIndex, my->strength, cpt + (size_t)lsys * UPS * NCp, u, CPF, F);
        buf ^= 1;
    };

    for (;;) {
        // ---- step initialisation (PB-SOL:2535-2549)
        if (leader && my->term == 0) {
            my->update = 1; my->isfin = 1; my->end = 0;
            my->dt = my->newDt;
            CP remaining;
            if (KAHAN) remaining = (CP)my->TD[1] - ((CP)my->t - (CP)my->tc);
            else remaining = my->TD[1] - my->t;
            if (my->dt > remaining) { my->dt = remaining; my->end = 1; }
            if (KAHAN) my->dtP = (P)my->dt;
            my->ratioBits = order_bits<CP>(CP(1e30));
            my->eventBits = ~0ull;            // no candidate yet (above every finite step)
            my->corrected = 0;
        }
        __syncthreads();
        const P h = (P)my->dt, t = my->t;
        P next[UD], inc[KAHAN ? UD : 1];
        CP err[UD];
        bool isfin = true;
        if (ALG == MPGOS_RK4) {
            // PB-STP:2016-2224
            P k[UD], Y[UD];
            rhs(next, X, t);
#pragma unroll
            for (int c = 0; c < UD; c++) Y[c] = fma(next[c] * P(0.5), h, X[c]);
            const P t2 = t + P(0.5) * h;
            rhs(k, Y, t2);
#pragma unroll
            for (int c = 0; c < UD; c++) { next[c] = fma(P(2), k[c], next[c]); Y[c] = fma(k[c] * P(0.5), h, X[c]); }
            rhs(k, Y, t2);
#pragma unroll
            for (int c = 0; c < UD; c++) { next[c] = fma(P(2.0), k[c], next[c]); Y[c] = fma(k[c], h, X[c]); }
            rhs(k, Y, t + h);
#pragma unroll
            for (int c = 0; c < UD; c++) {
                if (KAHAN) { inc[c] = h * (next[c] + k[c]) * P(1.0 / 6.0); next[c] = X[c] + inc[c]; }
                else next[c] = fma(h * (next[c] + k[c]), P(1.0 / 6.0), X[c]);
                if (!math::isfinite(next[c])) isfin = false;
            }
        } else {
            // PB-STP:2227-2544
            P k1[UD], k2[UD], k3[UD], k4[UD], k5[UD], k6[UD], Y[UD];
            rhs(k1, X, t);
#pragma unroll
            for (int c = 0; c < UD; c++) Y[c] = fma(k1[c] * P(1.0 / 5.0), h, X[c]);
            rhs(k2, Y, fma(P(1.0 / 5.0), h, t));
#pragma unroll
            for (int c = 0; c < UD; c++) Y[c] = fma(fma(k2[c], P(9.0 / 40.0), k1[c] * P(3.0 / 40.0)), h, X[c]);
            rhs(k3, Y, fma(P(3.0 / 10.0), h, t));
#pragma unroll
            for (int c = 0; c < UD; c++)
                Y[c] = fma(fma(k3[c], P(6.0 / 5.0), fma(k2[c], P(-9.0 / 10.0), k1[c] * P(3.0 / 10.0))), h, X[c]);
            rhs(k4, Y, fma(P(3.0 / 5.0), h, t));
#pragma unroll
            for (int c = 0; c < UD; c++)
                Y[c] = fma(fma(k4[c], P(35.0 / 27.0), fma(k3[c], P(-70.0 / 27.0), fma(k2[c], P(5.0 / 2.0),
                              k1[c] * P(-11.0 / 54.0)))), h, X[c]);
            rhs(k5, Y, t + h);
#pragma unroll
            for (int c = 0; c < UD; c++)
                Y[c] = fma(fma(k5[c], P(253.0 / 4096.0), fma(k4[c], P(44275.0 / 110592.0), fma(k3[c], P(575.0 / 13824.0),
                              fma(k2[c], P(175.0 / 512.0), k1[c] * P(1631.0 / 55296.0))))), h, X[c]);
            rhs(k6, Y, fma(P(7.0 / 8.0), h, t));
#pragma unroll
            for (int c = 0; c < UD; c++) {
                const P sum = fma(k6[c], P(512.0 / 1771.0), fma(k4[c], P(125.0 / 594.0), fma(k3[c], P(250.0 / 621.0),
                                  k1[c] * P(37.0 / 378.0))));
                if (KAHAN) {
                    inc[c] = sum * h;
                    next[c] = X[c] + inc[c];
                    // FP64 error norm over the FP32 stages
                    double e = (double)k1[c] * (37.0 / 378.0 - 2825.0 / 27648.0);
                    e = math::fma((double)k3[c], 250.0 / 621.0 - 18575.0 / 48384.0, e);
                    e = math::fma((double)k4[c], 125.0 / 594.0 - 13525.0 / 55296.0, e);
                    e = math::fma((double)k5[c], 0.0 - 277.0 / 14336.0, e);
                    e = math::fma((double)k6[c], 512.0 / 1771.0 - 1.0 / 4.0, e);
                    err[c] = math::fma((double)h, math::fabs(e), 1e-18);
                } else {
                    next[c] = fma(sum, h, X[c]);
                    P e = k1[c] * P(37.0 / 378.0 - 2825.0 / 27648.0);
                    e = fma(k3[c], P(250.0 / 621.0 - 18575.0 / 48384.0), e);
                    e = fma(k4[c], P(125.0 / 594.0 - 13525.0 / 55296.0), e);
                    e = fma(k5[c], P(0.0 - 277.0 / 14336.0), e);
                    e = fma(k6[c], P(512.0 / 1771.0 - 1.0 / 4.0), e);
                    err[c] = (CP)fma(h, math::fabs(e), P(1e-18));
                }
                if (!math::isfinite(next[c]) || !math::isfinite(err[c])) isfin = false;
            }
        }
        if (lane && my->term == 0 && !isfin) my->isfin = 0;
        // ---- controller (PB-CTL:424-542)
        if (ALG == MPGOS_RKCK45) {
            const bool part = lane && my->term == 0;
            if (part) {
                CP R = CP(1e30);
                int upd = 1;
#pragma unroll
                for (int c = 0; c < UD; c++) {
                    const CP tol = dmax<CP>(a.rtol[c] * dmax<CP>(math::fabs((CP)next[c]), math::fabs((CP)X[c])), a.atol[c]);
                    upd = upd & (err[c] < tol);
                    R = dmin<CP>(R, tol / err[c]);
                }
                atomicAnd(&my->update, upd);
                atomicMin(&my->ratioBits, order_bits<CP>(R));
            }
            __syncthreads();
            if (leader && my->term == 0) {
                const CP R = from_order_bits<CP>(my->ratioBits);
                CP fac = CP(0.8) * math::pow_ctrl(R, my->update == 1 ? CP(1.0 / 5.0) : CP(1.0 / 4.0));
                if (!math::isfinite(fac)) my->isfin = 0;
                if (my->isfin == 0) {
                    fac = a.shrink;
                    my->update = 0;
                    if (my->dt < a.dtmin * CP(1.01)) { my->term = 1; my->status |= MPGOS_STATUS_NONFINITE_MIN_STEP; }
                } else if (my->dt < a.dtmin * CP(1.01)) {
                    my->update = 1;
                    my->status |= MPGOS_STATUS_MIN_STEP_REACHED;
                }
                fac = dmin<CP>(fac, a.grow);
                fac = dmax<CP>(fac, a.shrink);
                CP nd = my->dt * fac;
                nd = dmin<CP>(nd, a.dtmax);
                nd = dmax<CP>(nd, a.dtmin);
                my->newDt = nd;
            }
        } else {
            __syncthreads();
            if (leader && my->term == 0) {
                if (my->isfin == 0) { my->term = 1; my->update = 0; my->status |= MPGOS_STATUS_NONFINITE_RK4; }
                my->newDt = a.dt0;
            }
        }
        __syncthreads();
        // ---- events (PB-SOL:2618-2655, PB-EVT:215-268)
        P EFn[Pos<NE>::value];
        if (NE > 0) {
            const P tn = my->t + (P)my->dt;
            if (lane && my->term == 0) {
                bool corr = false;
                CP ev = my->dt;
#pragma unroll
                for (int k = 0; k < kUnits; k++) {
                    // the event function of the candidate state, at the end of the step
                    Sys::template EventFunction<P>(gsys, u, EFn, tn, (P)my->newDt, my->TD, next, uPAR, my->sPAR, gPAR,
                                                   gPARi, uACC, uACCi, my->sACC, my->sACCi);
                    if (my->update == 1) {
#pragma unroll
                        for (int i = 0; i < NE; i++) {
                            const P tol = a.etol[i];
                            if ((EF[i] > tol && EFn[i] < -tol && a.edir[i] <= 0) ||
                                (EF[i] < -tol && EFn[i] > tol && a.edir[i] >= 0)) {
                                ev = dmin<CP>(ev, -(CP)EF[i] / ((CP)EFn[i] - (CP)EF[i]) * my->dt);
                                corr = true;
                            }
                        }
                    }
                }
                if (corr) {
                    atomicMin(&my->eventBits, order_bits<CP>(ev));
                    atomicOr(&my->corrected, 1);
                }
            }
            __syncthreads();
            if (leader && my->corrected == 1) {
                const CP ev = dmin<CP>(my->dt, from_order_bits<CP>(my->eventBits));   // corrected: one candidate at least
                if (ev < a.dtmin) my->status |= MPGOS_STATUS_EVENT_OMITTED;
                else { my->newDt = ev; my->update = 0; }
            }
            __syncthreads();
        }
        // ---- update (PB-SOL:2670-2681)
        const int upd = my->update;
        if (lane && upd == 1) {
#pragma unroll
            for (int c = 0; c < UD; c++) {
                if (KAHAN) {   // compensated x += inc
                    const P y = inc[c] - Xc[c];
                    const P sx = X[c] + y;
                    Xc[c] = (sx - X[c]) - y;
                    X[c] = sx;
                } else {
                    X[c] = next[c];
                }
            }
            if (REC) {
                const long long n = my->nacc;            // accepted steps before this one
                if (leader) {
                    if (n < a.recStepCap) { a.recT[(size_t)n * NS + gsys] = my->t; a.recH[(size_t)n * NS + gsys] = my->dt; }
                    else my->status |= MPGOS_STATUS_CHECKPOINT_OVERFLOW;
                }
                if ((n + 1) % a.recK == 0) {       // once per accepted step of the block, not per stage
                    const long long k = (n + 1) / a.recK;
                    if (k < a.recCkCap) {
#pragma unroll
                        for (int c = 0; c < UD; c++) a.recX[((size_t)k * UD + c) * NU + gu()] = X[c];
                    } else if (leader) {
                        my->status |= MPGOS_STATUS_CHECKPOINT_OVERFLOW;
                    }
                }
            }
        }
        __syncthreads();
        if (leader && upd == 1) {
            if (KAHAN) {   // compensated t += dt
                const P y = (P)my->dt - my->tc;
                const P st = my->t + y;
                my->tc = (st - my->t) - y;
                my->t = st;
            } else {
                my->t += my->dt;
            }
        }
        __syncthreads();
        if (lane && upd == 1) {
            Sys::template ActionAfterSuccessfulTimeStep<P>(gsys, u, my->udt, MPGOS_PB_USER(my->t, udt()));
        }
        __syncthreads();
        if (NE > 0) {
            if (lane && upd == 1) {
#pragma unroll
                for (int i = 0; i < NE; i++) {
                    const P tol = a.etol[i];
                    if ((EF[i] > tol && math::fabs(EFn[i]) < tol && a.edir[i] <= 0) ||
                        (EF[i] < -tol && math::fabs(EFn[i]) < tol && a.edir[i] >= 0))
                        Sys::template ActionAfterEventDetection<P>(gsys, u, i, my->udt, MPGOS_PB_USER(my->t, udt()));
                }
            }
            __syncthreads();
            if (lane && upd == 1) {
                Sys::template EventFunction<P>(gsys, u, EFn, MPGOS_PB_USER(my->t, (P)my->newDt));
            }
            __syncthreads();
            if (lane && upd == 1) {
#pragma unroll
                for (int i = 0; i < NE; i++) EF[i] = EFn[i];
            }
        }
        // ---- dense output (PB-DO:312-395)
        if (a.NDO > 0) {
            if (leader) {
                if (upd == 1) {
                    int st = (my->DOidx < a.NDO && my->doT < my->t && my->skipped >= a.doFreq - 1) ? 1 : 0;
                    if (my->DOidx < a.NDO && (my->end == 1 || my->udt == 1)) st = 1;
                    my->updDO = st;
                } else {
                    my->updDO = 0;
                }
            }
            __syncthreads();
            if (lane && my->updDO == 1 && upd == 1) {
                const int k = my->DOidx;
#pragma unroll
                for (int c = 0; c < UD; c++) a.DOx[gu() + c * NU + (size_t)k * NU * UD] = X[c];
                if (leader) a.DOt[gsys + (size_t)k * NS] = my->t;
            }
            __syncthreads();
            if (leader && upd == 1) {
                if (my->updDO == 1) {
                    my->DOidx++;
                    my->skipped = 0;
                    my->doT = dmin<P>(my->t + a.doMinDt, my->TD[1]);
                } else {
                    my->skipped++;
                }
            }
        }
        // ---- statistics and termination (PB-SOL:2797-2807)
        if (leader && my->term == 0) {
            if (upd == 1) {
                my->nacc++;
                if (my->end == 1 || my->udt == 1) { my->term = 1; my->update = 0; }
            } else {
                my->nrej++;
            }
        }
        __syncthreads();
        int done = 1;
        for (int q = 0; q < SPB; q++) done &= sys[q].term;
        if (done) break;
        __syncthreads();
    }
    __syncthreads();
    // ---- finalisation and write-back (PB-SOL:2814-2887)
    if (active) {
        Sys::template Finalization<P>(gsys, u, my->DOidx, MPGOS_PB_USER(my->t, udt()));
    }
    __syncthreads();
    if (exists) {
        const size_t g = gu();
#pragma unroll
        for (int c = 0; c < UD; c++) a.X[g + c * NU] = X[c];
#pragma unroll
        for (int c = 0; c < NUA; c++) a.uACC[g + c * NU] = uACC[c];
#pragma unroll
        for (int c = 0; c < NiUA; c++) a.uACCi[g + c * NU] = uACCi[c];
    }
    if (leader && active) {
        S& s = sys[lsys];
        a.T[gsys] = s.t;
        a.TD[gsys] = s.TD[0]; a.TD[gsys + NS] = s.TD[1];
        for (int i = 0; i < NSA; i++) a.sACC[gsys + i * NS] = s.sACC[i];
        for (int i = 0; i < NiSA; i++) a.sACCi[gsys + i * NS] = s.sACCi[i];
        a.DOidx[gsys] = s.DOidx;
        a.nacc[gsys] = s.nacc;
        a.nrej[gsys] = s.nrej;
        a.status[gsys] = s.status;
    }
#undef MPGOS_PB_USER
}

// Lane-per-pair form (GROUPED: a kernel of its own for the full matrices that sum
// their columns in groups); MAXT bounds the block size so that blocks of up to 256
// threads get the larger register budget.
template <class Sys, class P, int ALG, int MAXT, bool GROUPED, bool KAHAN = false>
__global__ void __launch_bounds__(MAXT) pb_kernel(Args<Sys, P, typename SysScope<Sys, P, KAHAN>::CP> a)
{
    pb_body<Sys, P, ALG, GROUPED, false, KAHAN>(a);
}

// Record pass of the discrete adjoint (FP64): the forward integration plus
// checkpoints.
template <class Sys, int ALG, int MAXT, bool GROUPED>
__global__ void __launch_bounds__(MAXT) pb_record_kernel(Args<Sys, double> a)
{
    pb_body<Sys, double, ALG, GROUPED, true>(a);
}

} // namespace pb
} // namespace mpgos
