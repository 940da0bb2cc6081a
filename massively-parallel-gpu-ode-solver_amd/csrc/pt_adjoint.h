// Discrete adjoint of the per-thread RK4 / RKCK45 integration (FP64).
//
// No counterpart in the reference: it differentiates the map the reference's
// solver computes (SourceCodes/SingleSystem_PerThread_Solver.cuh:197-394 with
// the steppers of SingleSystem_PerThread_ExplicitRungeKutta_Steppers.cuh),
// taking the accepted step sizes as given (the error controller and event step
// control are not differentiated -- "frozen" step sequence).
//
// Record pass (record_body): the ordinary lane loop, plus a checkpoint
// (x, t, proposed dt, event-function values, accessories and integer
// accessories) before accepted step 0 and after every K-th accepted step, SoA
// in HBM: ckpt[((k*(SD+2+NE+NA+NIA)) + c)*NT + i].  The reverse pass restores
// the accessories with the state, so callbacks and right-hand sides that read
// them replay the recorded values; control parameters and time domains are
// taken as the Solve left them (callbacks that change them during a Solve are
// outside what the adjoint differentiates).
// Reverse pass (reverse_body), one lane per instance, segments last to first:
//   1. restore the segment's checkpoint and re-run the same adaptive loop
//      (controller, rejections and all) -- identical arithmetic, so the same
//      accepted steps -- storing (x_n, t_n, h_n) of each accepted step in a
//      per-lane segment buffer, in LDS when K segment records of the
//      workgroup fit there (per wavefront: lds[(j*(SD+2) + c)*64 + lane]: the records
//      never leave the compute unit), else in HBM seg[((j*(SD+2)) + c)*NT + i],
//      j < K;
//   2. walk the segment backwards (while the next segment down is re-stepped
//      into the record slots already read: two independent chains in one
//      loop body, see reverse_body): recompute the step's stage values from x_n
//      and propagate the adjoint through the stages with the system's
//      vector-Jacobian product (Sys::OdeVJP):
//        x_{n+1} = x_n + h sum_j b_j k_j,  k_j = f(y_j, t_n + c_j h),
//        y_j = x_n + h sum_{l<j} a_jl k_l
//      kb_j = h b_j lam';  for j = s..1: (gy, gp) = VJP(kb_j at y_j);
//      lam += gy; mu += gp; kb_l += h a_jl gy (l < j);  lam_n = lam' + sum gy.
// Event step control is replayed as recorded (the event values are part of
// the checkpoint), so shortened steps recur; user actions at events are not
// differentiated.  Cost per accepted step: one forward step (recompute) +
// stage recompute + one VJP per stage; memory: NT * ceil(N/K) * (SD+2+NE+NA+NIA)
// doubles of checkpoints plus K * (SD+2) doubles of segment records per lane
// (LDS, or HBM when they do not fit).
#pragma once

#include "pt_device.h"

namespace mpgos {
namespace pt {

constexpr int MPGOS_STATUS_CHECKPOINT_OVERFLOW_BIT = 16;

template <class Sys>
struct AdjArgs {
    Args<Sys, double, double> a;   // forward buffers and options (NDO and event log disabled in the reverse pass)
    double* ckpt;
    double* seg;
    double* lam;                   // in: dL/dx(T); out: dL/dx(0)      [SD][NT]
    double* gp;                    // out: dL/dcPAR                    [NCP][NT]
    int K;
    int ckcap;
};

template <class Sys>
constexpr int checkpoint_words() { return Sys::SD + 2 + Sys::NE + Sys::NA + Sys::NIA; }

template <class Sys, int ALG>
__device__ __forceinline__ void store_checkpoint(const AdjArgs<Sys>& A, const Lane<Sys, double, false, ALG>& L, int k)
{
    constexpr int SD = Sys::SD, NE = Sys::NE;
    const int NT = A.a.NT;
    const size_t base = (size_t)k * checkpoint_words<Sys>();
#pragma unroll
    for (int c = 0; c < SD; c++) A.ckpt[(base + c) * NT + L.tid] = L.X[c];
    A.ckpt[(base + SD) * NT + L.tid] = L.t;
    A.ckpt[(base + SD + 1) * NT + L.tid] = L.newDt;
#pragma unroll
    for (int e = 0; e < NE; e++) A.ckpt[(base + SD + 2 + e) * NT + L.tid] = L.EF[e];
#pragma unroll
    for (int i = 0; i < Sys::NA; i++) A.ckpt[(base + SD + 2 + NE + i) * NT + L.tid] = L.ACC[i];
#pragma unroll
    for (int i = 0; i < Sys::NIA; i++) A.ckpt[(base + SD + 2 + NE + Sys::NA + i) * NT + L.tid] = (double)L.ACCi[i];
}

template <class Sys, int ALG, int GROUP>
__device__ __forceinline__ void record_body(const AdjArgs<Sys>& A)
{
    static_assert(offsetof(AdjArgs<Sys>, a) == 0, "Lane's rare paths read the Args at the start of the kernel arguments");
    const Args<Sys, double, double>& a = A.a;
    double* sPAR; int* sPARi;
    stage_shared(a, sPAR, sPARi);
    const int tid = threadIdx.x / GROUP + blockIdx.x * (blockDim.x / GROUP);
    const bool stores = GROUP == 1 || threadIdx.x % GROUP == 0;
    using L_t = Lane<Sys, double, false, ALG>;
    L_t L;
    typename L_t::C c(a, ALG == MPGOS_RKCK45);
    if constexpr (GROUP > 1) c.template set_nodes<GROUP>();
    int untilCk = A.K, k = 0;      // accepted steps to the next checkpoint (no division in the loop)
    if (tid < a.nActive) {
        L.load(a, tid, sPAR, sPARi);
        if (stores) store_checkpoint<Sys, ALG>(A, L, 0);
    } else {
        L.idle();
    }
    if constexpr (L_t::kCommonTime) {
        // checkpoints fall on the same step in every lane of the wavefront
        auto at = [&] {
            ++k;
            if (L.term == 0 && tid < a.nActive) {
                if (k < A.ckcap) store_checkpoint<Sys, ALG>(A, L, k);
                else L.status |= MPGOS_STATUS_CHECKPOINT_OVERFLOW_BIT;
            }
        };
        if ((blockDim.x & 63) == 0) {
            if (a.NDO > 0) L.template run_common_time<true>(c, sPAR, sPARi, A.K, untilCk, at);
            else L.template run_common_time<false>(c, sPAR, sPARi, A.K, untilCk, at);
        }
    }
    if (tid >= a.nActive) return;
    constexpr bool CARRY = L_t::NTT > 0 && GROUP == 1;
    double tt[Pos<L_t::NTT>::value];
    if (CARRY) L.time_terms(L.t, tt);
    bool ended = L.term != 0, accepted;
    while (!ended) {
        ended = L.template step<true, CARRY, GROUP>(c, sPAR, sPARi, accepted, tt);
        if (accepted && --untilCk == 0) {
            untilCk = A.K;
            ++k;
            if (!ended) {
                if (k >= A.ckcap) L.status |= MPGOS_STATUS_CHECKPOINT_OVERFLOW_BIT;
                else if (stores) store_checkpoint<Sys, ALG>(A, L, k);
            }
        }
    }
    if (stores) L.finish(a, sPAR, sPARi);
}

// ---------------------------------------------------------------- reverse steps
// TT: with the time terms tt at T
template <class Sys, bool TT = false>
struct Vjp {
    static constexpr int SD = Sys::SD, NCP = Sys::NCP;
    template <int NCPA>
    static __device__ __forceinline__ void apply(int tid, int NT, const double* kb, double* y, double T, double* cPAR,
                                                 double* sPAR, int* sPARi, double* ACC, int* ACCi, double* lam, double* mu,
                                                 double* gy, const double* tt = nullptr)
    {
        double gp[NCPA];
        if constexpr (TT) Sys::template OdeVJPTT<double>(tid, NT, kb, y, T, tt, cPAR, sPAR, sPARi, ACC, ACCi, gy, gp);
        else Sys::template OdeVJP<double>(tid, NT, kb, y, T, cPAR, sPAR, sPARi, ACC, ACCi, gy, gp);
#pragma unroll
        for (int c = 0; c < SD; c++) lam[c] += gy[c];
#pragma unroll
        for (int c = 0; c < NCP; c++) mu[c] += gp[c];
    }
};

// RK4 (stages as in Lane::rk4).  lam: in dL/dx_{n+1}, out dL/dx_n.  TT: with
// the time terms at t, t + h/2 and t + h.
template <class Sys, bool TT = false>
__device__ __forceinline__ void reverse_rk4(int tid, int NT, const double* x, double t, double h, double* cPAR, double* sPAR,
                                            int* sPARi, double* ACC, int* ACCi, double* lam, double* mu,
                                            const double* tt1 = nullptr, const double* ttm = nullptr, const double* tt4 = nullptr)
{
    using math::fma;
    constexpr int SD = Sys::SD, NCPA = Pos<Sys::NCP>::value;
    double k[SD], y2[SD], y3[SD], y4[SD], xx[SD];
#pragma unroll
    for (int c = 0; c < SD; c++) xx[c] = x[c];
    const double half = 0.5 * h;
    const double sixth = (1.0 / 6.0) * h;
    const double T2 = t + half, T4 = t + h;
    auto ode = [&](double* F, double* Y, double T, const double* tt) {
        if constexpr (TT) Sys::template OdeFunctionTT<double>(tid, NT, F, Y, T, tt, cPAR, sPAR, sPARi, ACC, ACCi);
        else Sys::template OdeFunction<double>(tid, NT, F, Y, T, cPAR, sPAR, sPARi, ACC, ACCi);
    };
    ode(k, xx, t, tt1);
#pragma unroll
    for (int c = 0; c < SD; c++) y2[c] = fma(k[c], half, xx[c]);
    ode(k, y2, T2, ttm);
#pragma unroll
    for (int c = 0; c < SD; c++) y3[c] = fma(k[c], half, xx[c]);
    ode(k, y3, T2, ttm);
#pragma unroll
    for (int c = 0; c < SD; c++) y4[c] = fma(k[c], h, xx[c]);

    double kb[SD], gy[SD], lo[SD];
#pragma unroll
    for (int c = 0; c < SD; c++) lo[c] = lam[c];
    // stage 4 (weight 1/6)
#pragma unroll
    for (int c = 0; c < SD; c++) kb[c] = sixth * lo[c];
    Vjp<Sys, TT>::template apply<NCPA>(tid, NT, kb, y4, T4, cPAR, sPAR, sPARi, ACC, ACCi, lam, mu, gy, tt4);
    // stage 3 (weight 2/6, plus h * dy4/dk3)
#pragma unroll
    for (int c = 0; c < SD; c++) kb[c] = fma(2.0 * sixth, lo[c], h * gy[c]);
    Vjp<Sys, TT>::template apply<NCPA>(tid, NT, kb, y3, T2, cPAR, sPAR, sPARi, ACC, ACCi, lam, mu, gy, ttm);
    // stage 2
#pragma unroll
    for (int c = 0; c < SD; c++) kb[c] = fma(2.0 * sixth, lo[c], half * gy[c]);
    Vjp<Sys, TT>::template apply<NCPA>(tid, NT, kb, y2, T2, cPAR, sPAR, sPARi, ACC, ACCi, lam, mu, gy, ttm);
    // stage 1
#pragma unroll
    for (int c = 0; c < SD; c++) kb[c] = fma(sixth, lo[c], half * gy[c]);
    Vjp<Sys, TT>::template apply<NCPA>(tid, NT, kb, xx, t, cPAR, sPAR, sPARi, ACC, ACCi, lam, mu, gy, tt1);
}

// Cash-Karp (stages as in Lane::rkck45, 5th-order weights b).  Time terms are
// evaluated once per stage, with several lanes per instance (GROUP, node) once or
// twice per step.
template <class Sys, int GROUP>
__device__ __forceinline__ void reverse_rkck45(int tid, int NT, const double* x, double t, double h, double* cPAR,
                                               double* sPAR, int* sPARi, double* ACC, int* ACCi, double* lam, double* mu,
                                               const double* node)
{
    constexpr bool TT = TimeTermsOf<Sys>::timeOnly;
    constexpr int NTT = TimeTermsOf<Sys>::n;
    using math::fma;
    constexpr int SD = Sys::SD, NCPA = Pos<Sys::NCP>::value;
    constexpr double a21 = 1.0 / 5.0;
    constexpr double a31 = 3.0 / 40.0, a32 = 9.0 / 40.0;
    constexpr double a41 = 3.0 / 10.0, a42 = -9.0 / 10.0, a43 = 6.0 / 5.0;
    constexpr double a51 = -11.0 / 54.0, a52 = 5.0 / 2.0, a53 = -70.0 / 27.0, a54 = 35.0 / 27.0;
    constexpr double a61 = 1631.0 / 55296.0, a62 = 175.0 / 512.0, a63 = 575.0 / 13824.0, a64 = 44275.0 / 110592.0,
                     a65 = 253.0 / 4096.0;
    constexpr double b1 = 37.0 / 378.0, b3 = 250.0 / 621.0, b4 = 125.0 / 594.0, b6 = 512.0 / 1771.0;

    double y[6][SD], k[5][SD];
    const double T[6] = {t, fma(h, 1.0 / 5.0, t), fma(h, 3.0 / 10.0, t), fma(h, 3.0 / 5.0, t), t + h, fma(h, 7.0 / 8.0, t)};
    double tt[6][Pos<NTT>::value];
    if constexpr (TT && GROUP > 1) {
        double all[group_evals<GROUP>()][Pos<NTT>::value];
#pragma unroll
        for (int e = 0; e < group_evals<GROUP>(); e++) Sys::template TimeTerms<double>(fma(h, node[e], t), cPAR, all[e]);
        auto take = [&](auto J) {
#pragma unroll
            for (int i = 0; i < NTT; i++) tt[J.value][i] = group_value<GROUP, J.value % GROUP>(all[J.value / GROUP][i]);
        };
        take(std::integral_constant<int, 0>{}); take(std::integral_constant<int, 1>{}); take(std::integral_constant<int, 2>{});
        take(std::integral_constant<int, 3>{}); take(std::integral_constant<int, 4>{}); take(std::integral_constant<int, 5>{});
    } else if constexpr (TT) {
#pragma unroll
        for (int j = 0; j < 6; j++) Sys::template TimeTerms<double>(T[j], cPAR, tt[j]);
    }
    auto ode = [&](double* F, int j) {
        if constexpr (TT) Sys::template OdeFunctionTT<double>(tid, NT, F, y[j], T[j], tt[j], cPAR, sPAR, sPARi, ACC, ACCi);
        else Sys::template OdeFunction<double>(tid, NT, F, y[j], T[j], cPAR, sPAR, sPARi, ACC, ACCi);
    };
    auto vjp = [&](int j, double* kb, double* gy) {
        Vjp<Sys, TT>::template apply<NCPA>(tid, NT, kb, y[j], T[j], cPAR, sPAR, sPARi, ACC, ACCi, lam, mu, gy, tt[j]);
    };
#pragma unroll
    for (int c = 0; c < SD; c++) y[0][c] = x[c];
    ode(k[0], 0);
#pragma unroll
    for (int c = 0; c < SD; c++) y[1][c] = fma(h, a21 * k[0][c], x[c]);
    ode(k[1], 1);
#pragma unroll
    for (int c = 0; c < SD; c++) y[2][c] = fma(h, fma(a32, k[1][c], a31 * k[0][c]), x[c]);
    ode(k[2], 2);
#pragma unroll
    for (int c = 0; c < SD; c++) y[3][c] = fma(h, fma(a43, k[2][c], fma(a42, k[1][c], a41 * k[0][c])), x[c]);
    ode(k[3], 3);
#pragma unroll
    for (int c = 0; c < SD; c++)
        y[4][c] = fma(h, fma(a54, k[3][c], fma(a53, k[2][c], fma(a52, k[1][c], a51 * k[0][c]))), x[c]);
    ode(k[4], 4);
#pragma unroll
    for (int c = 0; c < SD; c++)
        y[5][c] = fma(h, fma(a65, k[4][c], fma(a64, k[3][c], fma(a63, k[2][c], fma(a62, k[1][c], a61 * k[0][c])))), x[c]);

    // adjoints of the stage derivatives, seeded by the output weights
    double kb[6][SD], gy[SD];
#pragma unroll
    for (int c = 0; c < SD; c++) {
        const double hl = h * lam[c];
        kb[0][c] = b1 * hl; kb[1][c] = 0.0; kb[2][c] = b3 * hl; kb[3][c] = b4 * hl; kb[4][c] = 0.0; kb[5][c] = b6 * hl;
    }
    // stage 6 -> contributes to k1..k5
    vjp(5, kb[5], gy);
#pragma unroll
    for (int c = 0; c < SD; c++) {
        const double g = h * gy[c];
        kb[0][c] = fma(a61, g, kb[0][c]); kb[1][c] = fma(a62, g, kb[1][c]); kb[2][c] = fma(a63, g, kb[2][c]);
        kb[3][c] = fma(a64, g, kb[3][c]); kb[4][c] = fma(a65, g, kb[4][c]);
    }
    vjp(4, kb[4], gy);
#pragma unroll
    for (int c = 0; c < SD; c++) {
        const double g = h * gy[c];
        kb[0][c] = fma(a51, g, kb[0][c]); kb[1][c] = fma(a52, g, kb[1][c]); kb[2][c] = fma(a53, g, kb[2][c]);
        kb[3][c] = fma(a54, g, kb[3][c]);
    }
    vjp(3, kb[3], gy);
#pragma unroll
    for (int c = 0; c < SD; c++) {
        const double g = h * gy[c];
        kb[0][c] = fma(a41, g, kb[0][c]); kb[1][c] = fma(a42, g, kb[1][c]); kb[2][c] = fma(a43, g, kb[2][c]);
    }
    vjp(2, kb[2], gy);
#pragma unroll
    for (int c = 0; c < SD; c++) {
        const double g = h * gy[c];
        kb[0][c] = fma(a31, g, kb[0][c]); kb[1][c] = fma(a32, g, kb[1][c]);
    }
    vjp(1, kb[1], gy);
#pragma unroll
    for (int c = 0; c < SD; c++) kb[0][c] = fma(a21, h * gy[c], kb[0][c]);
    vjp(0, kb[0], gy);
}

// LDS bytes of the shared-parameter staging (16-byte aligned); the segment
// records of the LDS form follow.
template <class Sys>
__host__ __device__ constexpr size_t adjoint_shared_bytes(int preferShared)
{
    return preferShared ? (((size_t)Sys::NSP * sizeof(double) + (size_t)Sys::NISP * sizeof(int)) + 15) & ~(size_t)15 : 0;
}

// Reverse pass of a wavefront whose instances share their time (fixed steps,
// Lane::run_common_time): the time terms of a segment's steps come from one
// evaluation per segment, each lane's at another start or middle of a step,
// for the re-step of segment s - 1 and for the differentiation of segment s
// alike, and the records need no times and step sizes.  The last segment,
// whose last step may be clipped, goes the ordinary way.  Called by the whole
// wavefront; returns false, with nothing done, when the lanes' times, ends or
// step counts differ or a segment has more than 31 steps.
// Duffing with a quadrature state, 65536 instances x 32000 steps, K = 16 (one
// wavefront per SIMD, bound by the instructions of a step): 407 -> 174
// instructions per step, 26.1 -> 13.2 ms.
template <class Sys, int ALG, bool LDS_SEG, class Seg, class Restore, class Attempt, class Keep, class Back>
__device__ __forceinline__ bool common_time_reverse(const AdjArgs<Sys>& A, Lane<Sys, double, false, ALG>& L, bool mine, bool ok,
                                                    long long total, double* lam, double* mu, Seg& seg, double* sPAR, int* sPARi,
                                                    Restore& restore, Attempt& attempt, Keep& keep, Back& back, double* bPAR,
                                                    double* bACC, int* bACCi)
{
    constexpr int SD = Sys::SD, NTT = Lane<Sys, double, false, ALG>::NTT;
    const typename Lane<Sys, double, false, ALG>::C a(A.a, false);
    const int K = A.K;
    if ((blockDim.x & 63) != 0 || K > 31 || !(a.dt0 > 0.0)) return false;
    const uint64_t live = __ballot(mine);
    if (live == 0 || !__all(!mine || ok)) return false;
    const int first = __builtin_ctzll(live);
    const int steps = __builtin_amdgcn_readlane((int)total, first);
    if (!__all(!mine || total == (long long)steps)) return false;
    const int nseg = (steps + K - 1) / K;
    if (nseg < 2) return false;
    if (mine) restore(0);
    else { L.t = 0.0; L.newDt = 0.0; }
    const double h = a.dt0, half = 0.5 * h;
    const bool same = math::bits(L.t) == math::bits(lane_value(L.t, first)) && math::bits(L.newDt) == math::bits(h) &&
                      math::bits(L.TD[1]) == math::bits(lane_value(L.TD[1], first));
    if (!__all(!mine || same)) return false;

    // the last segment by itself
    if (mine) {
        restore(nseg - 1);
        int have = 0;
        const int cnt = steps - (nseg - 1) * K;
        while (have < cnt && L.term == 0) attempt(false, have);
        keep();
        for (int j = have - 1; j >= 0; j--) back(false, j);
    }
    // the start times (even lanes) of a segment's steps and the time terms at
    // their starts and middles (odd lanes)
    auto terms = [&](double t0, double& tv, double* tt) {
        double none = 0.0;
        tv = t0;
        advance_by_lane(tv, none, h);
        L.time_terms((__lane_id() & 1u) ? tv + half : tv, tt);
    };
    auto at = [&](const double* tt, int l, double* out) {
#pragma unroll
        for (int i = 0; i < NTT; i++) out[i] = lane_value(tt[i], l);
    };
    double tvF, ttF[NTT], tvB, ttB[NTT];
    // re-step j of the restored segment; its start state goes to `slot`
    auto forward = [&](int j, int slot) {
        double tt1[NTT], ttm[NTT], tt4[NTT], nx[SD], EFn[1], dtP = h;
        at(ttF, 2 * j, tt1); at(ttF, 2 * j + 1, ttm); at(ttF, 2 * j + 2, tt4);
#pragma unroll
        for (int c = 0; c < SD; c++)
            if (LDS_SEG || mine) seg((size_t)(slot * SD + c)) = L.X[c];   // HBM records end with the last instance
        L.rk4(a, h, nx, nullptr, sPAR, sPARi, tt1, ttm, tt4);
        L.accept(a, h, dtP, nx, nullptr, EFn, false, sPAR, sPARi);
    };
    // a step's record, read a step ahead of its use (as above: HBM records end
    // with the last instance)
    double x[SD];
    auto record = [&](int slot) {
#pragma unroll
        for (int c = 0; c < SD; c++) x[c] = LDS_SEG || mine ? seg((size_t)(slot * SD + c)) : 0.0;
    };
    auto reverse = [&](int j, int next) {
        double tt1[NTT], ttm[NTT], tt4[NTT], xj[SD];
        at(ttB, 2 * j, tt1); at(ttB, 2 * j + 1, ttm); at(ttB, 2 * j + 2, tt4);
#pragma unroll
        for (int c = 0; c < SD; c++) xj[c] = x[c];
        if (j > 0) record(next);
        reverse_rk4<Sys, true>(L.tid, a.NT, xj, lane_value(tvB, 2 * j), h, bPAR, sPAR, sPARi, bACC, bACCi, lam, mu, tt1, ttm, tt4);
    };
    auto start = [&](int s) {
        if (mine) restore(s);
        terms(lane_value(L.t, first), tvF, ttF);
    };
    bool flip = false;
    start(nseg - 2);
    for (int j = 0; j < K; j++) forward(j, j);
    for (int s = nseg - 2; s > 0; s--) {
        // segment s is in the buffer (step j in slot j, or K - 1 - j when
        // flipped); the re-step of s - 1 writes the slots just read
        if (mine) keep();
        tvB = tvF;
#pragma unroll
        for (int i = 0; i < NTT; i++) ttB[i] = ttF[i];
        start(s - 1);
        const int step = flip ? 1 : -1;
        int m = 0, slot = flip ? 0 : K - 1;
        record(slot);
        auto both = [&](int m, int slot) { reverse(K - 1 - m, slot + step); forward(m, slot); };
        for (; m + 2 <= K; m += 2, slot += 2 * step) { both(m, slot); both(m + 1, slot + step); }
        if (m < K) both(m, slot);
        flip = !flip;
    }
    if (mine) keep();
    tvB = tvF;
#pragma unroll
    for (int i = 0; i < NTT; i++) ttB[i] = ttF[i];
    record(flip ? 0 : K - 1);
    for (int j = K - 1; j >= 0; j--) reverse(j, flip ? K - j : j - 1);
    return true;
}

template <class Sys, int ALG, bool LDS_SEG, int GROUP>
__device__ __forceinline__ void reverse_body(const AdjArgs<Sys>& A)
{
    constexpr int SD = Sys::SD, NCP = Sys::NCP, NA = Sys::NA, NIA = Sys::NIA;
    static_assert(offsetof(AdjArgs<Sys>, a) == 0, "Lane's rare paths read the Args at the start of the kernel arguments");
    const Args<Sys, double, double>& a = A.a;
    double* sPAR; int* sPARi;
    stage_shared(a, sPAR, sPARi);
    using L_t = Lane<Sys, double, false, ALG>;
    constexpr bool COMMON = L_t::kCommonTime && Sys::HAS_VJP;
    const int tid = threadIdx.x / GROUP + blockIdx.x * (blockDim.x / GROUP);
    const bool mine = tid < a.nActive;
    if (!COMMON && !mine) return;      // with COMMON whole wavefronts stay together
    const int NT = a.NT;
    // segment record word w of this lane: in LDS one region per wavefront,
    // word-major with a lane stride of 64 doubles (a record's words are then
    // constant offsets from one address); in HBM word-major over all lanes
    extern __shared__ __align__(16) unsigned char mpgos_dyn_lds[];
    double* const segBase =
        LDS_SEG ? reinterpret_cast<double*>(mpgos_dyn_lds + adjoint_shared_bytes<Sys>(a.preferShared)) +
                      (size_t)(threadIdx.x >> 6) * ((size_t)A.K * (SD + 2) * 64) + (threadIdx.x & 63)
                : A.seg + tid;
    auto seg = [&](size_t w) -> double& {
        if constexpr (LDS_SEG) return segBase[w * 64];
        else return segBase[w * NT];
    };
    const long long total = mine ? a.nacc[tid] : 0;
    double lam[SD], mu[Pos<NCP>::value];
#pragma unroll
    for (int c = 0; c < SD; c++) lam[c] = mine ? A.lam[c * NT + tid] : 0.0;
#pragma unroll
    for (int c = 0; c < NCP; c++) mu[c] = 0.0;

    L_t L;
    L.tid = tid;
#pragma unroll
    for (int i = 0; i < 2; i++) L.TD[i] = mine ? a.TD[tid + i * NT] : 0.0;
#pragma unroll
    for (int i = 0; i < NCP; i++) L.cPAR[i] = mine ? a.cPAR[tid + i * NT] : 0.0;

    const bool ok = mine && (a.status[tid] & MPGOS_STATUS_CHECKPOINT_OVERFLOW_BIT) == 0;
    const long long nseg = ok ? (total + A.K - 1) / A.K : 0;
    const int K = A.K;
    typename L_t::C c(a, ALG == MPGOS_RKCK45);
    if constexpr (GROUP > 1) c.template set_nodes<GROUP>();
    constexpr bool CARRY = L_t::NTT > 0 && GROUP == 1;
    double tt[Pos<L_t::NTT>::value];
    // Restore segment s's checkpoint into the lane.
    auto restore = [&](long long s) {
        const size_t cb = (size_t)s * checkpoint_words<Sys>();
#pragma unroll
        for (int c = 0; c < SD; c++) L.X[c] = A.ckpt[(cb + c) * NT + tid];
        L.t = A.ckpt[(cb + SD) * NT + tid];
        L.newDt = A.ckpt[(cb + SD + 1) * NT + tid];
#pragma unroll
        for (int e = 0; e < Sys::NE; e++) L.EF[e] = A.ckpt[(cb + SD + 2 + e) * NT + tid];
#pragma unroll
        for (int i = 0; i < NA; i++) L.ACC[i] = A.ckpt[(cb + SD + 2 + Sys::NE + i) * NT + tid];
#pragma unroll
        for (int i = 0; i < NIA; i++) L.ACCi[i] = (int)A.ckpt[(cb + SD + 2 + Sys::NE + NA + i) * NT + tid];
        L.dt = L.newDt;
        L.tc = 0.0;
        L.term = 0; L.udt = 0; L.nacc = 0; L.nrej = 0; L.status = 0; L.nev = 0;
        L.doIdx = 0; L.skipped = 0; L.doT = 0.0;
        if (CARRY) L.time_terms(L.t, tt);
    };
    // accepted steps of segment s
    auto count = [&](long long s) { return (int)((total - s * K) < K ? (total - s * K) : K); };
    // One record buffer of K slots serves two segments at once: segment s is
    // differentiated (its records read last to first) while segment s - 1 is
    // re-stepped into the slots already read.  Segments alternate the slot
    // order -- step j in slot j, or in slot K - 1 - j -- so that the m-th
    // record written (step m of segment s - 1) goes to the slot the m-th read
    // (step cnt - 1 - m of segment s) has just freed; rejected attempts write
    // nothing, so writes never overtake reads.
    auto slot = [&](bool flip, int j) { return flip ? K - 1 - j : j; };
    // One attempted re-step of the lane; an accepted step stores (x_n, t_n, h_n)
    // of step j in its slot and advances j.
    auto attempt = [&](bool flip, int& j) {
        double xp[SD];
#pragma unroll
        for (int c = 0; c < SD; c++) xp[c] = L.X[c];
        const double tp = L.t;
        bool accepted;
        if (L.template step<false, CARRY, GROUP>(c, sPAR, sPARi, accepted, tt)) L.term = 1;
        if (accepted) {
            const size_t sb = (size_t)slot(flip, j) * (SD + 2);
#pragma unroll
            for (int c = 0; c < SD; c++) seg(sb + c) = xp[c];
            seg(sb + SD) = tp;
            seg(sb + SD + 1) = L.dt;
            j++;
        }
    };
    // Adjoint through step j of the segment whose records use slot order flip,
    // with the parameters and accessories the lane held at the end of that
    // segment's re-step (kept apart while the next segment is re-stepped)
    double bPAR[Pos<NCP>::value], bACC[Pos<NA>::value];
    int bACCi[Pos<NIA>::value];
    auto keep = [&]() {
#pragma unroll
        for (int i = 0; i < NCP; i++) bPAR[i] = L.cPAR[i];
#pragma unroll
        for (int i = 0; i < NA; i++) bACC[i] = L.ACC[i];
#pragma unroll
        for (int i = 0; i < NIA; i++) bACCi[i] = L.ACCi[i];
    };
    auto back = [&](bool flip, int j) {
        const size_t sb = (size_t)slot(flip, j) * (SD + 2);
        double x[SD];
#pragma unroll
        for (int c = 0; c < SD; c++) x[c] = seg(sb + c);
        const double tn = seg(sb + SD), hn = seg(sb + SD + 1);
        if (ALG == MPGOS_RK4)
            reverse_rk4<Sys>(tid, NT, x, tn, hn, bPAR, sPAR, sPARi, bACC, bACCi, lam, mu);
        else
            reverse_rkck45<Sys, GROUP>(tid, NT, x, tn, hn, bPAR, sPAR, sPARi, bACC, bACCi, lam, mu, c.node);
    };
    bool swept = false;
    if constexpr (COMMON) {
        swept = common_time_reverse<Sys, ALG, LDS_SEG>(A, L, mine, ok, total, lam, mu, seg, sPAR, sPARi, restore, attempt, keep,
                                                       back, bPAR, bACC, bACCi);
    }
    if (!mine) return;
    if (!swept && nseg > 0) {
        // the last segment alone
        bool flip = false;
        restore(nseg - 1);
        int have = 0;
        const int cntLast = count(nseg - 1);
        while (have < cntLast && L.term == 0) attempt(flip, have);
        for (long long s = nseg - 1; s >= 0; s--) {
            // `have` records of segment s are in the buffer (slot order flip)
            keep();
            if (s == 0) {
                for (int jj = have - 1; jj >= 0; jj--) back(flip, jj);
                break;
            }
            // segment s - 1 is full (K accepted steps, at least K attempts),
            // so the first `have` <= K iterations always hold one attempt and
            // one adjoint step: two independent chains in one block
            restore(s - 1);
            int next = 0;
            for (int m = 0; m < have; m++) {
                back(flip, have - 1 - m);
                attempt(!flip, next);
            }
            while (next < K && L.term == 0) attempt(!flip, next);
            have = next;
            flip = !flip;
        }
    }
#pragma unroll
    for (int c = 0; c < SD; c++) A.lam[c * NT + tid] = ok ? lam[c] : __builtin_nan("");
#pragma unroll
    for (int c = 0; c < NCP; c++) A.gp[c * NT + tid] = ok ? mu[c] : __builtin_nan("");
}

// GROUP: lanes per instance (Cash-Karp and systems with time terms only, else 1)
template <class Sys, int ALG, int GROUP = 1>
__global__ void __launch_bounds__(kMaxBlock) adjoint_record_kernel(AdjArgs<Sys> A) { record_body<Sys, ALG, GROUP>(A); }

template <class Sys, int ALG, bool LDS_SEG, int GROUP = 1>
__global__ void __launch_bounds__(kMaxBlock) adjoint_reverse_kernel(AdjArgs<Sys> A) { reverse_body<Sys, ALG, LDS_SEG, GROUP>(A); }

} // namespace pt
} // namespace mpgos
