// Discrete adjoint of the per-block RK4 / RKCK45 integration (FP64).
//
// No counterpart in the reference: it differentiates the map the reference's
// per-block solver computes (SourceCodes/CoupledSystmes_PerBlock_Solver.cuh:
// 2214-2888 with the steppers of
// CoupledSystems_PerBlock_ExplicitRungeKutta_Steppers.cuh:2016-2544 and the
// coupling terms at :2634-2713), with the accepted step sizes taken as given
// (frozen step sequence; the error controller and event step control are not
// differentiated; user actions that change the state are not replayed).
//
// Record pass (pb_record_kernel in pb_device.h, pb_dense_kernel): the forward integration
// storing the unit states every K accepted steps and (t_n, h_n) of every
// accepted step.
// Reverse pass (pb_reverse_kernel), lane per (system, unit), SPB systems per
// workgroup, segments last to first:
//   1. restore the segment's checkpoint and recompute its accepted steps with
//      the recorded (t_n, h_n) -- the stage arithmetic of the forward pass, so
//      the states are the recorded ones bit for bit -- keeping the state at
//      the start of each step in a segment buffer seg[(j * UD + c) * NU + unit];
//   2. walk the segment backwards: recompute the step's stage values Y_j,
//      their coupling values v_j and factors CPF_j, and propagate the adjoint
//      through the stages, next = x + h sum_j b_j k_j, Y_j = x + h sum_l a_jl k_l,
//      k_j = F(Y_j) + s CPF_j (M CPT(Y))_j:
//        kb_j = h b_j lam';  for j = s..1:
//          w = s CPF_j kb_j[ci]                       (per unit, into LDS)
//          kbCPT = M^T w,  kbCPF = s v_j kb_j[ci]      (transposed coupling)
//          (gy, gU, gS) = Sys::OdeVJP(kb_j, kbCPT, kbCPF at Y_j)
//          lam += gy;  kb_l += h a_jl gy (l < j);  muU += gU;  muS += gS
// The system-parameter gradient is summed over the units of a system in a
// fixed order at the end (deterministic).  Cost per accepted step: one
// recompute of the step (segment pass) + stage recompute + one transposed
// coupling product and one VJP per stage.
// The dense-contraction form (full FP64 matrix; below) runs the coupling
// products on MFMA and replaces the stage recompute by a stage buffer; it
// returns the same bits as the lane form.
#pragma once

#include "pb_dense.h"

namespace mpgos {
namespace pb {

template <class Sys>
struct AdjArgs {
    double* seg;          // [K][UD][NU] (lane form)
    double* stg;          // [K * rev_rows][NU] stage buffer (dense-contraction form)
    double* gSp;          // [NSP][NU] per-unit partials of dL/d(system parameters) (dense-contraction form)
    double* lam;          // in: dL/dx(end), out: dL/dx(start)      [UD][NU]
    double* gU;           // out: dL/d(unit parameters)             [NUP][NU]
    double* gS;           // out: dL/d(system parameters)           [NSP][NS]
    const double* cMatT;  // transposed coupling matrices in the stored form of cMat
    const double* cTileT; // their pair-tiled copy (dense-contraction form)
};

// sum over the matrix row u of M_i (any storage form) against vals[col * NCp + i]
template <class Sys>
__device__ __forceinline__ double coupling_dot(const Args<Sys, double>& a, const double* M, const double* vals, int u, int i)
{
    constexpr int NCp = Pos<Sys::NC>::value;
    const int UPS = a.UPS;
    double v = 0.0;
    if (a.CCI == 0 && a.CBW == 0) {
        const double* Mi = M + (size_t)i * UPS * UPS + u;
        for (int col = 0; col < UPS; col++) v = math::fma(Mi[(size_t)col * UPS], vals[col * NCp + i], v);
    } else {
        const int W = a.CBW > 0 ? 2 * a.CBW + 1 : UPS;
        for (int d = 0; d < W; d++) {
            int col = u + d - a.CBW;
            if (col >= UPS) col -= UPS;
            if (col < 0) col += UPS;
            const double m = a.CCI == 0 ? M[(size_t)i * UPS * W + u + (size_t)d * UPS] : M[(size_t)i * W + d];
            v = math::fma(m, vals[col * NCp + i], v);
        }
    }
    return v;
}

// System scope of the reverse pass (LDS) and the LDS layout: per-system
// scope, two coupling-term buffers, two adjoint-weight buffers, the
// system-parameter gradient partials, two block-wide counters.
template <class Sys>
struct RevScope {
    double sPAR[Pos<Sys::NSP>::value]; double sACC[Pos<Sys::NSA>::value]; double strength[Pos<Sys::NC>::value];
    int sACCi[Pos<Sys::NiSA>::value];
    long long nacc;
    int nseg, len, k, status;
};
struct RevLayout { size_t cpt, wb, red, blk, total; };

template <class Sys>
__host__ __device__ inline RevLayout reverse_layout(int SPB, int UPS)
{
    constexpr int NCp = Pos<Sys::NC>::value, NSPp = Pos<Sys::NSP>::value;
    RevLayout L;
    size_t o = ((size_t)SPB * sizeof(RevScope<Sys>) + 15) & ~(size_t)15;
    L.cpt = o;
    o += 2 * (size_t)SPB * UPS * NCp * sizeof(double);
    L.wb = o;
    o += 2 * (size_t)SPB * UPS * NCp * sizeof(double);
    L.red = o;
    o += (size_t)SPB * UPS * NSPp * sizeof(double);
    L.blk = o;
    o += 2 * sizeof(int);
    L.total = o;
    return L;
}

template <class Sys, int ALG>
__device__ void pb_reverse_body(const Args<Sys, double>& a, const AdjArgs<Sys>& A)
{
    using P = double;
    constexpr int UD = Sys::UD, NC = Sys::NC, NUP = Sys::NUP, NSP = Sys::NSP, NGP = Sys::NGP, NiGP = Sys::NiGP;
    constexpr int NUA = Sys::NUA, NiUA = Sys::NiUA, NSA = Sys::NSA, NiSA = Sys::NiSA;
    constexpr int NCp = Pos<NC>::value, NUPp = Pos<NUP>::value, NSPp = Pos<NSP>::value;
    constexpr int ST = ALG == MPGOS_RK4 ? 4 : 6;       // stages
    using math::fma;

    using Scope = RevScope<Sys>;
    extern __shared__ __align__(16) unsigned char mpgos_pb_lds[];
    const int UPS = a.UPS, NS = a.NS, SPB = a.SPB, K = a.recK;
    const RevLayout L = reverse_layout<Sys>(SPB, UPS);
    Scope* sys = reinterpret_cast<Scope*>(mpgos_pb_lds);
    P* cpt = reinterpret_cast<P*>(mpgos_pb_lds + L.cpt);
    P* wb = reinterpret_cast<P*>(mpgos_pb_lds + L.wb);
    P* red = reinterpret_cast<P*>(mpgos_pb_lds + L.red);            // [SPB][UPS][NSPp]
    int* blk = reinterpret_cast<int*>(mpgos_pb_lds + L.blk);         // [0] rounds, [1] longest segment
    const int stride = SPB * UPS * NCp;

    const int tid = threadIdx.x;
    const int lsys = tid / UPS;
    const int u = tid - lsys * UPS;
    const bool lane = lsys < SPB;
    const bool leader = lane && u == 0;
    const int gsys = blockIdx.x * SPB + lsys;
    const bool active = lane && gsys < a.nActive && gsys < NS;
    const size_t NU = (size_t)NS * UPS;
    const size_t gu = (size_t)gsys * UPS + u;
    Scope* my = lane ? &sys[lsys] : &sys[0];

    int cIndex[NCp];
#pragma unroll
    for (int i = 0; i < NC; i++) cIndex[i] = a.cIndex[i];
    if (tid < 2) blk[tid] = 0;
    if (leader) {
        my->status = 0;
        my->nseg = 0;
        if (active) {
            for (int i = 0; i < NSP; i++) my->sPAR[i] = a.sPAR[gsys + i * NS];
            for (int i = 0; i < NSA; i++) my->sACC[i] = a.sACC[gsys + i * NS];
            for (int i = 0; i < NiSA; i++) my->sACCi[i] = a.sACCi[gsys + i * NS];
            for (int i = 0; i < NC; i++) my->strength[i] = a.strength[gsys + i * NS];
            my->nacc = a.nacc[gsys];
            my->status = a.status[gsys];
            const bool ok = (my->status & MPGOS_STATUS_CHECKPOINT_OVERFLOW) == 0;
            my->nseg = ok ? (int)((my->nacc + K - 1) / K) : 0;
        }
    }
    P uPAR[NUPp], uACC[Pos<NUA>::value], lam[UD], muU[NUPp], muS[NSPp];
    int uACCi[Pos<NiUA>::value];
#pragma unroll
    for (int c = 0; c < NUP; c++) { uPAR[c] = active ? a.uPAR[gu + c * NU] : P(0); muU[c] = P(0); }
#pragma unroll
    for (int c = 0; c < NUA; c++) uACC[c] = active ? a.uACC[gu + c * NU] : P(0);
#pragma unroll
    for (int c = 0; c < NiUA; c++) uACCi[c] = active ? a.uACCi[gu + c * NU] : 0;
#pragma unroll
    for (int c = 0; c < UD; c++) lam[c] = active ? A.lam[gu + c * NU] : P(0);
#pragma unroll
    for (int c = 0; c < NSP; c++) muS[c] = P(0);
    __syncthreads();
    if (leader) atomicMax(&blk[0], my->nseg);
    __syncthreads();
    const int rounds = blk[0];

    P* gPAR = a.gPAR;
    int* gPARi = a.gPARi;
    int buf = 0, wbuf = 0;
    // forward right-hand sides (with coupling) at Y, time T; also the coupling
    // values v and factors CPF of this unit
    auto rhs = [&](bool run, P* F, P* Y, P T, P* v, P* CPF) {
        P* c = cpt + (size_t)buf * stride;
        if (run)
            Sys::template OdeFunction<P>(gsys, u, F, Y, T, uPAR, my->sPAR, gPAR, gPARi, uACC, uACCi, my->sACC, my->sACCi,
                                         c + (size_t)(lsys * UPS + u) * NCp, CPF);
        __syncthreads();
        if (run) {
#pragma unroll
            for (int i = 0; i < NC; i++) {
                v[i] = coupling_dot<Sys>(a, a.cMat, c + (size_t)lsys * UPS * NCp, u, i);
                Unit<Sys, P>::add(cIndex[i], my->strength[i] * CPF[i], v[i], F);
            }
        }
        buf ^= 1;
    };
    // adjoint of one stage: kb (adjoint of the stage derivative) at Y -> gy
    auto vjp = [&](bool run, const P* kb, P* Y, P T, const P* v, const P* CPF, P* gy) {
        P* w = wb + (size_t)wbuf * stride;
        P kbCPF[NCp], kbCPT[NCp];
        if (run) {
#pragma unroll
            for (int i = 0; i < NC; i++) {
                P g = P(0);
#pragma unroll
                for (int c = 0; c < UD; c++)
                    if (c == cIndex[i]) g = kb[c];
                w[(size_t)(lsys * UPS + u) * NCp + i] = my->strength[i] * CPF[i] * g;
                kbCPF[i] = my->strength[i] * v[i] * g;
            }
        }
        __syncthreads();
        if (run) {
#pragma unroll
            for (int i = 0; i < NC; i++) kbCPT[i] = coupling_dot<Sys>(a, A.cMatT, w + (size_t)lsys * UPS * NCp, u, i);
            P gU[NUPp], gS[NSPp];
            Sys::template OdeVJP<P>(gsys, u, kb, kbCPT, kbCPF, Y, T, uPAR, my->sPAR, gPAR, gPARi, uACC, uACCi, my->sACC,
                                    my->sACCi, gy, gU, gS);
#pragma unroll
            for (int c = 0; c < NUP; c++) muU[c] += gU[c];
#pragma unroll
            for (int c = 0; c < NSP; c++) muS[c] += gS[c];
        } else {
#pragma unroll
            for (int c = 0; c < UD; c++) gy[c] = P(0);
        }
        wbuf ^= 1;
    };

    // Butcher coefficients of the steppers as the forward pass evaluates them
    // (pb_device.h): Y_j = x + h sum_l A[j][l] k_l, next = x + h sum_j B[j] k_j
    constexpr int S6 = 6;
    P Acoef[S6][S6] = {};
    P Bcoef[S6] = {};
    P Ccoef[S6] = {};
    if (ALG == MPGOS_RK4) {
        Acoef[1][0] = 0.5; Acoef[2][1] = 0.5; Acoef[3][2] = 1.0;
        Bcoef[0] = 1.0 / 6.0; Bcoef[1] = 2.0 / 6.0; Bcoef[2] = 2.0 / 6.0; Bcoef[3] = 1.0 / 6.0;
    } else {
        Acoef[1][0] = 1.0 / 5.0;
        Acoef[2][0] = 3.0 / 40.0; Acoef[2][1] = 9.0 / 40.0;
        Acoef[3][0] = 3.0 / 10.0; Acoef[3][1] = -9.0 / 10.0; Acoef[3][2] = 6.0 / 5.0;
        Acoef[4][0] = -11.0 / 54.0; Acoef[4][1] = 5.0 / 2.0; Acoef[4][2] = -70.0 / 27.0; Acoef[4][3] = 35.0 / 27.0;
        Acoef[5][0] = 1631.0 / 55296.0; Acoef[5][1] = 175.0 / 512.0; Acoef[5][2] = 575.0 / 13824.0;
        Acoef[5][3] = 44275.0 / 110592.0; Acoef[5][4] = 253.0 / 4096.0;
        Bcoef[0] = 37.0 / 378.0; Bcoef[2] = 250.0 / 621.0; Bcoef[3] = 125.0 / 594.0; Bcoef[5] = 512.0 / 1771.0;
        (void)Ccoef;
    }

    // one forward step with the forward pass's exact arithmetic (pb_device.h);
    // optionally keeps stage values, coupling values and factors
    auto step = [&](bool run, P* X, P t, P h, P (*Ys)[UD], P (*vs)[NCp], P (*cpfs)[NCp]) {
        P next[UD];
        if (ALG == MPGOS_RK4) {
            P k[UD], Y[UD];
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[0][c] = X[c];
            rhs(run, next, X, t, vs[0], cpfs[0]);
#pragma unroll
            for (int c = 0; c < UD; c++) Y[c] = fma(next[c] * P(0.5), h, X[c]);
            const P t2 = t + P(0.5) * h;
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[1][c] = Y[c];
            rhs(run, k, Y, t2, vs[1], cpfs[1]);
#pragma unroll
            for (int c = 0; c < UD; c++) { next[c] = fma(P(2), k[c], next[c]); Y[c] = fma(k[c] * P(0.5), h, X[c]); }
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[2][c] = Y[c];
            rhs(run, k, Y, t2, vs[2], cpfs[2]);
#pragma unroll
            for (int c = 0; c < UD; c++) { next[c] = fma(P(2.0), k[c], next[c]); Y[c] = fma(k[c], h, X[c]); }
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[3][c] = Y[c];
            rhs(run, k, Y, t + h, vs[3], cpfs[3]);
#pragma unroll
            for (int c = 0; c < UD; c++) next[c] = fma(h * (next[c] + k[c]), P(1.0 / 6.0), X[c]);
        } else {
            P k1[UD], k2[UD], k3[UD], k4[UD], k5[UD], k6[UD], Y[UD];
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[0][c] = X[c];
            rhs(run, k1, X, t, vs[0], cpfs[0]);
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[1][c] = Y[c] = fma(k1[c] * P(1.0 / 5.0), h, X[c]);
            rhs(run, k2, Y, fma(P(1.0 / 5.0), h, t), vs[1], cpfs[1]);
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[2][c] = Y[c] = fma(fma(k2[c], P(9.0 / 40.0), k1[c] * P(3.0 / 40.0)), h, X[c]);
            rhs(run, k3, Y, fma(P(3.0 / 10.0), h, t), vs[2], cpfs[2]);
#pragma unroll
            for (int c = 0; c < UD; c++)
                Ys[3][c] = Y[c] = fma(fma(k3[c], P(6.0 / 5.0), fma(k2[c], P(-9.0 / 10.0), k1[c] * P(3.0 / 10.0))), h, X[c]);
            rhs(run, k4, Y, fma(P(3.0 / 5.0), h, t), vs[3], cpfs[3]);
#pragma unroll
            for (int c = 0; c < UD; c++)
                Ys[4][c] = Y[c] = fma(fma(k4[c], P(35.0 / 27.0), fma(k3[c], P(-70.0 / 27.0), fma(k2[c], P(5.0 / 2.0), k1[c] * P(-11.0 / 54.0)))), h, X[c]);
            rhs(run, k5, Y, t + h, vs[4], cpfs[4]);
#pragma unroll
            for (int c = 0; c < UD; c++)
                Ys[5][c] = Y[c] = fma(fma(k5[c], P(253.0 / 4096.0), fma(k4[c], P(44275.0 / 110592.0), fma(k3[c], P(575.0 / 13824.0),
                                      fma(k2[c], P(175.0 / 512.0), k1[c] * P(1631.0 / 55296.0))))), h, X[c]);
            rhs(run, k6, Y, fma(P(7.0 / 8.0), h, t), vs[5], cpfs[5]);
#pragma unroll
            for (int c = 0; c < UD; c++)
                next[c] = fma(fma(k6[c], P(512.0 / 1771.0), fma(k4[c], P(125.0 / 594.0), fma(k3[c], P(250.0 / 621.0), k1[c] * P(37.0 / 378.0)))), h, X[c]);
        }
        if (run) {
#pragma unroll
            for (int c = 0; c < UD; c++) X[c] = next[c];
        }
    };
    auto stage_time = [&](int j, P t, P h) -> P {
        if (ALG == MPGOS_RK4) return j == 0 ? t : (j == 3 ? t + h : t + P(0.5) * h);
        switch (j) {
        case 0: return t;
        case 1: return fma(P(1.0 / 5.0), h, t);
        case 2: return fma(P(3.0 / 10.0), h, t);
        case 3: return fma(P(3.0 / 5.0), h, t);
        case 4: return t + h;
        default: return fma(P(7.0 / 8.0), h, t);
        }
    };

    P Ys[S6][UD], vs[S6][NCp], cpfs[S6][NCp];
    for (int r = 0; r < rounds; r++) {
        // this round's segment of each system: the r-th from the end
        if (leader) {
            const int k = my->nseg - 1 - r;
            my->k = k;
            my->len = k >= 0 ? (int)((my->nacc - (long long)k * K) < K ? (my->nacc - (long long)k * K) : K) : 0;
        }
        if (tid == 0) blk[1] = 0;
        __syncthreads();
        if (leader) atomicMax(&blk[1], my->len);
        __syncthreads();
        const int maxlen = blk[1];
        const int k = my->k, len = lane ? my->len : 0;
        P X[UD];
        if (active && len > 0) {
#pragma unroll
            for (int c = 0; c < UD; c++) X[c] = a.recX[((size_t)k * UD + c) * NU + gu];
        } else {
#pragma unroll
            for (int c = 0; c < UD; c++) X[c] = P(0);
        }
        // 1. recompute the segment, keeping the state at the start of each step
        for (int j = 0; j < maxlen; j++) {
            const bool run = active && j < len;
            P t = P(0), h = P(0);
            if (run) {
                const size_t n = (size_t)k * K + j;
#pragma unroll
                for (int c = 0; c < UD; c++) A.seg[((size_t)j * UD + c) * NU + gu] = X[c];
                t = a.recT[n * NS + gsys];
                h = a.recH[n * NS + gsys];
            }
            step(run, X, t, h, Ys, vs, cpfs);
        }
        // 2. reverse through the segment
        for (int j = maxlen - 1; j >= 0; j--) {
            const bool run = active && j < len;
            P t = P(0), h = P(0);
            if (run) {
                const size_t n = (size_t)k * K + j;
#pragma unroll
                for (int c = 0; c < UD; c++) X[c] = A.seg[((size_t)j * UD + c) * NU + gu];
                t = a.recT[n * NS + gsys];
                h = a.recH[n * NS + gsys];
            }
            P Xs[UD];
#pragma unroll
            for (int c = 0; c < UD; c++) Xs[c] = X[c];
            step(run, Xs, t, h, Ys, vs, cpfs);         // stage values of this step
            P kb[S6][UD];
#pragma unroll
            for (int s = 0; s < S6; s++)
#pragma unroll
                for (int c = 0; c < UD; c++) kb[s][c] = h * Bcoef[s] * lam[c];
#pragma unroll
            for (int s = ST - 1; s >= 0; s--) {
                P gy[UD];
                vjp(run, kb[s], Ys[s], stage_time(s, t, h), vs[s], cpfs[s], gy);
#pragma unroll
                for (int c = 0; c < UD; c++) lam[c] += gy[c];
#pragma unroll
                for (int l = 0; l < S6; l++)
                    if (l < s && Acoef[s][l] != P(0)) {
#pragma unroll
                        for (int c = 0; c < UD; c++) kb[l][c] = fma(h * Acoef[s][l], gy[c], kb[l][c]);
                    }
            }
        }
        __syncthreads();
    }

    // outputs: dL/dx(start), dL/d(unit parameters), dL/d(system parameters)
    const bool bad = active && (my->status & MPGOS_STATUS_CHECKPOINT_OVERFLOW) != 0;
    if (active) {
        const P nan = __builtin_nan("");
#pragma unroll
        for (int c = 0; c < UD; c++) A.lam[gu + c * NU] = bad ? nan : lam[c];
#pragma unroll
        for (int c = 0; c < NUP; c++) A.gU[gu + c * NU] = bad ? nan : muU[c];
    }
    if (lane) {
#pragma unroll
        for (int c = 0; c < NSP; c++) red[((size_t)lsys * UPS + u) * NSPp + c] = muS[c];
    }
    __syncthreads();
    if (leader && active) {
        for (int c = 0; c < NSP; c++) {
            P s = P(0);
            for (int v = 0; v < UPS; v++) s += red[((size_t)lsys * UPS + v) * NSPp + c];
            A.gS[gsys + (size_t)c * NS] = bad ? __builtin_nan("") : s;
        }
    }
}

template <class Sys, int ALG, int MAXT>
__global__ void __launch_bounds__(MAXT) pb_reverse_kernel(Args<Sys, double> a, AdjArgs<Sys> A)
{
    pb_reverse_body<Sys, ALG>(a, A);
}

// ---------------------------------------------------------------- dense-contraction form
// Butcher coefficients of the steppers (the adjoint's coefficients; the forward
// arithmetic itself is written out in the steps below) and the stage times
// exactly as the forward pass computes them.
template <int ALG>
__device__ __forceinline__ double rk_b(int s)
{
    if (ALG == MPGOS_RK4) return (s == 0 || s == 3) ? 1.0 / 6.0 : 2.0 / 6.0;
    switch (s) {
    case 0: return 37.0 / 378.0;
    case 2: return 250.0 / 621.0;
    case 3: return 125.0 / 594.0;
    case 5: return 512.0 / 1771.0;
    default: return 0.0;
    }
}

template <int ALG>
__device__ __forceinline__ double rk_a(int s, int l)
{
    if (ALG == MPGOS_RK4) return (l == s - 1) ? (s == 3 ? 1.0 : 0.5) : 0.0;
    constexpr double A[6][5] = {{0, 0, 0, 0, 0},
                                {1.0 / 5.0, 0, 0, 0, 0},
                                {3.0 / 40.0, 9.0 / 40.0, 0, 0, 0},
                                {3.0 / 10.0, -9.0 / 10.0, 6.0 / 5.0, 0, 0},
                                {-11.0 / 54.0, 5.0 / 2.0, -70.0 / 27.0, 35.0 / 27.0, 0},
                                {1631.0 / 55296.0, 175.0 / 512.0, 575.0 / 13824.0, 44275.0 / 110592.0, 253.0 / 4096.0}};
    return l < s ? A[s][l] : 0.0;
}

// Input of stage st > 0 by the forward pass's arithmetic: x and the stages before.
template <int ALG, int UD, int ST>
__device__ __forceinline__ double rk_stage_input(int st, int c, double h, const double (&x)[UD], const double (&k)[ST][UD])
{
    using math::fma;
    if (ALG == MPGOS_RK4) return fma(st == 3 ? k[2][c] : k[st - 1][c] * 0.5, h, x[c]);
    double r = 0.0;
    switch (st) {
    case 1: r = k[0][c] * (1.0 / 5.0); break;
    case 2: r = fma(k[1][c], 9.0 / 40.0, k[0][c] * (3.0 / 40.0)); break;
    case 3: r = fma(k[2][c], 6.0 / 5.0, fma(k[1][c], -9.0 / 10.0, k[0][c] * (3.0 / 10.0))); break;
    case 4: r = fma(k[ST - 3][c], 35.0 / 27.0, fma(k[2][c], -70.0 / 27.0, fma(k[1][c], 5.0 / 2.0, k[0][c] * (-11.0 / 54.0)))); break;
    default:
        r = fma(k[ST - 2][c], 253.0 / 4096.0, fma(k[ST - 3][c], 44275.0 / 110592.0, fma(k[2][c], 575.0 / 13824.0,
                fma(k[1][c], 175.0 / 512.0, k[0][c] * (1631.0 / 55296.0)))));
    }
    return fma(r, h, x[c]);
}

// Reverse pass in the dense-contraction form (full FP64 coupling matrices, up
// to 256 units): the layout of pb_dense.h, every coupling product on
// v_mfma_f64_4x4x4f64 -- M CPT(Y) in the segment replay, M^T w in the adjoint
// sweep.  Round r handles the r-th segment from the end of every system in two
// launches:
//   pb_replay_kernel: restore checkpoint k = nseg - 1 - r and replay the
//     segment's recorded steps, keeping each stage's coupling values v_s, and
//     the step's state or each stage's input Y_s, in the stage buffer of rows
//     [row][NU], rev_rows() of them per step;
//   pb_sweep_kernel: the adjoint sweep through the segment from the stage
//     buffer (no forward coupling product again); dL/dx, the unit-parameter gradient and
//     the per-unit system-parameter partials carry over between rounds in HBM
//     (lam, gU, gSp);
// pb_reverse_finish_kernel sums the partials per system in unit order.  Two
// kernels instead of one keep the stage vectors of the replay and the adjoints
// of the sweep from being live together, and let each hold its own matrix (M,
// M^T) in LDS.  Sums run in the same order as in the lane form, so both forms
// return the same bits.
//
// What bounds it: the latency of a step (1024 x 128 units: two wavefronts per
// SIMD) and, with 8 systems of 256 units, the registers (78 of the sweep's
// values per lane spill).  Reverse pass of two periods of 1024 x 128 units
// 24.6 -> 6.8 ms, one period of 300 x 256 25.6 -> 14.6, 4096 x 128 21.1 -> 14.3,
// 4096 x 256 57.1 -> 49.8 ms against products through LDS with 8 systems per
// workgroup; 1000 x 100 units 40.5 -> 2.9 ms against one lane per unit.
// Stage buffer: with one result per lane the step's state and the stages'
// coupling values, from which the sweep makes the stage inputs again (all of them
// stay in its registers); with more the inputs themselves.  At 1024 x 128 units of
// the ring with a quadrature state a step moves 9 rows, 9.4 MB each way, instead
// of 24, 25 MB: reverse pass of two periods 7.1 -> 6.8 ms, smaller ones unchanged
// (the sweep makes up for it with the right-hand sides it evaluates).
template <class Sys>
__host__ __device__ inline size_t rev_lds_bytes(int SPB, int UPS, int ldsPairs)
{
    return dense_layout<RevScope<Sys>, Sys::NC, 0, 0>(SPB, UPS, 0, ldsPairs).total + 2 * sizeof(double) * (size_t)SPB * 64;
}
template <int NSL, int MT> __host__ __device__ constexpr bool rev_remake() { return NSL * dense_tt(MT) == 1; }
template <class Sys> __host__ __device__ constexpr int rev_rows(bool remake, int ST)
{
    return remake ? Sys::UD + ST * Sys::NC : ST * (Sys::UD + Sys::NC);
}

template <class Sys, int NSL, int MT>
struct DenseRev {
    static constexpr int TT = dense_tt(MT);
    static constexpr int NC = Sys::NC, SPB = 4 * NSL, NTT = TimeTermsOf<Sys>::n, PER = 64 / SPB;
    static constexpr int kTimes = 64;
    using Scope = RevScope<Sys>;
    using Place = DensePlace<NSL, TT>;
    Scope* sys; double* cptBuf; const double* Ml; double* times;
    int cptStride, maxlen;
    size_t NU;
    Place at;
    bool active[NSL];
    int k[NSL], len[NSL];
    double strength[NSL][Pos<NC>::value];

    // LDS, system scope and this round's segment of each system
    // (k = nseg - 1 - r, len steps; maxlen over the workgroup)
    __device__ __forceinline__ DenseRev(const Args<Sys, double>& a, const double* Mt, unsigned char* lds, int r)
        : at(a.UPS, a.NS)
    {
        const DenseLayout L = dense_layout<Scope, NC, 0, 0>(SPB, a.UPS, 0, a.ldsPairs);
        sys = reinterpret_cast<Scope*>(lds);
        cptBuf = reinterpret_cast<double*>(lds + L.cpt);
        Ml = reinterpret_cast<const double*>(lds + L.mt);
        times = reinterpret_cast<double*>(lds + L.total);
        int* blk = reinterpret_cast<int*>(lds + L.blk);
        cptStride = NC * SPB * dense_row(a.UPS);
        NU = (size_t)a.NS * a.UPS;
        const int K = a.recK;
        if (threadIdx.x == 0) blk[0] = 0;
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            const int g = at.gsys(s);
            active[s] = g < a.NS && g < a.nActive;
            if (!at.leads(s)) continue;
            Scope& y = sys[at.sys(s)];
            y.status = 0; y.k = -1; y.len = 0;
            for (int i = 0; i < Sys::NSP; i++) y.sPAR[i] = active[s] ? a.sPAR[g + i * a.NS] : 0.0;
            if (active[s]) {
                for (int i = 0; i < Sys::NSA; i++) y.sACC[i] = a.sACC[g + i * a.NS];
                for (int i = 0; i < Sys::NiSA; i++) y.sACCi[i] = a.sACCi[g + i * a.NS];
                for (int i = 0; i < NC; i++) y.strength[i] = a.strength[g + i * a.NS];
                y.nacc = a.nacc[g];
                y.status = a.status[g];
                const bool ok = (y.status & MPGOS_STATUS_CHECKPOINT_OVERFLOW) == 0;
                const int kk = (ok ? (int)((y.nacc + K - 1) / K) : 0) - 1 - r;
                y.k = kk;
                y.len = kk >= 0 ? (int)((y.nacc - (long long)kk * K) < K ? (y.nacc - (long long)kk * K) : K) : 0;
            }
        }
        __syncthreads();
        if (threadIdx.x < SPB) atomicMax(&blk[0], sys[threadIdx.x].len);
        __syncthreads();
        maxlen = blk[0];
        if (maxlen == 0) return;                       // workgroup-uniform
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            k[s] = sys[at.sys(s)].k;
            len[s] = active[s] ? sys[at.sys(s)].len : 0;
#pragma unroll
            for (int i = 0; i < NC; i++) strength[s][i] = sys[at.sys(s)].strength[i];
        }
        for (int i = threadIdx.x; i < 2 * cptStride; i += blockDim.x) cptBuf[i] = 0.0;   // padded units and absent systems stay zero
        dense_stage_matrix(Mt, lds + L.mt, NC, a.UPS, a.ldsPairs);
        __syncthreads();
    }
    __device__ __forceinline__ bool has(int s, int q) const { return len[s] > 0 && at.has(q); }
    __device__ __forceinline__ unsigned unit(int s, int q) const { return (unsigned)at.gsys(s) * (unsigned)at.UPS + (unsigned)at.unit(q); }
    // row r of a unit-scope array [rows][NU]: wave-uniform row base, 32-bit lane offset
    template <class T>
    __device__ __forceinline__ T* row(T* base, size_t r) const { return base + r * NU; }
    // (t, h) of step j of each of the lane's systems, 0 where it has none, from
    // kTimes steps of them in LDS (read from global memory where they are used,
    // they wait for the stage buffer's stores as well, which the same counter
    // counts: replay of 32 steps of 1024 x 128 units 0.30 -> 0.22 ms).  Called by
    // the whole workgroup.
    __device__ __forceinline__ void step_times(const Args<Sys, double>& a, int j, int& chunk, double* t, double* h) const
    {
        if (j >= 0 && j < maxlen && j / kTimes != chunk) {
            chunk = j / kTimes;
            __syncthreads();
            for (int e = threadIdx.x; e < kTimes * SPB; e += blockDim.x) {
                const int s = e % SPB, jj = chunk * kTimes + e / SPB;
                const bool run = jj < sys[s].len;
                const size_t n = ((size_t)sys[s].k * a.recK + jj) * a.NS + ((size_t)blockIdx.x * SPB + s);
                times[e] = run ? a.recT[n] : 0.0;
                times[kTimes * SPB + e] = run ? a.recH[n] : 0.0;
            }
            __syncthreads();
        }
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            const bool run = j >= 0 && j < len[s];
            const int e = (j % kTimes) * SPB + at.sys(s);
            t[s] = run ? times[e] : 0.0;
            h[s] = run ? times[kTimes * SPB + e] : 0.0;
        }
    }
    // the time terms of a step's stages as in the forward pass: lane l
    // evaluates stage e * PER + l / SPB of system l % SPB
    template <int ALG, int N>
    __device__ __forceinline__ void time_terms(const double* t, const double* h, double (&tt)[N][Pos<NTT>::value]) const
    {
        if constexpr (NTT > 0) {
            double t0 = t[0], h0 = h[0];
            if constexpr (NSL > 1) {
                // opaque values: a select between array elements would become an
                // indexed load, which moves the arrays to scratch memory
                double t1 = t[NSL - 1], h1 = h[NSL - 1];
                asm("" : "+v"(t0), "+v"(h0), "+v"(t1), "+v"(h1));
                const bool own = (at.l % SPB) < 4;
                t0 = own ? t0 : t1;
                h0 = own ? h0 : h1;
            }
#pragma unroll
            for (int e = 0; e < N; e++)
                Sys::template TimeTerms<double>(rk_stage_time<ALG>(e * PER + at.l / SPB, t0, h0), sys[at.l % SPB].sPAR, tt[e]);
        }
    }
    template <int N>
    __device__ __forceinline__ void stage_terms(int stage, const double (&tterm)[N][Pos<NTT>::value], double (&tt)[NSL][Pos<NTT>::value]) const
    {
#pragma unroll
        for (int s = 0; s < NSL; s++)
#pragma unroll
            for (int i = 0; i < NTT; i++) tt[s][i] = __shfl(tterm[stage / PER][i], (stage % PER) * SPB + at.sys(s));
    }
};

#define MPGOS_PB_EACH(s, q) _Pragma("unroll") for (int s = 0; s < NSL; s++) _Pragma("unroll") for (int q = 0; q < TT; q++)

template <class Sys, int ALG, int NSL, int MT>
__device__ void pb_replay_body(const Args<Sys, double>& a, const AdjArgs<Sys>& A, int r)
{
    constexpr int TT = dense_tt(MT);
    using P = double;
    constexpr int UD = Sys::UD, NC = Sys::NC, NUP = Sys::NUP, NUA = Sys::NUA, NiUA = Sys::NiUA;
    constexpr int NCp = Pos<NC>::value, NTT = TimeTermsOf<Sys>::n, ST = ALG == MPGOS_RK4 ? 4 : 6, SW = UD + NC;
    constexpr bool REMAKE = rev_remake<NSL, MT>();
    constexpr int ROWS = rev_rows<Sys>(REMAKE, ST);
    using math::fma;
    using R = DenseRev<Sys, NSL, MT>;
    extern __shared__ __align__(16) unsigned char mpgos_pb_lds[];
    const R C(a, a.cTile, mpgos_pb_lds, r);
    if (C.maxlen == 0) return;
    DenseContraction<Sys, NSL, MT> product(a.cTile, C.Ml, a.ldsPairs, a.UPS);
    const int RS = dense_row(a.UPS);

    int cIndex[NCp];
#pragma unroll
    for (int i = 0; i < NC; i++) cIndex[i] = a.cIndex[i];
    P uPAR[NSL][TT][Pos<NUP>::value], uACC[NSL][TT][Pos<NUA>::value], X[NSL][TT][UD];
    int uACCi[NSL][TT][Pos<NiUA>::value];
    MPGOS_PB_EACH(s, q) {
        const bool ld = C.has(s, q);
        const unsigned u = C.unit(s, q);
#pragma unroll
        for (int c = 0; c < NUP; c++) uPAR[s][q][c] = ld ? C.row(a.uPAR, c)[u] : P(0);
#pragma unroll
        for (int c = 0; c < NUA; c++) uACC[s][q][c] = ld ? C.row(a.uACC, c)[u] : P(0);
#pragma unroll
        for (int c = 0; c < NiUA; c++) uACCi[s][q][c] = ld ? C.row(a.uACCi, c)[u] : 0;
#pragma unroll
        for (int c = 0; c < UD; c++) X[s][q][c] = ld ? a.recX[((size_t)C.k[s] * UD + c) * C.NU + u] : P(0);
    }

    int buf = 0;
    P tterm[(ST + R::PER - 1) / R::PER][Pos<NTT>::value], tt[NSL][Pos<NTT>::value];
    P t[NSL], h[NSL], tn[NSL], hn[NSL];
    int chunk = -1;
    // right-hand sides of the lane's units at (Y, T) plus the coupling terms of
    // stage st of step j; Y and the coupling values (M CPT)_u are kept.  The
    // barriers order LDS only, so the stage-buffer stores stay in flight.
    auto rhs = [&](int st, int j, P (*F)[TT][UD], P (*Y)[TT][UD]) {
        P CPF[NSL][TT][NCp], v[NCp][NSL][TT];
        P* cpt = C.cptBuf + (size_t)buf * C.cptStride;
        product.prefetch();
        MPGOS_PB_EACH(s, q) {
            if (j < C.len[s] && C.at.has(q)) {
                P cp[NCp];
#pragma unroll
                for (int i = 0; i < NC; i++) cp[i] = CPF[s][q][i] = P(0);
                auto& y = C.sys[C.at.sys(s)];
                const P T = rk_stage_time<ALG>(st, t[s], h[s]);
                if constexpr (NTT > 0)
                    Sys::template OdeFunctionTT<P>(C.at.gsys(s), C.at.unit(q), F[s][q], Y[s][q], T, tt[s], uPAR[s][q], y.sPAR, a.gPAR, a.gPARi,
                                                   uACC[s][q], uACCi[s][q], y.sACC, y.sACCi, cp, CPF[s][q]);
                else
                    Sys::template OdeFunction<P>(C.at.gsys(s), C.at.unit(q), F[s][q], Y[s][q], T, uPAR[s][q], y.sPAR, a.gPAR, a.gPARi,
                                                 uACC[s][q], uACCi[s][q], y.sACC, y.sACCi, cp, CPF[s][q]);
#pragma unroll
                for (int i = 0; i < NC; i++) cpt[(i * R::SPB + C.at.sys(s)) * RS + C.at.unit(q)] = cp[i];
                if (!REMAKE || st == 0) {
                    const size_t base = REMAKE ? (size_t)j * ROWS : ((size_t)j * ST + st) * SW;
#pragma unroll
                    for (int c = 0; c < UD; c++) C.row(A.stg, base + c)[C.unit(s, q)] = Y[s][q][c];
                }
            }
        }
        if (st + 1 < ST) C.stage_terms(st + 1, tterm, tt);
        lds_barrier();
        product.run(cpt, v);
        MPGOS_PB_EACH(s, q) {
#pragma unroll
            for (int i = 0; i < NC; i++)
                Unit<Sys, P>::add(cIndex[i], C.strength[s][i] * CPF[s][q][i], v[i][s][q], F[s][q]);
            if (j < C.len[s] && C.at.has(q)) {
                const size_t base = REMAKE ? (size_t)j * ROWS + UD + st * NC : ((size_t)j * ST + st) * SW + UD;
#pragma unroll
                for (int i = 0; i < NC; i++) C.row(A.stg, base + i)[C.unit(s, q)] = v[i][s][q];
            }
        }
        buf ^= 1;
    };
    auto fill = [&](P (*Y)[TT][UD], auto&& value) {
        MPGOS_PB_EACH(s, q) {
#pragma unroll
            for (int c = 0; c < UD; c++) Y[s][q][c] = value(s, q, c);
        }
    };
    C.step_times(a, 0, chunk, tn, hn);
    for (int j = 0; j < C.maxlen; j++) {
#pragma unroll
        for (int s = 0; s < NSL; s++) { t[s] = tn[s]; h[s] = hn[s]; }
        C.step_times(a, j + 1, chunk, tn, hn);                 // one step ahead
        C.template time_terms<ALG>(t, h, tterm);
        C.stage_terms(0, tterm, tt);
        // the forward pass's stage arithmetic (pb_dense_body)
        P next[NSL][TT][UD], k[NSL][TT][UD], Y[NSL][TT][UD];
        if (ALG == MPGOS_RK4) {
            rhs(0, j, next, X);
            fill(Y, [&](int s, int q, int c) { return fma(next[s][q][c] * P(0.5), h[s], X[s][q][c]); });
            rhs(1, j, k, Y);
            fill(next, [&](int s, int q, int c) { return fma(P(2), k[s][q][c], next[s][q][c]); });
            fill(Y, [&](int s, int q, int c) { return fma(k[s][q][c] * P(0.5), h[s], X[s][q][c]); });
            rhs(2, j, k, Y);
            fill(next, [&](int s, int q, int c) { return fma(P(2.0), k[s][q][c], next[s][q][c]); });
            fill(Y, [&](int s, int q, int c) { return fma(k[s][q][c], h[s], X[s][q][c]); });
            rhs(3, j, k, Y);
            fill(next, [&](int s, int q, int c) { return fma(h[s] * (next[s][q][c] + k[s][q][c]), P(1.0 / 6.0), X[s][q][c]); });
        } else {
            P k1[NSL][TT][UD], k2[NSL][TT][UD], k3[NSL][TT][UD], sum6[NSL][TT][UD];
            rhs(0, j, k1, X);
            fill(Y, [&](int s, int q, int c) { return fma(k1[s][q][c] * P(1.0 / 5.0), h[s], X[s][q][c]); });
            rhs(1, j, k2, Y);
            fill(Y, [&](int s, int q, int c) { return fma(fma(k2[s][q][c], P(9.0 / 40.0), k1[s][q][c] * P(3.0 / 40.0)), h[s], X[s][q][c]); });
            rhs(2, j, k3, Y);
            fill(Y, [&](int s, int q, int c) {
                return fma(fma(k3[s][q][c], P(6.0 / 5.0), fma(k2[s][q][c], P(-9.0 / 10.0), k1[s][q][c] * P(3.0 / 10.0))), h[s], X[s][q][c]);
            });
            rhs(3, j, k, Y);
            fill(Y, [&](int s, int q, int c) {
                return fma(fma(k[s][q][c], P(35.0 / 27.0), fma(k3[s][q][c], P(-70.0 / 27.0), fma(k2[s][q][c], P(5.0 / 2.0),
                           k1[s][q][c] * P(-11.0 / 54.0)))), h[s], X[s][q][c]);
            });
            fill(sum6, [&](int s, int q, int c) {
                return fma(k[s][q][c], P(44275.0 / 110592.0), fma(k3[s][q][c], P(575.0 / 13824.0),
                           fma(k2[s][q][c], P(175.0 / 512.0), k1[s][q][c] * P(1631.0 / 55296.0))));
            });
            fill(next, [&](int s, int q, int c) {
                return fma(k[s][q][c], P(125.0 / 594.0), fma(k3[s][q][c], P(250.0 / 621.0), k1[s][q][c] * P(37.0 / 378.0)));
            });
            rhs(4, j, k, Y);
            fill(Y, [&](int s, int q, int c) { return fma(fma(k[s][q][c], P(253.0 / 4096.0), sum6[s][q][c]), h[s], X[s][q][c]); });
            rhs(5, j, k, Y);
            fill(next, [&](int s, int q, int c) { return fma(fma(k[s][q][c], P(512.0 / 1771.0), next[s][q][c]), h[s], X[s][q][c]); });
        }
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            if (j < C.len[s]) {
#pragma unroll
                for (int q = 0; q < TT; q++)
#pragma unroll
                    for (int c = 0; c < UD; c++) X[s][q][c] = next[s][q][c];
            }
        }
    }
}

template <class Sys, int ALG, int NSL, int MT>
__device__ void pb_sweep_body(const Args<Sys, double>& a, const AdjArgs<Sys>& A, int r)
{
    constexpr int TT = dense_tt(MT);
    using P = double;
    constexpr int UD = Sys::UD, NC = Sys::NC, NUP = Sys::NUP, NSP = Sys::NSP, NUA = Sys::NUA, NiUA = Sys::NiUA;
    constexpr int NCp = Pos<NC>::value, NUPp = Pos<NUP>::value, NSPp = Pos<NSP>::value, NTT = TimeTermsOf<Sys>::n;
    constexpr int ST = ALG == MPGOS_RK4 ? 4 : 6, SW = UD + NC;
    constexpr bool REMAKE = rev_remake<NSL, MT>();
    constexpr int ROWS = rev_rows<Sys>(REMAKE, ST), FETCH = REMAKE ? ROWS : SW;
    using math::fma;
    using R = DenseRev<Sys, NSL, MT>;
    extern __shared__ __align__(16) unsigned char mpgos_pb_lds[];
    const R C(a, A.cTileT, mpgos_pb_lds, r);
    if (C.maxlen == 0) return;
    DenseContraction<Sys, NSL, MT> product(A.cTileT, C.Ml, a.ldsPairs, a.UPS);
    const int RS = dense_row(a.UPS);

    int cIndex[NCp];
#pragma unroll
    for (int i = 0; i < NC; i++) cIndex[i] = a.cIndex[i];
    // adjoint state carried between rounds; round 0 starts the gradients at zero
    P uPAR[NSL][TT][NUPp], uACC[NSL][TT][Pos<NUA>::value], lam[NSL][TT][UD], muU[NSL][TT][NUPp], muS[NSL][TT][NSPp];
    int uACCi[NSL][TT][Pos<NiUA>::value];
    MPGOS_PB_EACH(s, q) {
        const bool ld = C.has(s, q);
        const unsigned u = C.unit(s, q);
#pragma unroll
        for (int c = 0; c < NUP; c++) {
            uPAR[s][q][c] = ld ? C.row(a.uPAR, c)[u] : P(0);
            muU[s][q][c] = (ld && r > 0) ? C.row(A.gU, c)[u] : P(0);
        }
#pragma unroll
        for (int c = 0; c < NUA; c++) uACC[s][q][c] = ld ? C.row(a.uACC, c)[u] : P(0);
#pragma unroll
        for (int c = 0; c < NiUA; c++) uACCi[s][q][c] = ld ? C.row(a.uACCi, c)[u] : 0;
#pragma unroll
        for (int c = 0; c < UD; c++) lam[s][q][c] = ld ? C.row(A.lam, c)[u] : P(0);
#pragma unroll
        for (int c = 0; c < NSP; c++) muS[s][q][c] = (ld && r > 0) ? C.row(A.gSp, c)[u] : P(0);
    }
    // a stage's inputs and coupling values, loaded one stage ahead where the
    // registers hold them (with 4 results per lane they would be spilled:
    // reverse pass of 4096 x 256 units 54.6 against 49.8 ms); REMAKE: a step's
    // state and coupling values, loaded one step ahead
    constexpr bool AHEAD = NSL * TT < 4;
    P ahead[NSL][TT][FETCH];
    auto fetch = [&](int j, int st) {
        const size_t base = REMAKE ? (size_t)j * ROWS : ((size_t)j * ST + st) * SW;
        MPGOS_PB_EACH(s, q) {
            const bool ld = j >= 0 && j < C.len[s] && C.at.has(q);
#pragma unroll
            for (int c = 0; c < FETCH; c++) ahead[s][q][c] = ld ? C.row(A.stg, base + c)[C.unit(s, q)] : P(0);
        }
    };

    int buf = 0;
    P tterm[(ST + R::PER - 1) / R::PER][Pos<NTT>::value], tt[NSL][Pos<NTT>::value];
    P t[NSL], h[NSL], tn[NSL], hn[NSL];
    int chunk = -1;
    C.step_times(a, C.maxlen - 1, chunk, tn, hn);
    if (AHEAD) fetch(C.maxlen - 1, ST - 1);
    for (int j = C.maxlen - 1; j >= 0; j--) {
#pragma unroll
        for (int s = 0; s < NSL; s++) { t[s] = tn[s]; h[s] = hn[s]; }
        C.step_times(a, j - 1, chunk, tn, hn);                 // one step ahead
        C.template time_terms<ALG>(t, h, tterm);
        // REMAKE: the stage inputs by the forward pass's arithmetic
        // (pb_dense_body) from the coupling values; Ys, cpfs, tts of every stage
        P Ys[REMAKE ? ST : 1][UD], vs[REMAKE ? ST : 1][NCp], cpfs[REMAKE ? ST : 1][NCp], tts[REMAKE ? ST : 1][NSL][Pos<NTT>::value];
        if constexpr (REMAKE) {
            P k[ST][UD];
#pragma unroll
            for (int st = 0; st < ST; st++) {
                C.stage_terms(st, tterm, tts[st]);
#pragma unroll
                for (int i = 0; i < NC; i++) { vs[st][i] = ahead[0][0][UD + st * NC + i]; cpfs[st][i] = P(0); }
            }
#pragma unroll
            for (int c = 0; c < UD; c++) Ys[0][c] = ahead[0][0][c];
            fetch(j - 1, 0);
            const bool run = j < C.len[0] && C.at.has(0);
#pragma unroll
            for (int st = 0; st < ST; st++) {
#pragma unroll
                for (int c = 0; c < UD; c++)
                    if (st > 0) Ys[st][c] = rk_stage_input<ALG, UD>(st, c, h[0], Ys[0], k);
                if (run) {
                    auto& y = C.sys[C.at.sys(0)];
                    P cp[NCp];
                    const P T = rk_stage_time<ALG>(st, t[0], h[0]);
                    if constexpr (NTT > 0)
                        Sys::template OdeFunctionTT<P>(C.at.gsys(0), C.at.unit(0), k[st], Ys[st], T, tts[st][0], uPAR[0][0], y.sPAR, a.gPAR,
                                                       a.gPARi, uACC[0][0], uACCi[0][0], y.sACC, y.sACCi, cp, cpfs[st]);
                    else
                        Sys::template OdeFunction<P>(C.at.gsys(0), C.at.unit(0), k[st], Ys[st], T, uPAR[0][0], y.sPAR, a.gPAR, a.gPARi,
                                                     uACC[0][0], uACCi[0][0], y.sACC, y.sACCi, cp, cpfs[st]);
#pragma unroll
                    for (int i = 0; i < NC; i++) Unit<Sys, P>::add(cIndex[i], C.strength[0][i] * cpfs[st][i], vs[st][i], k[st]);
                }
            }
        } else {
            C.stage_terms(ST - 1, tterm, tt);
        }
        P kb[ST][NSL][TT][UD];
#pragma unroll
        for (int st = 0; st < ST; st++)
            MPGOS_PB_EACH(s, q) {
#pragma unroll
                for (int c = 0; c < UD; c++) kb[st][s][q][c] = h[s] * rk_b<ALG>(st) * lam[s][q][c];
            }
#pragma unroll
        for (int st = ST - 1; st >= 0; st--) {
            P Y[NSL][TT][UD], kbCPF[NSL][TT][NCp], w[NCp][NSL][TT];
            P* wb = C.cptBuf + (size_t)buf * C.cptStride;
            if (!AHEAD) fetch(j, st);
            if constexpr (REMAKE) {
#pragma unroll
                for (int i = 0; i < NTT; i++) tt[0][i] = tts[st][0][i];
            }
            MPGOS_PB_EACH(s, q) {
#pragma unroll
                for (int c = 0; c < UD; c++) Y[s][q][c] = REMAKE ? Ys[REMAKE ? st : 0][c] : ahead[s][q][c];
                if (j < C.len[s] && C.at.has(q)) {
                    P F[UD], cp[NCp], cpf[NCp];
#pragma unroll
                    for (int i = 0; i < NC; i++) cpf[i] = REMAKE ? cpfs[REMAKE ? st : 0][i] : P(0);
                    auto& y = C.sys[C.at.sys(s)];
                    const P T = rk_stage_time<ALG>(st, t[s], h[s]);
                    if constexpr (REMAKE) {
                    } else if constexpr (NTT > 0)
                        Sys::template OdeFunctionTT<P>(C.at.gsys(s), C.at.unit(q), F, Y[s][q], T, tt[s], uPAR[s][q], y.sPAR, a.gPAR, a.gPARi,
                                                       uACC[s][q], uACCi[s][q], y.sACC, y.sACCi, cp, cpf);
                    else
                        Sys::template OdeFunction<P>(C.at.gsys(s), C.at.unit(q), F, Y[s][q], T, uPAR[s][q], y.sPAR, a.gPAR, a.gPARi,
                                                     uACC[s][q], uACCi[s][q], y.sACC, y.sACCi, cp, cpf);
#pragma unroll
                    for (int i = 0; i < NC; i++) {
                        P g = P(0);
#pragma unroll
                        for (int c = 0; c < UD; c++)
                            if (c == cIndex[i]) g = kb[st][s][q][c];
                        wb[(i * R::SPB + C.at.sys(s)) * RS + C.at.unit(q)] = C.strength[s][i] * cpf[i] * g;
                        kbCPF[s][q][i] = C.strength[s][i] * (REMAKE ? vs[REMAKE ? st : 0][i] : ahead[s][q][REMAKE ? 0 : UD + i]) * g;
                    }
                }
            }
            if (AHEAD && !REMAKE) {
                if (st > 0) fetch(j, st - 1);
                else fetch(j - 1, ST - 1);
            }
            product.prefetch();
            lds_barrier();
            product.run(wb, w);
            buf ^= 1;
            MPGOS_PB_EACH(s, q) {
                P gy[UD];
                if (j < C.len[s] && C.at.has(q)) {
                    P kbCPT[NCp], gU[NUPp], gS[NSPp];
#pragma unroll
                    for (int i = 0; i < NC; i++) kbCPT[i] = w[i][s][q];
                    auto& y = C.sys[C.at.sys(s)];
                    const P T = rk_stage_time<ALG>(st, t[s], h[s]);
                    if constexpr (TimeTermsOf<Sys>::timeOnly)
                        Sys::template OdeVJPTT<P>(C.at.gsys(s), C.at.unit(q), kb[st][s][q], kbCPT, kbCPF[s][q], Y[s][q], T, tt[s], uPAR[s][q],
                                                  y.sPAR, a.gPAR, a.gPARi, uACC[s][q], uACCi[s][q], y.sACC, y.sACCi, gy, gU, gS);
                    else
                        Sys::template OdeVJP<P>(C.at.gsys(s), C.at.unit(q), kb[st][s][q], kbCPT, kbCPF[s][q], Y[s][q], T, uPAR[s][q], y.sPAR,
                                                a.gPAR, a.gPARi, uACC[s][q], uACCi[s][q], y.sACC, y.sACCi, gy, gU, gS);
#pragma unroll
                    for (int c = 0; c < NUP; c++) muU[s][q][c] += gU[c];
#pragma unroll
                    for (int c = 0; c < NSP; c++) muS[s][q][c] += gS[c];
                } else {
#pragma unroll
                    for (int c = 0; c < UD; c++) gy[c] = P(0);
                }
#pragma unroll
                for (int c = 0; c < UD; c++) lam[s][q][c] += gy[c];
#pragma unroll
                for (int l = 0; l < ST; l++)
                    if (l < st && rk_a<ALG>(st, l) != P(0)) {
#pragma unroll
                        for (int c = 0; c < UD; c++) kb[l][s][q][c] = fma(h[s] * rk_a<ALG>(st, l), gy[c], kb[l][s][q][c]);
                    }
            }
            if (!REMAKE && st > 0) C.stage_terms(st - 1, tterm, tt);
        }
    }
    MPGOS_PB_EACH(s, q) {
        if (C.has(s, q)) {
            const unsigned u = C.unit(s, q);
#pragma unroll
            for (int c = 0; c < UD; c++) C.row(A.lam, c)[u] = lam[s][q][c];
#pragma unroll
            for (int c = 0; c < NUP; c++) C.row(A.gU, c)[u] = muU[s][q][c];
#pragma unroll
            for (int c = 0; c < NSP; c++) C.row(A.gSp, c)[u] = muS[s][q][c];
        }
    }
}
#undef MPGOS_PB_EACH

template <class Sys, int ALG, int NSL, int MT>
__global__ void __launch_bounds__(512, 2) pb_replay_kernel(Args<Sys, double> a, AdjArgs<Sys> A, int r)
{
    pb_replay_body<Sys, ALG, NSL, MT>(a, A, r);
}

template <class Sys, int ALG, int NSL, int MT>
__global__ void __launch_bounds__(512, 2) pb_sweep_kernel(Args<Sys, double> a, AdjArgs<Sys> A, int r)
{
    pb_sweep_body<Sys, ALG, NSL, MT>(a, A, r);
}

// Outputs of the dense-contraction reverse pass, one thread per unit: systems
// without accepted steps get zero gradients (dL/dx unchanged), systems whose
// record overflowed NaN; dL/d(system parameters) sums the per-unit partials in
// unit order (thread 0 of the system's units).
template <class Sys>
__global__ void pb_reverse_finish_kernel(Args<Sys, double> a, AdjArgs<Sys> A)
{
    constexpr int UD = Sys::UD, NUP = Sys::NUP, NSP = Sys::NSP;
    const size_t NU = (size_t)a.NS * a.UPS;
    const size_t g = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (g >= NU) return;
    const int gsys = (int)(g / a.UPS), u = (int)(g - (size_t)gsys * a.UPS);
    if (gsys >= a.nActive) return;
    const bool bad = (a.status[gsys] & MPGOS_STATUS_CHECKPOINT_OVERFLOW) != 0;
    const bool none = a.nacc[gsys] == 0;
    const double nan = __builtin_nan("");
    if (bad) {
        for (int c = 0; c < UD; c++) A.lam[g + c * NU] = nan;
        for (int c = 0; c < NUP; c++) A.gU[g + c * NU] = nan;
    } else if (none) {
        for (int c = 0; c < NUP; c++) A.gU[g + c * NU] = 0.0;
    }
    if (u == 0) {
        for (int c = 0; c < NSP; c++) {
            double s = 0.0;
            if (!none)
                for (int v = 0; v < a.UPS; v++) s += A.gSp[(size_t)c * NU + g + v];
            A.gS[gsys + (size_t)c * a.NS] = bad ? nan : s;
        }
    }
}

} // namespace pb
} // namespace mpgos
