// Dense-contraction form of the per-block solver (full FP64 coupling matrices,
// up to 256 units per system) on v_mfma_f64_4x4x4f64.  Semantics as in
// pb_device.h; the coupling products C . [CPT_s0 CPT_s1 ...] of a workgroup's
// systems run on the matrix cores.
//
// The instruction computes four independent 4 x 4 x 4 products (block b = lanes
// with (lane / 4) % 4 == b: A[i][k] in lane i + 4b + 16k, B[k][j] in lane
// j + 4b + 16k, D[i][j] in lane j + 4b + 16i) and accumulates its four products
// as a chain of fused multiply-adds in k order (both probed on the MI355X), so
// chaining the column blocks in order equals the sequential
// fma(M[u][col], CPT[col], v) over col = 0 .. UPS-1 of the lane-per-pair form bit
// for bit.  Its four blocks take the four 4-row slices of a 16-unit tile
// against the same 4 systems.
//
// Layout.  A workgroup holds SPB = 4 NSL systems; wave w owns the 16-unit tiles
// w, w + waves, ... (TT of them), and lane l the units 16 tile + 4 ((l / 4) % 4)
// + l / 16 of the systems 4 slot + l % 4, slot < NSL: exactly the results that
// its own matrix instructions deliver.  Products therefore stay in registers;
// only the coupling terms (the B operand) go through LDS, in two buffers used
// in turn, with one barrier per stage.
// Units are padded to whole tiles: the matrix copy holds -0 in padded rows and
// columns and the coupling terms +0, so a padded column adds -0, which leaves
// every accumulator as it is; padded units are never stored.
//
// The matrix is read from a copy tiled per lane in column-block pairs
// (tile_pair_matrix): one 16-byte load per lane feeds two column blocks.  The
// leading pairs of every tile that fit into the LDS the workgroup leaves free are
// copied there at the start; the others stream from L2, one group ahead.
//
// What bounds it: 4096 rings of 256 units, the matrix cores, busy for 65 % of the
// cycles (34.6 of 53.2 million per SIMD and period; the rest are the right-hand
// sides and stage sums between the barriers, which all wavefronts of a workgroup
// reach together); few or small systems, the latency of a step.  Four periods
// of 4096 x 256 units 105.5 -> 90.7 ms and 1000 x 100 units 43.4 -> 8.9 ms
// against the forms before (products through LDS with two barriers per stage;
// one lane per unit where the units are no multiple of 32).
#pragma once

#include "pb_device.h"
#include "systems/system_base.h"

namespace mpgos {
namespace pb {

using systems::TimeTermsOf;

constexpr int kDenseMaxUnits = 256;
// Kernels for up to MT = 4, 8 and 16 tiles: one tile per wavefront up to 8, else
// two, so at most 8 wavefronts; the wavefronts per SIMD that they aim at.
__host__ __device__ constexpr int dense_tt(int MT) { return MT > 8 ? 2 : 1; }
__host__ __device__ constexpr int dense_waves(int MT) { return MT / dense_tt(MT); }
__host__ __device__ constexpr int dense_per_simd(int NSL, int MT) { return MT > 8 ? 2 : (MT > 4 ? 4 : 5) - NSL; }
constexpr int kDenseGroup = 2;             // column-block pairs per tile and load group
__host__ __device__ constexpr int dense_tiles(int UPS) { return (UPS + 15) >> 4; }
// column-block pairs of a tile, whole load groups
__host__ __device__ constexpr int dense_pairs(int UPS) { return ((UPS + 8 * kDenseGroup - 1) / (8 * kDenseGroup)) * kDenseGroup; }
// LDS row of one system's coupling terms: all columns of the padded matrix, 2
// doubles apart from a multiple of 16 so that the rows of 4 systems start 4
// banks apart
__host__ __device__ constexpr int dense_row(int UPS) { return dense_pairs(UPS) * 8 + 2; }
__host__ __device__ constexpr size_t dense_matrix_size(int UPS) { return (size_t)dense_tiles(UPS) * dense_pairs(UPS) * 128; }

// The pair-tiled copy of the dense coupling matrices (of their transposes for
// the adjoint sweep): for matrix i, tile t, column-block pair cp, lane l and j
// in {0, 1},
//   Mt[(((i * tiles + t) * pairs + cp) * 64 + l) * 2 + j] = M_i[row + col * UPS],
//   row = 16 t + l % 16, col = 4 (2 cp + j) + l / 16,
// and -0 where row or col lies outside the matrix.
template <bool TRANSPOSED>
__global__ void tile_pair_matrix(const double* M, double* Mt, int UPS, int NC)
{
    const int tiles = dense_tiles(UPS), pairs = dense_pairs(UPS);
    const size_t n = (size_t)NC * dense_matrix_size(UPS);
    const size_t k = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n) return;
    const int j = (int)(k & 1), l = (int)((k >> 1) & 63);
    size_t r = k >> 7;
    const int cp = (int)(r % pairs); r /= pairs;
    const int t = (int)(r % tiles);
    const int i = (int)(r / tiles);
    int row = t * 16 + (l & 15), col = 4 * (2 * cp + j) + (l >> 4);
    if (TRANSPOSED) { const int x = row; row = col; col = x; }
    Mt[k] = row < UPS && col < UPS ? M[(size_t)i * UPS * UPS + row + (size_t)col * UPS] : -0.0;
}

// System scope of the dense form (LDS): SysScope with the result of the last
// step kept apart from the flags the next one reduces.
template <class Sys>
struct DenseScope : SysScope<Sys, double> {
    int upd;                    // the last step was accepted
};

struct DenseLayout { size_t cpt, g, gi, blk, mt, total; };

template <class Scope, int NC, int NGP, int NiGP>
__host__ __device__ inline DenseLayout dense_layout(int SPB, int UPS, int sharedGlobals, int ldsPairs)
{
    constexpr int NCp = Pos<NC>::value;
    DenseLayout L;
    size_t o = ((size_t)SPB * sizeof(Scope) + 15) & ~(size_t)15;
    L.cpt = o;
    o += 2 * (size_t)NCp * SPB * dense_row(UPS) * sizeof(double);
    L.g = o;
    if (sharedGlobals) o += (size_t)NGP * sizeof(double);
    L.gi = o;
    if (sharedGlobals) o += (size_t)NiGP * sizeof(int);
    o = (o + 15) & ~(size_t)15;
    L.blk = o;
    o += 16;
    L.mt = o;
    o += (size_t)NCp * dense_tiles(UPS) * ldsPairs * 64 * 16;
    L.total = o;
    return L;
}

// The wave's index in the workgroup, in a scalar register.
__device__ __forceinline__ int wave_index() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

// Place of a lane in the workgroup (see the layout above).
template <int NSL, int TT>
struct DensePlace {
    static constexpr int SPB = 4 * NSL, PAIRS = NSL * TT;
    int l, w, nw, tiles, UPS, NS, urow;
    __device__ __forceinline__ DensePlace(int UPS_, int NS_)
        : l(threadIdx.x & 63), w(wave_index()), nw(blockDim.x >> 6), tiles(dense_tiles(UPS_)), UPS(UPS_), NS(NS_),
          urow(4 * ((threadIdx.x >> 2) & 3) + ((threadIdx.x & 63) >> 4)) {}
    __device__ __forceinline__ int sys(int s) const { return 4 * s + (l & 3); }                       // within the workgroup
    __device__ __forceinline__ int gsys(int s) const { return (int)blockIdx.x * SPB + sys(s); }
    __device__ __forceinline__ int unit(int k) const { return 16 * (w + k * nw) + urow; }
    __device__ __forceinline__ bool has(int k) const { return unit(k) < UPS; }
    __device__ __forceinline__ size_t at(int s, int k) const { return (size_t)gsys(s) * UPS + unit(k); }
    // one lane per system does its system-scope work: lane l % 4 of wave s % waves
    __device__ __forceinline__ bool leads(int s) const { return l < 4 && w == s % nw; }
};

// acc[i][s][k] = sum over columns of M_i of the wave's tiles against the coupling
// terms of the workgroup's systems (cptB: rows [coupling][system]), accumulated
// in column order.  Mt: tiled matrices in global memory, Ml: their leading
// ldsPairs pairs in LDS.
//
// One matrix, one tile per wave (up to 128 units) and few enough results per
// lane: the tile stays in registers (4 to 32 column blocks of one double per
// lane) for the whole Solve, and a stage reads only the coupling terms from
// LDS.  One period, from the streamed form: 1000 x 64 units 1.56 -> 1.36 ms,
// 2000 x 7 0.92 -> 0.81, 4096 x 64 3.0 -> 2.7, 1024 x 128 2.7 -> 2.6, 1000 x 100
// 2.4 (unchanged); the adjoint of 1024 x 128 units over two periods 12.2 -> 11.1 ms.
// What remains of a step of 1000 x 100 units (6.7 us): the products of two
// wavefronts on a SIMD (6 x 28 x 2 of 16 cycles, 2.4 us), right-hand sides,
// barriers and the controller (2.9 us without any products), and the first reads
// of each stage.
template <class Sys, int NSL, int MT>
__host__ __device__ constexpr bool dense_resident() { return Sys::NC == 1 && dense_tt(MT) == 1 && NSL * Sys::UD <= 4; }

template <int NSL, int MT>
struct ResidentContraction {
    using LD = const __attribute__((address_space(3))) double*;
    static constexpr int kBlocks = 4 * MT;   // column blocks of 16 MT units
    double a[kBlocks];
    int nb, RS, l;

    __device__ __forceinline__ ResidentContraction(const double* Mt, const double*, int, int UPS)
    {
        l = threadIdx.x & 63;
        nb = 2 * dense_pairs(UPS);           // a multiple of 4
        RS = dense_row(UPS);
        const double2* At = reinterpret_cast<const double2*>(Mt) + (size_t)wave_index() * dense_pairs(UPS) * 64 + l;
#pragma unroll
        for (int p = 0; p < kBlocks / 2; p++) {
            const double2 v = 2 * p < nb ? At[p * 64] : double2{0.0, 0.0};
            a[2 * p] = v.x;
            a[2 * p + 1] = v.y;
        }
    }
    __device__ __forceinline__ void prefetch() {}
    __device__ __forceinline__ void run(const double* cptB, double (&acc)[1][NSL][1]) const
    {
        const LD B = (LD)(cptB + (l & 3) * RS + (l >> 4));
        double b[2][4][NSL];
        auto terms = [&](int g) {
#pragma unroll
            for (int d = 0; d < 4; d++)
#pragma unroll
                for (int s = 0; s < NSL; s++) b[g & 1][d][s] = B[(4 * g + d) * 4 + s * 4 * RS];
        };
#pragma unroll
        for (int s = 0; s < NSL; s++) acc[0][s][0] = 0.0;
        terms(0);
#pragma unroll
        for (int g = 0; g < kBlocks / 4; g++) {
            const bool more = 4 * (g + 1) < nb;
            if (more) terms(g + 1);
#pragma unroll
            for (int d = 0; d < 4; d++)
#pragma unroll
                for (int s = 0; s < NSL; s++)
                    acc[0][s][0] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[4 * g + d], b[g & 1][d][s], acc[0][s][0], 0, 0, 0);
            if (!more) break;
        }
    }
};

// Otherwise both operands are streamed: A from LDS and L2, one group of pairs
// ahead (the wave's loads of the first global group are issued by prefetch()
// before the barrier).
template <int NC, int NSL, int TT>
struct StreamedContraction {
    struct alignas(16) Pair { double x, y; };
    using GP = const __attribute__((address_space(1))) Pair*;
    using LP = const __attribute__((address_space(3))) Pair*;
    using LD = const __attribute__((address_space(3))) double*;
    static constexpr int G = kDenseGroup;
    const Pair* At;              // the wave's first tile (uniform), lane offsets added at the load
    const Pair* Al;
    int gs, gi, ls, li, lp, pairs, RS, bi, l, nt;
    double a0[TT][2 * G];

    __device__ __forceinline__ StreamedContraction(const double* Mt, const double* Ml, int ldsPairs, int UPS)
    {
        const int w = wave_index(), nw = blockDim.x >> 6, tiles = dense_tiles(UPS);
        l = threadIdx.x & 63;
        pairs = dense_pairs(UPS);
        lp = ldsPairs;
        RS = dense_row(UPS);
        bi = 4 * NSL * RS;
        // tiles past the last one (waves with fewer than TT) repeat a tile; their results are not used
        At = reinterpret_cast<const Pair*>(Mt) + (size_t)(w < tiles ? w : 0) * pairs * 64;
        Al = reinterpret_cast<const Pair*>(Ml) + (w < tiles ? w : 0) * lp * 64;
        gs = nw * pairs * 64;
        gi = tiles * pairs * 64;
        ls = nw * lp * 64;
        li = tiles * lp * 64;
        nt = 0;
        for (int k = 0; k < TT; k++) if (w + k * nw < tiles) nt = k + 1;
    }
    __device__ __forceinline__ void load(double (*a)[2 * G], int i, int p) const
    {
#pragma unroll
        for (int k = 0; k < TT; k++) {
            const Pair* base = At + (i * gi + (k < nt ? k : 0) * gs + p * 64);
#pragma unroll
            for (int d = 0; d < G; d++) {
                const GP q = (GP)(base + (unsigned)(l + d * 64));
                a[k][2 * d] = q->x;
                a[k][2 * d + 1] = q->y;
            }
        }
    }
    __device__ __forceinline__ void load_lds(double (*a)[2 * G], int i, int p) const
    {
#pragma unroll
        for (int k = 0; k < TT; k++) {
            const Pair* base = Al + (i * li + (k < nt ? k : 0) * ls + p * 64);
#pragma unroll
            for (int d = 0; d < G; d++) {
                const LP q = (LP)(base + l + d * 64);
                a[k][2 * d] = q->x;
                a[k][2 * d + 1] = q->y;
            }
        }
    }
    __device__ __forceinline__ void group(const double (*a)[2 * G], LD B, int p, double (&acc)[NSL][TT]) const
    {
#pragma unroll
        for (int d = 0; d < 2 * G; d++) {
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                const double b = B[(2 * p + d) * 4 + s * 4 * RS];
#pragma unroll
                for (int k = 0; k < TT; k++) acc[s][k] = __builtin_amdgcn_mfma_f64_4x4x4f64(a[k][d], b, acc[s][k], 0, 0, 0);
            }
        }
    }
    __device__ __forceinline__ void prefetch()
    {
        if (lp < pairs) load(a0, 0, lp);
    }
    __device__ __forceinline__ void run(const double* cptB, double (&acc)[Pos<NC>::value][NSL][TT])
    {
#pragma unroll
        for (int i = 0; i < NC; i++) {
#pragma unroll
            for (int s = 0; s < NSL; s++)
#pragma unroll
                for (int k = 0; k < TT; k++) acc[i][s][k] = 0.0;
            const LD B = (LD)(cptB + (size_t)i * bi + (l & 3) * RS + (l >> 4));
            if (i > 0 && lp < pairs) load(a0, i, lp);
            double a1[TT][2 * G];
            for (int p = 0; p < lp; p += G) {
                load_lds(a1, i, p);
                group(a1, B, p, acc[i]);
            }
            if (lp < pairs) {
                // every load in the loop body is unconditional, so the wait
                // before a group's products counts only that group's loads
                int p = lp;
                for (; p + 2 * G < pairs; p += 2 * G) {
                    load(a1, i, p + G);
                    group(a0, B, p, acc[i]);
                    load(a0, i, p + 2 * G);
                    group(a1, B, p + G, acc[i]);
                }
                if (p + G < pairs) {
                    load(a1, i, p + G);
                    group(a0, B, p, acc[i]);
                    group(a1, B, p + G, acc[i]);
                } else {
                    group(a0, B, p, acc[i]);
                }
            }
        }
    }
};

template <class Sys, int NSL, int MT>
using DenseContraction = typename std::conditional<dense_resident<Sys, NSL, MT>(), ResidentContraction<NSL, MT>,
                                                   StreamedContraction<Sys::NC, NSL, dense_tt(MT)>>::type;

// Copies the leading ldsPairs pairs of every tile of the tiled matrices into LDS.
__device__ __forceinline__ void dense_stage_matrix(const double* Mt, unsigned char* lds, int NC, int UPS, int ldsPairs)
{
    using Q = double2;
    Q* lm = reinterpret_cast<Q*>(lds);
    const Q* src = reinterpret_cast<const Q*>(Mt);
    const int pairs = dense_pairs(UPS), n = NC * dense_tiles(UPS) * ldsPairs * 64;
    for (int k = threadIdx.x; k < n; k += blockDim.x) {
        const int r = k >> 6;
        lm[k] = src[((size_t)(r / ldsPairs) * pairs + r % ldsPairs) * 64 + (k & 63)];
    }
}

// min over the lanes of a 16-lane row that share l % 4 (in every lane of the row)
__device__ __forceinline__ double row_min4(double v)
{
    auto ror = [](double x, auto n) {
        const uint64_t b = math::bits(x);
        const uint32_t lo = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)b, 0x120 + decltype(n)::value, 0xf, 0xf, true);
        const uint32_t hi = (uint32_t)__builtin_amdgcn_update_dpp(0, (int)(uint32_t)(b >> 32), 0x120 + decltype(n)::value, 0xf, 0xf, true);
        return math::from_bits(((uint64_t)hi << 32) | lo);
    };
    v = __builtin_fmin(v, ror(v, std::integral_constant<int, 4>{}));
    return __builtin_fmin(v, ror(v, std::integral_constant<int, 8>{}));
}

// Stage times of the steppers as the forward pass evaluates them.
template <int ALG>
__device__ __forceinline__ double rk_stage_time(int s, double t, double h)
{
    using math::fma;
    if (ALG == MPGOS_RK4) return s == 0 ? t : (s == 3 ? t + h : t + 0.5 * h);
    switch (s) {
    case 0: return t;
    case 1: return fma(1.0 / 5.0, h, t);
    case 2: return fma(3.0 / 10.0, h, t);
    case 3: return fma(3.0 / 5.0, h, t);
    case 4: return t + h;
    default: return fma(7.0 / 8.0, h, t);
    }
}

// QUIET: no events, no user action after a step and no dense output (a.NDO == 0)
template <class Sys, int ALG, int NSL, int MT, bool REC, bool QUIET>
__device__ void pb_dense_body(const Args<Sys, double>& a)
{
    constexpr int TT = dense_tt(MT);
    using P = double;
    using CP = double;
    constexpr int UD = Sys::UD, NC = Sys::NC, NUP = Sys::NUP, NSP = Sys::NSP, NGP = Sys::NGP, NiGP = Sys::NiGP;
    constexpr int NUA = Sys::NUA, NiUA = Sys::NiUA, NSA = Sys::NSA, NiSA = Sys::NiSA, NE = Sys::NE;
    constexpr int NCp = Pos<NC>::value, NTT = TimeTermsOf<Sys>::n, ST = ALG == MPGOS_RK4 ? 4 : 6;
    using Place = DensePlace<NSL, TT>;
    constexpr int SPB = Place::SPB;
    using S = DenseScope<Sys>;
    using U = Unit<Sys, P>;
    using math::fma;

    extern __shared__ __align__(16) unsigned char mpgos_pb_lds[];
    const DenseLayout L = dense_layout<S, NC, NGP, NiGP>(SPB, a.UPS, a.sharedGlobals, a.ldsPairs);
    S* sys = reinterpret_cast<S*>(mpgos_pb_lds);
    P* cptBuf = reinterpret_cast<P*>(mpgos_pb_lds + L.cpt);
    int* blk = reinterpret_cast<int*>(mpgos_pb_lds + L.blk);      // [0] systems still running
    const int UPS = a.UPS, NS = a.NS, RS = dense_row(UPS);
    const int cptStride = NCp * SPB * RS;
    const size_t NU = (size_t)NS * UPS;
    const Place at(UPS, NS);
    const int tid = threadIdx.x;

    P* gPAR = a.gPAR;
    int* gPARi = a.gPARi;
    if (a.sharedGlobals) {
        P* lg = reinterpret_cast<P*>(mpgos_pb_lds + L.g);
        int* lgi = reinterpret_cast<int*>(mpgos_pb_lds + L.gi);
        for (int i = tid; i < NGP; i += blockDim.x) lg[i] = a.gPAR[i];
        for (int i = tid; i < NiGP; i += blockDim.x) lgi[i] = a.gPARi[i];
        gPAR = lg;
        gPARi = lgi;
    }
    for (int i = tid; i < 2 * cptStride; i += blockDim.x) cptBuf[i] = P(0);   // padded units and absent systems stay zero
    dense_stage_matrix(a.cTile, mpgos_pb_lds + L.mt, NC, UPS, a.ldsPairs);
    DenseContraction<Sys, NSL, MT> product(a.cTile, reinterpret_cast<const double*>(mpgos_pb_lds + L.mt), a.ldsPairs, UPS);
    int cIndex[NCp];
#pragma unroll
    for (int i = 0; i < NC; i++) cIndex[i] = a.cIndex[i];
    if (tid == 0) {
        const int first = (int)blockIdx.x * SPB, lim = a.nActive < NS ? a.nActive : NS;
        blk[0] = lim - first < SPB ? (lim > first ? lim - first : 0) : SPB;
    }

    // ---- system scope (PB-SOL:2285-2335)
    bool active[NSL];
#pragma unroll
    for (int s = 0; s < NSL; s++) active[s] = at.gsys(s) < NS && at.gsys(s) < a.nActive;
#pragma unroll
    for (int s = 0; s < NSL; s++) {
        if (at.leads(s)) {
            S& y = sys[at.sys(s)];
            const int g = at.gsys(s);
            if (active[s]) {
                y.TD[0] = a.TD[g]; y.TD[1] = a.TD[g + NS];
                y.t = a.T[g];
                y.dt = a.dt0; y.newDt = a.dt0;
                y.tc = P(0); y.dtP = a.dt0;
                for (int i = 0; i < NSP; i++) y.sPAR[i] = a.sPAR[g + i * NS];
                for (int i = 0; i < NSA; i++) y.sACC[i] = a.sACC[g + i * NS];
                for (int i = 0; i < NiSA; i++) y.sACCi[i] = a.sACCi[g + i * NS];
                for (int i = 0; i < NC; i++) y.strength[i] = a.strength[g + i * NS];
                y.DOidx = a.DOidx[g];
                y.updDO = 1; y.skipped = 0; y.term = 0; y.udt = 0; y.update = 0; y.doT = P(0);
            } else {
                y.t = y.dt = y.newDt = P(0);
                for (int i = 0; i < NSP; i++) y.sPAR[i] = P(0);   // time terms are evaluated for it
                y.term = 1; y.update = 0; y.updDO = 0;
            }
            y.upd = 0;
            y.nacc = 0; y.nrej = 0; y.status = 0;
        }
    }

    // ---- unit scope in registers
    P X[NSL][TT][UD], uPAR[NSL][TT][Pos<NUP>::value], uACC[NSL][TT][Pos<NUA>::value], EF[NSL][TT][Pos<NE>::value];
    int uACCi[NSL][TT][Pos<NiUA>::value];
    auto each = [&](auto&& f) {
#pragma unroll
        for (int s = 0; s < NSL; s++)
#pragma unroll
            for (int k = 0; k < TT; k++) f(s, k);
    };
    // this lane has a unit of an active system there
    auto mine = [&](int s, int k) { return active[s] && at.has(k); };
    each([&](int s, int k) {
        const bool m = mine(s, k);
        const size_t g = at.at(s, k);
#pragma unroll
        for (int c = 0; c < UD; c++) X[s][k][c] = m ? a.X[g + c * NU] : P(0);
#pragma unroll
        for (int c = 0; c < NUP; c++) uPAR[s][k][c] = m ? a.uPAR[g + c * NU] : P(0);
#pragma unroll
        for (int c = 0; c < NUA; c++) uACC[s][k][c] = m ? a.uACC[g + c * NU] : P(0);
#pragma unroll
        for (int c = 0; c < NiUA; c++) uACCi[s][k][c] = m ? a.uACCi[g + c * NU] : 0;
    });
    __syncthreads();

#define MPGOS_PB_MY(s) sys[at.sys(s)]
#define MPGOS_PB_USER(s, k, TT_, DTT) TT_, DTT, MPGOS_PB_MY(s).TD, X[s][k], uPAR[s][k], MPGOS_PB_MY(s).sPAR, gPAR, gPARi, uACC[s][k], uACCi[s][k], MPGOS_PB_MY(s).sACC, MPGOS_PB_MY(s).sACCi
    // ---- initialisation (PB-SOL:2465-2528)
    each([&](int s, int k) {
        if (mine(s, k)) Sys::template Initialization<P>(at.gsys(s), at.unit(k), MPGOS_PB_MY(s).DOidx, MPGOS_PB_USER(s, k, MPGOS_PB_MY(s).t, MPGOS_PB_MY(s).dt));
    });
    __syncthreads();
    if (NE > 0) {
        each([&](int s, int k) {
            if (mine(s, k)) Sys::template EventFunction<P>(at.gsys(s), at.unit(k), EF[s][k], MPGOS_PB_USER(s, k, MPGOS_PB_MY(s).t, MPGOS_PB_MY(s).dt));
        });
        __syncthreads();
    }
    if (!QUIET && a.NDO > 0) {
        // first store (the reference stores unconditionally; skipped once the buffer is full)
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            if (active[s] && MPGOS_PB_MY(s).DOidx < a.NDO) {
                const int d = MPGOS_PB_MY(s).DOidx;
#pragma unroll
                for (int k = 0; k < TT; k++)
#pragma unroll
                    for (int c = 0; c < UD; c++)
                        if (at.has(k)) a.DOx[at.at(s, k) + c * NU + (size_t)d * NU * UD] = X[s][k][c];
                if (at.leads(s)) a.DOt[at.gsys(s) + (size_t)d * NS] = MPGOS_PB_MY(s).t;
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            S& y = MPGOS_PB_MY(s);
            if (at.leads(s) && active[s] && y.DOidx < a.NDO) {
                y.DOidx++;
                y.skipped = 0;
                y.doT = dmin<P>(y.t + a.doMinDt, y.TD[1]);
            }
        }
        __syncthreads();
    }
    if (REC) {                  // checkpoint 0: the initial unit states
        each([&](int s, int k) {
#pragma unroll
            for (int c = 0; c < UD; c++)
                if (mine(s, k)) a.recX[(size_t)c * NU + at.at(s, k)] = X[s][k][c];
        });
    }

    // ---- step initialisation of a running system (PB-SOL:2535-2549)
    auto begin_step = [&](auto& y) {
        y.update = 1; y.isfin = 1; y.end = 0;
        y.dt = y.newDt;
        const CP remaining = y.TD[1] - y.t;
        if (y.dt > remaining) { y.dt = remaining; y.end = 1; }
        y.ratioBits = order_bits<CP>(CP(1e30));
        y.eventBits = ~0ull;            // no candidate yet (above every finite step)
        y.corrected = 0;
    };
    // ---- controller of a running system (PB-CTL:424-542)
    auto control = [&](auto& y) {
        if (ALG == MPGOS_RKCK45) {
            const CP R = from_order_bits<CP>(y.ratioBits);
            CP fac = CP(0.8) * math::pow_ctrl(R, y.update == 1 ? CP(1.0 / 5.0) : CP(1.0 / 4.0));
            if (!math::isfinite(fac)) y.isfin = 0;
            if (y.isfin == 0) {
                fac = a.shrink;
                y.update = 0;
                if (y.dt < a.dtmin * CP(1.01)) { y.term = 1; y.status |= MPGOS_STATUS_NONFINITE_MIN_STEP; }
            } else if (y.dt < a.dtmin * CP(1.01)) {
                y.update = 1;
                y.status |= MPGOS_STATUS_MIN_STEP_REACHED;
            }
            fac = dmin<CP>(fac, a.grow);
            fac = dmax<CP>(fac, a.shrink);
            CP nd = y.dt * fac;
            nd = dmin<CP>(nd, a.dtmax);
            nd = dmax<CP>(nd, a.dtmin);
            y.newDt = nd;
        } else {
            if (y.isfin == 0) { y.term = 1; y.update = 0; y.status |= MPGOS_STATUS_NONFINITE_RK4; }
            y.newDt = a.dt0;
        }
    };
    // (t, h) of the accepted step n of system g (record pass)
    auto record_step = [&](auto& y, int g) {
        const long long n = y.nacc;
        if (n < a.recStepCap) { a.recT[(size_t)n * NS + g] = y.t; a.recH[(size_t)n * NS + g] = y.dt; }
        else y.status |= MPGOS_STATUS_CHECKPOINT_OVERFLOW;
        if ((n + 1) % a.recK == 0 && (n + 1) / a.recK >= a.recCkCap) y.status |= MPGOS_STATUS_CHECKPOINT_OVERFLOW;
    };
    auto record_state = [&](int s, long long n) {   // after accepted step n
        if ((n + 1) % a.recK != 0) return;
        const long long c0 = (n + 1) / a.recK;
        if (c0 >= a.recCkCap) return;
#pragma unroll
        for (int k = 0; k < TT; k++)
#pragma unroll
            for (int c = 0; c < UD; c++)
                if (at.has(k)) a.recX[((size_t)c0 * UD + c) * NU + at.at(s, k)] = X[s][k][c];
    };

    int buf = 0;
    // right-hand sides of this lane's units at (Y, T), then the coupling terms
    constexpr int PER = 64 / SPB;        // stages whose time terms one evaluation covers
    P tterm[(ST + PER - 1) / PER][Pos<NTT>::value], tt[NSL][Pos<NTT>::value];
    auto fetch_terms = [&](int stage) {
#pragma unroll
        for (int s = 0; s < NSL; s++)
#pragma unroll
            for (int i = 0; i < NTT; i++) tt[s][i] = __shfl(tterm[stage / PER][i], (stage % PER) * SPB + at.sys(s));
    };
    // coupling strengths and, where no user code can change them during the
    // steps, system parameters in registers: a stage waits for LDS only where
    // it needs the other units' coupling terms
    constexpr bool keepPar = QUIET && NSP <= 4;
    P strength[NSL][NCp], par[NSL][Pos<NSP>::value];
#pragma unroll
    for (int s = 0; s < NSL; s++) {
#pragma unroll
        for (int i = 0; i < NC; i++) strength[s][i] = MPGOS_PB_MY(s).strength[i];
#pragma unroll
        for (int i = 0; i < NSP; i++) par[s][i] = keepPar ? MPGOS_PB_MY(s).sPAR[i] : P(0);
    }
    auto rhs = [&](int stage, P (*F)[TT][UD], P (*Y)[TT][UD], const P* T, const bool* run) {
        P* cpt = cptBuf + (size_t)buf * cptStride;
        P CPF[NSL][TT][NCp];
        product.prefetch();
        each([&](int s, int k) {
            if (run[s] && at.has(k)) {
                P cp[NCp];
#pragma unroll
                for (int i = 0; i < NC; i++) cp[i] = CPF[s][k][i] = P(0);
                S& y = MPGOS_PB_MY(s);
                P* sPAR = keepPar ? par[s] : y.sPAR;
                if constexpr (NTT > 0)
                    Sys::template OdeFunctionTT<P>(at.gsys(s), at.unit(k), F[s][k], Y[s][k], T[s], tt[s], uPAR[s][k], sPAR, gPAR,
                                                   gPARi, uACC[s][k], uACCi[s][k], y.sACC, y.sACCi, cp, CPF[s][k]);
                else
                    Sys::template OdeFunction<P>(at.gsys(s), at.unit(k), F[s][k], Y[s][k], T[s], uPAR[s][k], sPAR, gPAR, gPARi,
                                                 uACC[s][k], uACCi[s][k], y.sACC, y.sACCi, cp, CPF[s][k]);
#pragma unroll
                for (int i = 0; i < NC; i++) cpt[(i * SPB + at.sys(s)) * RS + at.unit(k)] = cp[i];
            }
        });
        if (stage + 1 < ST) fetch_terms(stage + 1);
        lds_barrier();
        P v[NCp][NSL][TT];
        product.run(cpt, v);
        each([&](int s, int k) {
#pragma unroll
            for (int i = 0; i < NC; i++) U::add(cIndex[i], strength[s][i] * CPF[s][k][i], v[i][s][k], F[s][k]);
        });
        buf ^= 1;
    };

#pragma unroll
    for (int s = 0; s < NSL; s++)
        if (at.leads(s) && MPGOS_PB_MY(s).term == 0) begin_step(MPGOS_PB_MY(s));
    __syncthreads();
    while (blk[0] > 0) {
        P h[NSL], t[NSL], T[NSL];
        bool run[NSL];
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            h[s] = MPGOS_PB_MY(s).dt;
            t[s] = MPGOS_PB_MY(s).t;
            run[s] = MPGOS_PB_MY(s).term == 0;
        }
        if constexpr (NTT > 0) {
            // the time terms of the step's stages: each lane evaluates those of
            // one stage of one system, once per wavefront instead of every
            // stage in every lane; rhs() fetches them from there
#pragma unroll
            for (int e = 0; e * PER < ST; e++)
                Sys::template TimeTerms<P>(rk_stage_time<ALG>(e * PER + at.l / SPB, sys[at.l % SPB].t, sys[at.l % SPB].dt),
                                           sys[at.l % SPB].sPAR, tterm[e]);
            fetch_terms(0);
        }
        P next[NSL][TT][UD], err[NSL][TT][UD];
        auto stage_time = [&](int st) {
#pragma unroll
            for (int s = 0; s < NSL; s++) T[s] = rk_stage_time<ALG>(st, t[s], h[s]);
        };
        // Y = value(s, k, c) for every unit component of the lane
        auto fill = [&](P (*Y)[TT][UD], auto&& value) {
            each([&](int s, int k) {
#pragma unroll
                for (int c = 0; c < UD; c++) Y[s][k][c] = value(s, k, c);
            });
        };
        if (ALG == MPGOS_RK4) {
            // PB-STP:2016-2224
            P k[NSL][TT][UD], Y[NSL][TT][UD];
            stage_time(0);
            rhs(0, next, X, T, run);
            fill(Y, [&](int s, int q, int c) { return fma(next[s][q][c] * P(0.5), h[s], X[s][q][c]); });
            stage_time(1);
            rhs(1, k, Y, T, run);
            fill(next, [&](int s, int q, int c) { return fma(P(2), k[s][q][c], next[s][q][c]); });
            fill(Y, [&](int s, int q, int c) { return fma(k[s][q][c] * P(0.5), h[s], X[s][q][c]); });
            stage_time(2);
            rhs(2, k, Y, T, run);
            fill(next, [&](int s, int q, int c) { return fma(P(2.0), k[s][q][c], next[s][q][c]); });
            fill(Y, [&](int s, int q, int c) { return fma(k[s][q][c], h[s], X[s][q][c]); });
            stage_time(3);
            rhs(3, k, Y, T, run);
            fill(next, [&](int s, int q, int c) { return fma(h[s] * (next[s][q][c] + k[s][q][c]), P(1.0 / 6.0), X[s][q][c]); });
        } else {
            // PB-STP:2227-2544, the sums over stages formed as the stages become
            // known (in their order): at most three stage vectors live across a
            // contraction
            P k1[NSL][TT][UD], k2[NSL][TT][UD], k3[NSL][TT][UD], k[NSL][TT][UD], Y[NSL][TT][UD], sum6[NSL][TT][UD];
            stage_time(0);
            rhs(0, k1, X, T, run);
            fill(Y, [&](int s, int q, int c) { return fma(k1[s][q][c] * P(1.0 / 5.0), h[s], X[s][q][c]); });
            stage_time(1);
            rhs(1, k2, Y, T, run);
            fill(Y, [&](int s, int q, int c) { return fma(fma(k2[s][q][c], P(9.0 / 40.0), k1[s][q][c] * P(3.0 / 40.0)), h[s], X[s][q][c]); });
            stage_time(2);
            rhs(2, k3, Y, T, run);
            fill(Y, [&](int s, int q, int c) {
                return fma(fma(k3[s][q][c], P(6.0 / 5.0), fma(k2[s][q][c], P(-9.0 / 10.0), k1[s][q][c] * P(3.0 / 10.0))), h[s], X[s][q][c]);
            });
            stage_time(3);
            rhs(3, k, Y, T, run);
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
            fill(err, [&](int s, int q, int c) {
                return fma(k[s][q][c], P(125.0 / 594.0 - 13525.0 / 55296.0), fma(k3[s][q][c], P(250.0 / 621.0 - 18575.0 / 48384.0),
                           k1[s][q][c] * P(37.0 / 378.0 - 2825.0 / 27648.0)));
            });
            stage_time(4);
            rhs(4, k, Y, T, run);
            fill(Y, [&](int s, int q, int c) { return fma(fma(k[s][q][c], P(253.0 / 4096.0), sum6[s][q][c]), h[s], X[s][q][c]); });
            fill(err, [&](int s, int q, int c) { return fma(k[s][q][c], P(0.0 - 277.0 / 14336.0), err[s][q][c]); });
            stage_time(5);
            rhs(5, k, Y, T, run);
            fill(next, [&](int s, int q, int c) { return fma(fma(k[s][q][c], P(512.0 / 1771.0), next[s][q][c]), h[s], X[s][q][c]); });
            fill(err, [&](int s, int q, int c) {
                return fma(h[s], math::fabs(fma(k[s][q][c], P(512.0 / 1771.0 - 1.0 / 4.0), err[s][q][c])), P(1e-18));
            });
        }
        // ---- acceptance, finiteness and step ratio of each system over its units
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            CP R = CP(1e30);
            bool ok = true, fin = true;
#pragma unroll
            for (int k = 0; k < TT; k++) {
                if (!at.has(k)) continue;
#pragma unroll
                for (int c = 0; c < UD; c++) {
                    fin = fin && math::isfinite(next[s][k][c]);
                    if (ALG == MPGOS_RKCK45) {
                        const CP tol = dmax<CP>(a.rtol[c] * dmax<CP>(math::fabs(next[s][k][c]), math::fabs(X[s][k][c])), a.atol[c]);
                        fin = fin && math::isfinite(err[s][k][c]);
                        ok = ok && err[s][k][c] < tol;
                        R = dmin<CP>(R, tol / err[s][k][c]);
                    }
                }
            }
            S& y = MPGOS_PB_MY(s);
            if (run[s]) {
                if (!fin) y.isfin = 0;
                if (!ok) y.update = 0;
            }
            if (ALG == MPGOS_RKCK45) {
                // one LDS atomic per 16-lane row and system (min does not
                // depend on the order); absent and finished systems' words are
                // never read
                R = row_min4(R);
                if ((at.l & 12) == 0) atomicMin(&y.ratioBits, order_bits<CP>(R));
            }
        }
        if (QUIET) lds_barrier();           // no user code: what lanes exchange is in LDS
        else __syncthreads();
        if constexpr (QUIET) {
            // no user code between controller and next step: one lane per
            // system does all of its system scope
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                if (at.leads(s)) {
                    // read and written back as a whole: the LDS accesses of a
                    // statement by statement form wait for one another (with
                    // LDS-only barriers around: 2000 x 7 units 0.81 -> 0.76 ms,
                    // 1000 x 64 1.33 -> 1.29, 1000 x 100 2.36 -> 2.31)
                    S& z = MPGOS_PB_MY(s);
                    DenseScope<Sys> y;
                    y.term = z.term; y.isfin = z.isfin; y.update = z.update; y.end = z.end; y.status = z.status;
                    y.nacc = z.nacc; y.nrej = z.nrej; y.ratioBits = z.ratioBits; y.dt = z.dt; y.t = z.t; y.TD[1] = z.TD[1];
                    y.newDt = z.newDt;
                    y.upd = 0;
                    if (y.term == 0) {
                        control(y);
                        y.upd = y.update;
                        if (y.upd) {
                            if (REC) record_step(y, at.gsys(s));
                            y.t += y.dt;
                            y.nacc++;
                            if (y.end == 1) y.term = 1;
                        } else if (y.term == 0) {
                            y.nrej++;
                        }
                        if (y.term == 0) begin_step(y);
                        else atomicSub(&blk[0], 1);
                        z.dt = y.dt; z.t = y.t; z.newDt = y.newDt; z.ratioBits = y.ratioBits;
                        z.isfin = y.isfin; z.update = y.update; z.end = y.end; z.status = y.status;
                        z.nacc = y.nacc; z.nrej = y.nrej; z.term = y.term;
                    }
                    z.upd = y.upd;
                }
            }
            lds_barrier();
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                if (MPGOS_PB_MY(s).upd) {
#pragma unroll
                    for (int k = 0; k < TT; k++)
#pragma unroll
                        for (int c = 0; c < UD; c++) X[s][k][c] = next[s][k][c];
                    if (REC) record_state(s, MPGOS_PB_MY(s).nacc - 1);
                }
            }
        } else {
        // ---- with user code, as the reference orders it
#pragma unroll
        for (int s = 0; s < NSL; s++)
            if (at.leads(s) && MPGOS_PB_MY(s).term == 0) control(MPGOS_PB_MY(s));
        __syncthreads();
        // events (PB-SOL:2618-2655, PB-EVT:215-268)
        P EFn[NSL][TT][Pos<NE>::value];
        if (NE > 0) {
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                S& y = MPGOS_PB_MY(s);
                const P tn = y.t + y.dt;
                if (y.term == 0) {
                    bool corr = false;
                    CP ev = y.dt;
#pragma unroll
                    for (int k = 0; k < TT; k++) {
                        if (!at.has(k)) continue;
                        // the event function of the candidate state, at the end of the step
                        Sys::template EventFunction<P>(at.gsys(s), at.unit(k), EFn[s][k], tn, y.newDt, y.TD, next[s][k], uPAR[s][k], y.sPAR,
                                                       gPAR, gPARi, uACC[s][k], uACCi[s][k], y.sACC, y.sACCi);
                        if (y.update == 1) {
#pragma unroll
                            for (int i = 0; i < NE; i++) {
                                const P tol = a.etol[i];
                                if ((EF[s][k][i] > tol && EFn[s][k][i] < -tol && a.edir[i] <= 0) ||
                                    (EF[s][k][i] < -tol && EFn[s][k][i] > tol && a.edir[i] >= 0)) {
                                    ev = dmin<CP>(ev, -EF[s][k][i] / (EFn[s][k][i] - EF[s][k][i]) * y.dt);
                                    corr = true;
                                }
                            }
                        }
                    }
                    if (corr) {
                        atomicMin(&y.eventBits, order_bits<CP>(ev));
                        atomicOr(&y.corrected, 1);
                    }
                }
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                S& y = MPGOS_PB_MY(s);
                if (at.leads(s) && y.term == 0 && y.corrected == 1) {
                    const CP ev = dmin<CP>(y.dt, from_order_bits<CP>(y.eventBits));   // corrected: one candidate at least
                    if (ev < a.dtmin) y.status |= MPGOS_STATUS_EVENT_OMITTED;
                    else { y.newDt = ev; y.update = 0; }
                }
            }
            __syncthreads();
        }
        // update (PB-SOL:2670-2681): a finished system's update flag stays 0
        bool upd[NSL];
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            upd[s] = run[s] && MPGOS_PB_MY(s).update == 1;
            if (upd[s]) {
#pragma unroll
                for (int k = 0; k < TT; k++)
#pragma unroll
                    for (int c = 0; c < UD; c++) X[s][k][c] = next[s][k][c];
                if (REC) {
                    record_state(s, MPGOS_PB_MY(s).nacc);
                    if (at.leads(s)) record_step(MPGOS_PB_MY(s), at.gsys(s));
                }
            }
        }
        __syncthreads();
#pragma unroll
        for (int s = 0; s < NSL; s++)
            if (at.leads(s) && upd[s]) MPGOS_PB_MY(s).t += MPGOS_PB_MY(s).dt;
        __syncthreads();
        each([&](int s, int k) {
            if (upd[s] && at.has(k))
                Sys::template ActionAfterSuccessfulTimeStep<P>(at.gsys(s), at.unit(k), MPGOS_PB_MY(s).udt, MPGOS_PB_USER(s, k, MPGOS_PB_MY(s).t, MPGOS_PB_MY(s).dt));
        });
        __syncthreads();
        if (NE > 0) {
            each([&](int s, int k) {
                if (upd[s] && at.has(k)) {
#pragma unroll
                    for (int i = 0; i < NE; i++) {
                        const P tol = a.etol[i];
                        if ((EF[s][k][i] > tol && math::fabs(EFn[s][k][i]) < tol && a.edir[i] <= 0) ||
                            (EF[s][k][i] < -tol && math::fabs(EFn[s][k][i]) < tol && a.edir[i] >= 0))
                            Sys::template ActionAfterEventDetection<P>(at.gsys(s), at.unit(k), i, MPGOS_PB_MY(s).udt, MPGOS_PB_USER(s, k, MPGOS_PB_MY(s).t, MPGOS_PB_MY(s).dt));
                    }
                }
            });
            __syncthreads();
            each([&](int s, int k) {
                if (upd[s] && at.has(k)) {
                    Sys::template EventFunction<P>(at.gsys(s), at.unit(k), EFn[s][k], MPGOS_PB_USER(s, k, MPGOS_PB_MY(s).t, MPGOS_PB_MY(s).newDt));
#pragma unroll
                    for (int i = 0; i < NE; i++) EF[s][k][i] = EFn[s][k][i];
                }
            });
            __syncthreads();
        }
        // dense output (PB-DO:312-395)
        if (a.NDO > 0) {
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                S& y = MPGOS_PB_MY(s);
                if (at.leads(s)) {
                    int st = 0;
                    if (upd[s]) {
                        st = (y.DOidx < a.NDO && y.doT < y.t && y.skipped >= a.doFreq - 1) ? 1 : 0;
                        if (y.DOidx < a.NDO && (y.end == 1 || y.udt == 1)) st = 1;
                    }
                    y.updDO = st;
                }
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                S& y = MPGOS_PB_MY(s);
                if (y.updDO == 1 && upd[s]) {
                    const int d = y.DOidx;
#pragma unroll
                    for (int k = 0; k < TT; k++)
#pragma unroll
                        for (int c = 0; c < UD; c++)
                            if (at.has(k)) a.DOx[at.at(s, k) + c * NU + (size_t)d * NU * UD] = X[s][k][c];
                    if (at.leads(s)) a.DOt[at.gsys(s) + (size_t)d * NS] = y.t;
                }
            }
            __syncthreads();
#pragma unroll
            for (int s = 0; s < NSL; s++) {
                S& y = MPGOS_PB_MY(s);
                if (at.leads(s) && upd[s]) {
                    if (y.updDO == 1) {
                        y.DOidx++;
                        y.skipped = 0;
                        y.doT = dmin<P>(y.t + a.doMinDt, y.TD[1]);
                    } else {
                        y.skipped++;
                    }
                }
            }
        }
        // statistics and termination (PB-SOL:2797-2807)
#pragma unroll
        for (int s = 0; s < NSL; s++) {
            S& y = MPGOS_PB_MY(s);
            if (at.leads(s) && run[s]) {
                if (upd[s]) {
                    y.nacc++;
                    if (y.end == 1 || y.udt == 1) y.term = 1;
                } else if (y.term == 0) {
                    y.nrej++;
                }
                if (y.term == 0) begin_step(y);
                else atomicSub(&blk[0], 1);
            }
        }
        __syncthreads();
        }
    }
    __syncthreads();
    // ---- finalisation and write-back (PB-SOL:2814-2887)
    each([&](int s, int k) {
        if (mine(s, k)) Sys::template Finalization<P>(at.gsys(s), at.unit(k), MPGOS_PB_MY(s).DOidx, MPGOS_PB_USER(s, k, MPGOS_PB_MY(s).t, MPGOS_PB_MY(s).dt));
    });
    __syncthreads();
    each([&](int s, int k) {
        if (mine(s, k)) {
            const size_t g = at.at(s, k);
#pragma unroll
            for (int c = 0; c < UD; c++) a.X[g + c * NU] = X[s][k][c];
#pragma unroll
            for (int c = 0; c < NUA; c++) a.uACC[g + c * NU] = uACC[s][k][c];
#pragma unroll
            for (int c = 0; c < NiUA; c++) a.uACCi[g + c * NU] = uACCi[s][k][c];
        }
    });
#pragma unroll
    for (int s = 0; s < NSL; s++) {
        if (at.leads(s) && active[s]) {
            const S& y = MPGOS_PB_MY(s);
            const int g = at.gsys(s);
            a.T[g] = y.t;
            a.TD[g] = y.TD[0]; a.TD[g + NS] = y.TD[1];
            for (int i = 0; i < NSA; i++) a.sACC[g + i * NS] = y.sACC[i];
            for (int i = 0; i < NiSA; i++) a.sACCi[g + i * NS] = y.sACCi[i];
            a.DOidx[g] = y.DOidx;
            a.nacc[g] = y.nacc;
            a.nrej[g] = y.nrej;
            a.status[g] = y.status;
        }
    }
#undef MPGOS_PB_USER
#undef MPGOS_PB_MY
}

// Wavefronts per SIMD that the registers have to allow: one result per lane 4
// with at most 4 tiles and 3 with 8; two results 3 and 2; else 2.
template <class Sys, int ALG, int NSL, int MT, bool REC, bool QUIET>
__global__ void __launch_bounds__(64 * dense_waves(MT), dense_per_simd(NSL, MT)) pb_dense_kernel(Args<Sys, double> a)
{
    pb_dense_body<Sys, ALG, NSL, MT, REC, QUIET>(a);
}

} // namespace pb
} // namespace mpgos
