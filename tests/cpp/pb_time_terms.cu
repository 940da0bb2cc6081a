// A per-block system of one's own whose time terms depend on a parameter: it
// names them (NTT, TimeTerms, OdeFunctionTT) and brings OdeVJP but no OdeVJPTT,
// which only systems with terms of the time alone provide.  Gradient and end
// state in the matrix-core form, with one and with several results per lane,
// against one lane per unit, which evaluates no shared terms, bit for bit.
// Prints "same" and returns 0, or says what differs and returns 1.  With an
// argument: the forms it would choose, without a device.
#include <cstdio>
#include <string>
#include <utility>
#include <vector>

#include "pb_engine.h"
#include "systems/system_base.h"

namespace mpgos {
void set_error(const std::string& msg) { std::fprintf(stderr, "%s\n", msg.c_str()); }
} // namespace mpgos

// x'' + k x' + x = B cos(w t) + coupling, sPAR = (B, w)
struct Named : mpgos::systems::PBNoCallbacks {
    static constexpr const char* name = "named";
    static constexpr int UD = 2, NC = 1, NUP = 1, NSP = 2, NGP = 0, NiGP = 0, NUA = 0, NiUA = 0, NSA = 0, NiSA = 0, NE = 0;
    static constexpr int NTT = 1;
    static constexpr bool TT_TIME_ONLY = false;
    template <class P> __device__ static void TimeTerms(P T, P* sPAR, P* tt) { tt[0] = mpgos::math::cos(sPAR[1] * T); }
    template <class P>
    __device__ static void OdeFunctionTT(int, int, P* F, P* X, P, const P* tt, P* uPAR, P* sPAR, P*, int*, P*, int*, P*, int*, P* CPT, P* CPF)
    {
        F[0] = X[1];
        F[1] = mpgos::math::fma(-uPAR[0], X[1], sPAR[0] * tt[0]) - X[0];
        CPT[0] = X[0];
        CPF[0] = P(1);
    }
    template <class P>
    __device__ static void OdeFunction(int sid, int uid, P* F, P* X, P T, P* uPAR, P* sPAR, P* gPAR, int* gPARi, P* uACC, int* uACCi, P* sACC,
                                       int* sACCi, P* CPT, P* CPF)
    {
        P tt[NTT];
        TimeTerms<P>(T, sPAR, tt);
        OdeFunctionTT<P>(sid, uid, F, X, T, tt, uPAR, sPAR, gPAR, gPARi, uACC, uACCi, sACC, sACCi, CPT, CPF);
    }
    template <class P>
    __device__ static void OdeVJP(int, int, const P* kbF, const P* kbCPT, const P*, P* X, P T, P* uPAR, P* sPAR, P*, int*, P*, int*, P*, int*,
                                  P* gX, P* gU, P* gS)
    {
        gX[0] = kbCPT[0] - kbF[1];
        gX[1] = kbF[0] - uPAR[0] * kbF[1];
        gU[0] = -X[1] * kbF[1];
        gS[0] = mpgos::math::cos(sPAR[1] * T) * kbF[1];
        gS[1] = -sPAR[0] * mpgos::math::sin(sPAR[1] * T) * T * kbF[1];
    }
    template <class P>
    __device__ static void Initialization(int, int uid, int&, P& T, P&, P* TD, P*, P*, P*, P*, int*, P*, int*, P*, int*)
    {
        if (uid == 0) T = TD[0];
    }
};

static bool run(int algorithm, int ns, int ups, int kernel, std::vector<unsigned char>& out)
{
    mpgos::pb::Solver<Named, double> S;
    if (S.init(algorithm, ns, ups, 1, 0, 0, 0, 0) || S.option(MPGOS_PB_COUPLING_KERNEL, 0, kernel)) return false;
    const int nu = ns * ups;
    for (int i = 0; i < ns; i++) {
        S.TD.h[ns + i] = 2.0 + 0.01 * (i % 7);
        S.sPAR.h[i] = 0.5 + 0.01 * (i % 50);
        S.sPAR.h[ns + i] = 1.0 + 0.001 * (i % 90);
        S.strength.h[i] = 1.0;
    }
    for (int u = 0; u < nu; u++) {
        S.uPAR.h[u] = 0.2 + 0.001 * (u % 11);
        for (int c = 0; c < 2; c++) {
            S.X.h[c * nu + u] = 0.1 * ((u + 3 * c) % 13) - 0.6;
            S.lamB.h[c * nu + u] = 0.3 - 0.05 * ((u + c) % 9);
        }
    }
    for (int k = 0; k < ups * ups; k++) S.cMat.h[k] = 0.01 * (k % 5 - 2);
    S.cIndex.h[0] = 1;
    for (int c = 0; c < 2; c++) { S.rtol[c] = 1e-8; S.atol[c] = 1e-8; }
    S.dt0 = 0.02;
    if (S.sync(MPGOS_PB_ALL, true) || S.sync(MPGOS_PB_ADJOINT_STATE, true) || S.adjoint_record(16, 40, 400) || S.adjoint_reverse() ||
        S.sync(MPGOS_PB_ALL, false) || S.sync(MPGOS_PB_ADJOINT_STATE, false) || S.sync(MPGOS_PB_UNIT_PARAMETER_GRADIENT, false) ||
        S.sync(MPGOS_PB_SYSTEM_PARAMETER_GRADIENT, false) || S.synchronise_device())
        return false;
    auto add = [&](const auto& b) { out.insert(out.end(), (const unsigned char*)b.h, (const unsigned char*)b.h + b.bytes()); };
    add(S.X); add(S.T); add(S.nacc); add(S.status); add(S.lamB); add(S.gUB); add(S.gSB);
    for (int i = 0; i < ns; i++)
        if (S.status.h[i] != 0 || S.nacc.h[i] < 16) return false;
    return true;
}

// The choice of the reverse pass where the LDS holds the Solve's data and not
// the step sizes of the reverse pass as well (no device needed).
static int forms()
{
    mpgos::pb::Solver<Named, double> S;
    S.NS = 40; S.UPS = 100; S.cus = 256;
    using namespace mpgos::pb;
    const size_t solve = dense_layout<DenseScope<Named>, 1, 0, 0>(4, 100, 1, 0).total, reverse = rev_lds_bytes<Named>(4, 100, 0);
    bool ok = reverse > solve;
    S.ldsMax = reverse;
    ok = ok && S.coupling_form() == kDenseCoupling && S.reverse_form() == kDenseCoupling;
    S.ldsMax = solve;
    ok = ok && S.coupling_form() == kDenseCoupling && S.reverse_form() == kLaneCoupling;
    S.couplingKernel = 2;                              // asked for: refused later, as too large
    ok = ok && S.reverse_form() == kDenseCoupling;
    std::printf(ok ? "forms\n" : "wrong form\n");
    return ok ? 0 : 1;
}

int main(int argc, char**)
{
    if (argc > 1) return forms();
    for (int algorithm : {MPGOS_RK4, MPGOS_RKCK45})
        for (auto shape : {std::pair<int, int>{5, 20}, {3, 130}, {2100, 130}}) {
            std::vector<unsigned char> a, b;
            if (!run(algorithm, shape.first, shape.second, 0, a) || !run(algorithm, shape.first, shape.second, 1, b)) {
                std::printf("failed\n");
                return 1;
            }
            size_t n = 0;
            for (size_t i = 0; i < a.size(); i++) n += a[i] != b[i];
            if (n) {
                std::printf("%d x %d: %zu bytes differ\n", shape.first, shape.second, n);
                return 1;
            }
        }
    std::printf("same\n");
    return 0;
}
