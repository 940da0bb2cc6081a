// Fixed-step Solves with dense output of a system whose step action ends an
// instance: a system of one's own with time terms, whose wavefronts share their
// time (workgroups of 64), against the same Solve one lane per instance
// (workgroups of 100, which are no whole wavefronts).  Every point of the
// dense-output buffers has to be the same, those past an instance's end, which
// hold what was uploaded, included.  Prints "same" and returns 0, or says what
// differs and returns 1.
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "pt_engine.h"
#include "systems/duffing.h"

namespace mpgos {
void set_error(const std::string& msg) { std::fprintf(stderr, "%s\n", msg.c_str()); }
} // namespace mpgos

// a forced oscillator that ends after cPAR[2] accepted steps
struct CountedSteps : mpgos::systems::DuffingQ {
    static constexpr int NCP = 3, NA = 1;
    static constexpr bool HAS_VJP = false;
    template <class P> __device__ static void Initialization(int, int, int&, P&, P&, P*, P*, P*, P*, int*, P* ACC, int*) { ACC[0] = P(0); }
    template <class P>
    __device__ static void ActionAfterSuccessfulTimeStep(int, int, int& UDT, P&, P&, P*, P*, P* cPAR, P*, int*, P* ACC, int*)
    {
        ACC[0] += P(1);
        if (ACC[0] == cPAR[2]) UDT = 1;
    }
};

static const int NT = 130, NDO = 48, STEPS = 150;
typedef mpgos::pt::Solver<CountedSteps, double, false> Solver;

static bool run(int block, int freq, std::vector<unsigned char>& out)
{
    Solver S;
    if (S.init(MPGOS_RK4, NT, NDO, 0)) return false;
    const double h = 0.0625;
    for (int i = 0; i < NT; i++) {
        S.TD.h[NT + i] = STEPS * h;
        for (int c = 0; c < 3; c++) S.X.h[c * NT + i] = 0.1 * c - 0.003 * i;
        S.cPAR.h[i] = 0.2;
        S.cPAR.h[NT + i] = 0.3 + 0.05 * i;
        // the first wavefront ends in the middle of its blocks of steps, the second at their ends, the third not at all
        S.cPAR.h[2 * NT + i] = i < 64 ? 3 + 2 * i : i < 128 ? 31 * (1 + i % 5) : 1e9;
    }
    for (size_t i = 0; i < S.DOt.n; i++) S.DOt.h[i] = -7.0;
    for (size_t i = 0; i < S.DOx.n; i++) S.DOx.h[i] = -8.0;
    if (S.option(MPGOS_PT_THREADS_PER_BLOCK, 0, block) || S.option(MPGOS_PT_INITIAL_TIME_STEP, 0, h) ||
        S.option(MPGOS_PT_DENSE_OUTPUT_SAVE_FREQUENCY, 0, freq) || S.sync(MPGOS_PT_ALL, true) || S.solve() ||
        S.sync(MPGOS_PT_ALL, false) || S.synchronise_device())
        return false;
    auto add = [&](const auto& b) { out.insert(out.end(), (const unsigned char*)b.h, (const unsigned char*)b.h + b.bytes()); };
    add(S.DOt); add(S.DOx); add(S.X); add(S.T); add(S.ACC); add(S.DOidx); add(S.nacc); add(S.status);
    return true;
}

int main()
{
    for (int freq : {1, 4}) {
        std::vector<unsigned char> shared, single;
        if (!run(64, freq, shared) || !run(100, freq, single)) return 1;
        size_t n = 0;
        for (size_t i = 0; i < shared.size(); i++) n += shared[i] != single[i];
        if (n) {
            std::printf("every %d steps: %zu bytes differ\n", freq, n);
            return 1;
        }
    }
    std::printf("same\n");
    return 0;
}
