// Solves whose k-th device allocation fails, for every k: the call that made it
// says so and launches nothing, and the next call allocates what is missing and
// gives the results of an undisturbed Solve (an earlier state of the code took
// the first buffer of a group for all of them).  Sliced, relaunched and sorted
// forms and the queue order.  Prints "same" and returns 0, or says what differs
// and returns 1.
#include <cstdio>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

static int g_left = 0;      // allocations until one fails; 0: none does
static hipError_t counted_malloc(void** p, size_t n)
{
    if (g_left > 0 && --g_left == 0) return hipErrorOutOfMemory;
    return hipMalloc(p, n);
}
#define hipMalloc(p, n) counted_malloc((void**)(p), n)
#include "pt_engine.h"
#undef hipMalloc
#include "systems/lorenz.h"

namespace mpgos {
void set_error(const std::string& msg) { std::fprintf(stderr, "%s\n", msg.c_str()); }
} // namespace mpgos

static const int NT = 200, SLICED = 9;
typedef mpgos::pt::Solver<mpgos::systems::Lorenz, double, false> Solver;

static int solve(Solver& S, int mode)
{
    if (mode != SLICED) return S.solve();
    int left = 1;
    while (left > 0)
        if (int rc = S.solve_slice(40, &left)) return rc;
    return MPGOS_OK;
}

// fails: the allocation of the Solve that fails; `met` whether there was one
static bool run(int mode, int fails, bool& met, std::vector<unsigned char>& out)
{
    Solver S;
    if (S.init(MPGOS_RKCK45, NT, 0, 0)) return false;
    for (int i = 0; i < NT; i++) {
        S.TD.h[NT + i] = 0.1 + 0.004 * i;
        for (int c = 0; c < 3; c++) S.X.h[c * NT + i] = 1.0 + 0.1 * c + 0.01 * i;
        S.cPAR.h[i] = 10.0 + 0.05 * i;
    }
    if (S.option(MPGOS_PT_RELAUNCH_STEPS, 0, 30) || S.option(MPGOS_PT_RELATIVE_TOLERANCE, 0, 1e-9) || S.sync(MPGOS_PT_ALL, true))
        return false;
    if (mode != SLICED && S.option(MPGOS_PT_KERNEL_MODE, 0, mode)) return false;
    if (mode == MPGOS_KERNEL_PERSISTENT && S.option(MPGOS_PT_QUEUE_ORDER, 0, MPGOS_QUEUE_LONGEST_FIRST)) return false;
    g_left = fails;
    const int rc = solve(S, mode);
    met = fails > 0 && g_left == 0;
    g_left = 0;
    if (rc != (met ? MPGOS_E_MEMORY : MPGOS_OK)) return false;
    if (met && solve(S, mode)) return false;
    if (S.sync(MPGOS_PT_ALL, false) || S.synchronise_device()) return false;
    out.clear();
    auto add = [&](const auto& b) { out.insert(out.end(), (const unsigned char*)b.h, (const unsigned char*)b.h + b.bytes()); };
    add(S.X); add(S.T); add(S.nacc); add(S.nrej); add(S.status);
    return true;
}

int main()
{
    std::vector<unsigned char> ref, got;
    bool met;
    if (!run(MPGOS_KERNEL_PLAIN, 0, met, ref)) { std::printf("reference Solve failed\n"); return 1; }
    const struct { int mode, least; } forms[] = {{SLICED, 4}, {MPGOS_KERNEL_RELAUNCH, 5}, {MPGOS_KERNEL_SORTED, 7}, {MPGOS_KERNEL_PERSISTENT, 1}};
    for (const auto& f : forms) {
        int k = 0;
        do {
            k++;
            std::fprintf(stderr, "form %d, allocation %d fails\n", f.mode, k);
            if (!run(f.mode, k, met, got)) { std::printf("form %d: allocation %d: wrong return\n", f.mode, k); return 1; }
            if (got != ref) { std::printf("form %d: allocation %d: results differ\n", f.mode, k); return 1; }
        } while (met && k < 20);
        if (k <= f.least) { std::printf("form %d: only %d allocations\n", f.mode, k - 1); return 1; }
    }
    std::printf("same\n");
    return 0;
}
