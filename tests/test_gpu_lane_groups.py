"""Several lanes per instance (adaptive steps of systems with time terms, few
instances): at the instance counts where 8, 4 and 1 lanes meet, in every
precision, with events, dense output and user termination, in the sorted form
with long and short instances side by side, and in the adjoint, bit for bit
against the oracle or against one lane per instance."""
import numpy as np
import pytest

from helpers import assert_bitwise, run_gpu
from mpgos import Algorithms, ListOfSolverOptions as O, Precision, ProblemSolver
from mpgos import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("X", "T", "ACC", "ACCi", "nacc", "nrej", "status", "nev", "evlog", "evlogidx", "DOidx", "DOt", "DOx")


def _eps(nt, cap):
    s = W.config2_duffing_uneven(nt=nt, evcap=4)
    s["TD"][1] = cap * np.random.RandomState(nt).uniform(0.05, 1.0, nt)
    return s


@pytest.mark.parametrize("nt,block", [(1, 64), (7, 64), (9, 128), (100, 100), (8192, 256), (8193, 64), (16384, 64), (16385, 64)])
def test_plain(gpu, oracle, nt, block):
    s = _eps(nt, 12.0)
    assert_bitwise(run_gpu(s, block=block), oracle.run("duffing_eps", s), keys=KEYS, label=f"{nt} instances")


@pytest.mark.parametrize("precision", [Precision.DOUBLE, Precision.FLOAT, Precision.FLOAT_KAHAN])
@pytest.mark.parametrize("nt", [130, 9000])
def test_precisions_and_dense_output(gpu, nt, precision):
    s = W.new_spec("duffing_dw", Algorithms.RKCK45, nt, ndo=20)
    r = np.random.RandomState(5)
    s["TD"][1] = r.uniform(1.0, 9.0, nt)
    s["X"][0] = -0.5 + 0.1 * r.uniform(-1, 1, nt)
    s["cPAR"][0] = W.linspace(0.2, 0.3, nt)
    s["sPAR"][0] = 0.3
    s["rtol"] = s["atol"] = 1e-9 if precision == Precision.DOUBLE else 1e-5
    s["edir"] = np.array([-1, 0])
    several, one = ({k: v.astype(np.float64) if v.dtype == np.float32 else v for k, v in run_gpu(s, precision, variant=n).items()}
                    for n in (0, 1))
    assert_bitwise(several, one, keys=KEYS, label=f"{nt} {precision}")


@pytest.mark.parametrize("nt,block,cap", [(50, 64, 40.0), (6200, 128, 40.0), (20000, 64, 40.0), (70001, 256, 8.0)])
def test_sorted(gpu, oracle, nt, block, cap):
    s = _eps(nt, cap)
    s["n_active"] = nt - nt // 50
    out = run_gpu(s, kernel_mode=3, block=block, relaunch_steps=20)
    assert_bitwise(out, oracle.run("duffing_eps", s), keys=KEYS, label=f"sorted {nt}")


@pytest.mark.parametrize("nt,K", [(5, 3), (600, 200), (8200, 16), (16390, 16)])
def test_adjoint(gpu, nt, K):
    s = W.config3_duffing_adjoint(nt=nt, algorithm=Algorithms.RKCK45, periods=2)
    s["TD"][1] = np.random.RandomState(nt).uniform(1.0, 6.0, nt)
    lam = np.random.RandomState(3).standard_normal((3, nt))
    outs = []
    for variant in (1, 0):
        p = ProblemSolver("duffing_q", nt, Algorithms.RKCK45)
        try:
            W.load(p, s)
            p.SolverOption(O.LaunchVariant, variant)
            outs.append(p.adjoint(lam, K, 600 // K + 2))
        finally:
            p.close()
    for a, b in zip(*outs):
        assert np.isfinite(a).all() and np.abs(a).max() > 0
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))
