"""Fixed-step RK4 of systems with time terms: wavefronts whose instances share
their time evaluate the terms of many steps at once.  Results are held bit for
bit to the oracle (FP64) and to the per-lane path (workgroups that are no whole
wavefronts), at the edges of the blocks of 31 (compensated form: 21) steps."""
import numpy as np
import pytest

from helpers import assert_bitwise, run_gpu
from mpgos import Algorithms, ListOfSolverOptions as O, Precision, ProblemSolver
from mpgos import workloads as W

pytestmark = pytest.mark.gpu


def duffing(nt, steps, system="duffing", ndo=0, part=0.0):
    s = W.new_spec(system, Algorithms.RK4, nt, ndo=ndo)
    s["options"]["dt0"] = 2.0 * W.PI / 100.0
    s["TD"][1] = (steps + part) * s["options"]["dt0"]
    rs = W.Stream(stream=17)
    s["X"][:2] = rs.uniform(2 * nt, -1.0, 1.0).reshape(2, nt)
    if system == "duffing_dw":
        s["cPAR"][0] = 0.25
        s["sPAR"][0] = 0.3
    else:
        s["cPAR"][0] = 0.2
        s["cPAR"][1] = W.linspace(0.3, 10.0, nt)
    return s


@pytest.mark.parametrize("steps,part", [(0, 0.5), (1, 0.0), (20, 0.3), (21, 0.0), (22, 0.1), (30, 0.5), (31, 0.0), (31, 0.5), (32, 0.0),
                                        (62, 0.9), (63, 0.0), (64, 0.1), (1000, 0.5)])
def test_block_edges(gpu, oracle, steps, part):
    spec = duffing(130, steps, part=part)
    ref = oracle.run("duffing", spec)
    for block in (64, 128, 100):
        assert_bitwise(run_gpu(spec, block=block), ref, label=f"steps {steps} block {block}")


@pytest.mark.parametrize("nt,active", [(1, 1), (63, 63), (65, 65), (200, 130), (200, 1)])
def test_ragged(gpu, oracle, nt, active):
    spec = duffing(nt, 150, part=0.25)
    spec["n_active"] = active
    assert_bitwise(run_gpu(spec, block=128), oracle.run("duffing", spec), label=f"{active} of {nt}")


def test_different_times(gpu, oracle):
    # one wavefront of a common time, one with two ends, one with two starts
    spec = duffing(192, 100)
    spec["TD"][1, 64:96] *= 0.5
    spec["TD"][0, 130] = 0.1
    assert_bitwise(run_gpu(spec), oracle.run("duffing", spec), label="different times")


def test_instances_that_end_early(gpu, oracle):
    # overflow at different steps in some lanes of a wavefront
    spec = duffing(128, 200)
    spec["X"][0, 5] = 1e60
    spec["X"][0, 40] = 40.0
    spec["X"][1, 70] = 3e3
    ref = oracle.run("duffing", spec)
    assert (ref["status"] != 0).any() and (ref["nacc"] < 200).any()
    assert_bitwise(run_gpu(spec), ref, label="non-finite")


@pytest.mark.parametrize("ndo,freq", [(10, 1), (40, 3), (300, 1)])
def test_dense_output(gpu, oracle, ndo, freq):
    spec = duffing(100, 170, ndo=ndo, part=0.5)
    spec["options"]["do_freq"] = freq
    assert_bitwise(run_gpu(spec), oracle.run("duffing", spec), keys=("X", "T", "ACC", "nacc", "DOidx", "DOt", "DOx"),
                   label=f"dense {ndo} {freq}")


@pytest.mark.parametrize("precision", [Precision.FLOAT, Precision.FLOAT_KAHAN])
@pytest.mark.parametrize("steps", [20, 21, 22, 63, 500])
def test_single_precision_equals_the_per_lane_path(gpu, precision, steps):
    spec = duffing(150, steps, part=0.5)
    assert_bitwise(run_gpu(spec, precision=precision, block=64), run_gpu(spec, precision=precision, block=100),
                   keys=("nacc", "status"), label=f"{precision} counts")
    a, b = run_gpu(spec, precision=precision, block=64), run_gpu(spec, precision=precision, block=100)
    for k in ("X", "T", "ACC"):
        assert a[k].tobytes() == b[k].tobytes(), k


@pytest.mark.parametrize("k", [1, 2, 7, 16, 30, 31, 32, 40])
@pytest.mark.parametrize("steps,part", [(5, 0.0), (64, 0.0), (161, 0.5)])
def test_adjoint_equals_the_per_lane_path(gpu, k, steps, part):
    nt = 130
    spec = duffing(nt, steps, system="duffing_q", part=part)
    spec["TD"][1, 128:] = 1.5
    lam = W.Stream(stream=18).normal(3 * nt).reshape(3, nt)
    got = []
    for block in (64, 100):
        s = ProblemSolver("duffing_q", nt, Algorithms.RK4)
        W.load(s, spec)
        s.SolverOption(O.ThreadsPerBlock, block)
        got.append(s.adjoint(lam, k, max(steps, 24) // k + 2))   # 24 steps end at 1.5
        s.close()
    assert np.isfinite(got[0][0]).all()
    assert got[0][0].tobytes() == got[1][0].tobytes() and got[0][1].tobytes() == got[1][1].tobytes()
