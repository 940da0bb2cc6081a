"""Lane-per-pair form, full matrices: the kernels that sum the columns in groups
against those that sum one after the other (with the matrix in LDS, which the
grouped kernels do not take), bit for bit, at the remainders of the groups and
on both sides of every line of the choice; FP64 against the oracle as well."""
import numpy as np
import pytest

from mpgos import Algorithms, Precision
from mpgos import workloads as W
from mpgos.perblock import PBOption, PBProblemSolver

pytestmark = pytest.mark.gpu

KEYS = ("X", "T", "uACC", "uACCi", "sACC", "sACCi", "nacc", "nrej", "status")


def ring(system, algorithm, ns, ups):
    s = W.new_pb_spec(system, algorithm, ns, ups)
    rs = W.Stream(stream=23)
    s["cMat"][:] = rs.normal(s["cMat"].size, 0.3 / np.sqrt(ups))
    s["strength"][:] = 0.5
    s["TD"][1] = 1.0
    s["X"][:2] = rs.uniform(2 * ns * ups, -1.0, 1.0).reshape(2, ns * ups)
    if system == "ring_dw":
        s["cIndex"][:] = (0, 1)
        s["uPAR"][:] = np.array([0.5, 0.24, 1.3])[:, None]
        s["gPAR"][0] = 0.004
        s["edir"] = -1
    else:
        s["cIndex"][0] = 1
        s["uPAR"][0] = 0.2
        s["sPAR"][0] = rs.uniform(ns, 0.5, 5.0)
    if algorithm == Algorithms.RK4:
        s["options"]["dt0"] = 0.05
    return s


def run(spec, precision, shared):
    s = PBProblemSolver(spec["system"], spec["ns"], spec["ups"], spec["algorithm"], precision, spb=spec["spb"], cbw=0, cci=0, ndo=0)
    W.load_pb(s, spec)
    s.SolverOption(PBOption.CouplingKernel, 1)
    s.SolverOption(PBOption.SharedCouplingMatrices, shared)
    s.solve_blocking()
    out = W.read_pb(s)
    s.close()
    return out


@pytest.mark.parametrize("precision", [Precision.DOUBLE, Precision.FLOAT, Precision.FLOAT_KAHAN])
@pytest.mark.parametrize("algorithm", [Algorithms.RK4, Algorithms.RKCK45])
@pytest.mark.parametrize("system", ["ring_duffing", "ring_dw"])
def test_sizes(gpu, oracle, system, algorithm, precision):
    for ups in (1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 23, 24, 25, 26, 31, 64, 65, 66, 67, 70):
        spec = ring(system, algorithm, 3, ups)
        spec["spb"] = max(1, 64 // ups)
        a, b = run(spec, precision, 0), run(spec, precision, 1)
        assert a["nacc"].min() > 3
        ref = oracle.run_pb(system, spec) if precision == Precision.DOUBLE else b
        for k in KEYS:
            assert a[k].tobytes() == b[k].tobytes(), (ups, k)
            assert a[k].tobytes() == np.asarray(ref[k]).astype(a[k].dtype).tobytes(), (ups, k)


def test_more_wavefronts_than_the_card_holds(gpu):
    spec = ring("ring_dw", Algorithms.RKCK45, 3500, 10)
    spec["spb"] = 1
    a, b = run(spec, Precision.FLOAT, 0), run(spec, Precision.FLOAT, 1)
    for k in KEYS:
        assert a[k].tobytes() == b[k].tobytes(), k
