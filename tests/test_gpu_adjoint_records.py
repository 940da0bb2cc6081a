"""Segment records of the fixed-step adjoint in HBM (K records of a workgroup
above 64 KiB) with fewer instances than lanes: the wavefront that shares its
time holds lanes without an instance, and the records end with the last one."""
import pytest

from test_gpu_common_time import duffing
from mpgos import Algorithms, ListOfSolverOptions as O, ProblemSolver
from mpgos import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt,block,k", [(1, 64, 26), (1, 64, 31), (2, 64, 31), (1, 512, 4), (2, 512, 5), (1, 512, 31), (63, 512, 4)])
def test_few_instances(gpu, nt, block, k):
    spec = duffing(nt, 161, system="duffing_q", part=0.5)
    lam = W.Stream(stream=19).normal(3 * nt).reshape(3, nt)
    got = []
    for b in (block, 100):     # 100: no whole wavefronts, one lane per instance
        s = ProblemSolver("duffing_q", nt, Algorithms.RK4)
        W.load(s, spec)
        s.SolverOption(O.ThreadsPerBlock, b)
        got.append(s.adjoint(lam, k, 161 // k + 2))
        s.close()
    assert got[0][0].tobytes() == got[1][0].tobytes() and got[0][1].tobytes() == got[1][1].tobytes()
