"""A record pass that fails: the reverse pass refuses when the earlier record
went with its buffers, and runs on the earlier record when that is untouched."""
import numpy as np
import pytest

from mpgos import Algorithms, MPGOSError, PB, ProblemSolver
from mpgos import ListOfVariables as V
from mpgos import workloads as W
from mpgos.perblock import PBOption, PBProblemSolver

pytestmark = pytest.mark.gpu


NS = 64
MOST = 2**31 - 1        # checkpoints of terabytes; 1.1 TB of step times for 64 systems


def _per_block(ups):
    spec = W.config4_ring(ns=NS, ups=ups, periods=1, algorithm=Algorithms.RKCK45, system="ring_duffing_q")
    spec["TD"][1] = 0.5
    s = PBProblemSolver(spec["system"], NS, ups, spec["algorithm"], spb=spec.get("spb", 1), cbw=0, cci=0)
    W.load_pb(s, spec)
    return s, spec, np.random.RandomState(ups).standard_normal((3, NS * ups))


def _reverse(s, var, lam):
    s.host_array(var)[...] = lam
    s.SynchroniseFromHostToDevice(var)
    s.adjoint_reverse()
    s.SynchroniseFromDeviceToHost(var)
    s.InsertSynchronisationPoint()
    s.SynchroniseSolver()
    return s.host_array(var).tobytes()


@pytest.mark.parametrize("ups", [32, 50])
@pytest.mark.parametrize("capacities", [(MOST, 300), (400, MOST)], ids=["checkpoints", "steps"])
def test_per_block_allocation(gpu, ups, capacities):
    s, spec, lam = _per_block(ups)
    s.adjoint_record(8, 300, 300)
    gradient = _reverse(s, PB.AdjointState, lam)
    with pytest.raises(MPGOSError, match="allocation"):
        s.adjoint_record(1, *capacities)
    with pytest.raises(MPGOSError, match="no record pass"):
        s.adjoint_reverse()
    W.load_pb(s, spec)
    s.adjoint_record(8, 300, 300)
    assert _reverse(s, PB.AdjointState, lam) == gradient
    s.close()


def test_per_block_refusal(gpu):
    s, _, lam = _per_block(50)
    s.adjoint_record(8, 300, 300)
    gradient = _reverse(s, PB.AdjointState, lam)
    s.SolverOption(PBOption.CouplingKernel, 2)      # not for 50 units
    with pytest.raises(MPGOSError):
        s.adjoint_record(1, 300, 300)
    s.SolverOption(PBOption.CouplingKernel, 0)
    assert _reverse(s, PB.AdjointState, lam) == gradient
    s.close()


@pytest.mark.parametrize("algorithm", [Algorithms.RK4, Algorithms.RKCK45])
def test_per_thread(gpu, algorithm):
    spec = W.config3_duffing_adjoint(nt=512, algorithm=algorithm, periods=1)
    lam = np.random.RandomState(1).standard_normal((3, 512))
    s = ProblemSolver(spec["system"], 512, spec["algorithm"])
    W.load(s, spec)
    s.adjoint_record(16, 100)
    gradient = _reverse(s, V.AdjointState, lam)
    with pytest.raises(MPGOSError, match="segment"):
        s.adjoint_record(MOST, 100)                 # the checkpoints stay as they are
    assert _reverse(s, V.AdjointState, lam) == gradient
    with pytest.raises(MPGOSError, match="checkpoint"):
        s.adjoint_record(16, MOST)
    with pytest.raises(MPGOSError, match="no recorded forward pass"):
        s.adjoint_reverse()
    W.load(s, spec)
    s.adjoint_record(16, 100)
    assert _reverse(s, V.AdjointState, lam) == gradient
    s.close()
