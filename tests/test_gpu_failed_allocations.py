"""A device allocation that fails is reported by the call that made it, or
answered by a smaller one, and leaves nothing behind for later calls."""
import pytest

import torch
from mpgos import Algorithms, MPGOSError, ProblemSolver
from mpgos import workloads as W
from mpgos.perblock import PBOption, PBProblemSolver

pytestmark = pytest.mark.gpu


def test_solve_after_a_failed_record(gpu):
    spec = W.config3_duffing_adjoint(nt=64, algorithm=Algorithms.RK4)
    spec["TD"][1] = 1.0
    s = ProblemSolver(spec["system"], 64, spec["algorithm"])
    W.load(s, spec)
    with pytest.raises(MPGOSError, match="allocation failed"):
        s.adjoint_record(16, 2**31 - 1)         # 8 TB of checkpoints
    s.solve_blocking()
    s.close()


def test_reverse_pass_that_fits_one_lane_per_unit_only(gpu):
    """8 systems of 100 units per workgroup: the stage buffer of the
    matrix-core form has 24 rows per step, the segment buffer of the other 3."""
    ns, ups = 1100, 100
    total = torch.cuda.get_device_properties(0).total_memory
    k = int(1.05 * total) // (24 * ns * ups * 8)
    spec = W.config4_ring(ns=ns, ups=ups, periods=1, algorithm=Algorithms.RKCK45, system="ring_duffing_q")
    spec["TD"][1] = 0.5
    w = W.Stream(stream=21).normal(3 * ns * ups).reshape(3, ns * ups)
    got = []
    for interval, kernel in ((k, 0), (16, 1)):
        s = PBProblemSolver(spec["system"], ns, ups, spec["algorithm"], spb=spec.get("spb", 1), cbw=0, cci=0)
        W.load_pb(s, spec)
        s.SolverOption(PBOption.CouplingKernel, kernel)
        got.append(s.adjoint(w, interval, 300 // interval + 2, 300))
        s.close()
    for a, b in zip(*got):
        assert a.tobytes() == b.tobytes()
