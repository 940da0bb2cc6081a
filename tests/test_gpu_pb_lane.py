"""The lane-per-pair form's sum over a full matrix, bit for bit against the
oracle: unit counts at the remainders of its groups of eight and four columns,
one unit, and above the dense-contraction form's largest, from L2 and from LDS."""
import pytest

from mpgos import workloads as W
from mpgos.enums import Algorithms
from test_gpu_perblock import assert_pb_bitwise, run_pb_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("ups", [1, 2, 3, 4, 5, 7, 8, 9, 11, 12, 15, 16, 23, 257, 300])
def test_column_remainders(oracle, ups):
    import pyoracle
    s = W.config4_ring(ns=5, ups=ups, periods=1, algorithm=Algorithms.RKCK45)
    s["TD"][1] = 0.5
    print(f"lane form 5 x {ups}", flush=True)
    ref = pyoracle.run_pb("ring_duffing", s)
    for spb, shm in ((1, 0), (2 if ups > 64 else 3, 1)):
        assert_pb_bitwise(run_pb_gpu(s, spb=spb, shared_matrix=shm, kernel=1), ref, f"spb={spb} shared_matrix={shm}")
