"""The dense-contraction form of the per-block solver at the edges of its
layout, bit for bit against the oracle and the lane-per-pair form: unit counts
around the 16-unit tiles (one unit, one tile, padded tiles, one and two tiles
per wavefront), system counts around its 4 and 8 systems per workgroup with
inactive systems at the end, both algorithms; the form with events, user
termination, accessories and dense output at an odd unit count; and the system
counts from which a workgroup holds 8 systems."""
import numpy as np
import pytest

from mpgos import workloads as W
from mpgos.enums import Algorithms
from mpgos.perblock import PB, PBOption, PBProblemSolver
from test_gpu_perblock import assert_pb_bitwise, run_pb_gpu

pytestmark = pytest.mark.gpu


def _ring(ns, ups, alg, end, off):
    s = W.config4_ring(ns=ns, ups=ups, periods=1, algorithm=alg)
    s["TD"][1] = np.linspace(0.5 * end, end, ns)
    s["n_active"] = ns - off
    if alg == Algorithms.RK4:
        s["options"]["dt0"] = 0.01
    return s


@pytest.mark.parametrize("ups,ns,off", [(1, 5, 0), (9, 4, 1), (13, 8, 0), (16, 9, 2), (17, 3, 0), (100, 6, 1), (128, 4, 3),
                                        (129, 7, 5), (250, 5, 0), (256, 2, 0)])
@pytest.mark.parametrize("alg", [Algorithms.RKCK45, Algorithms.RK4], ids=["rkck45", "rk4"])
def test_unit_counts(oracle, ups, ns, off, alg):
    import pyoracle
    s = _ring(ns, ups, alg, 1.0, off)
    print(f"dense form {ns} x {ups} alg={int(alg)}", flush=True)
    ref = pyoracle.run_pb("ring_duffing", s)
    assert len(np.unique(ref["nacc"][:ns - off])) > 1 or ns - off < 3
    assert_pb_bitwise(run_pb_gpu(s), ref, "automatic")
    assert_pb_bitwise(run_pb_gpu(s, kernel=1), ref, "lane per pair")
    assert_pb_bitwise(run_pb_gpu(s, shared_matrix=1, shared_globals=0), ref, "options")


@pytest.mark.parametrize("ns,ups", [(1027, 129), (2053, 113), (16390, 12)])
def test_eight_systems_per_workgroup(oracle, ns, ups):
    import pyoracle
    s = _ring(ns, ups, Algorithms.RKCK45, 0.25, 3)
    print(f"dense form {ns} x {ups}", flush=True)
    ref = pyoracle.run_pb("ring_duffing", s)
    assert_pb_bitwise(run_pb_gpu(s), ref, "automatic")


@pytest.mark.parametrize("ns,ups,ndo", [(5, 14, 64), (3, 150, 7), (1025, 130, 3), (2050, 114, 0)])
def test_events_and_dense_output(oracle, ns, ups, ndo):
    import pyoracle
    base = W.tutorial_ring_dw(ns=25, ups=ups)
    s = W.new_pb_spec("ring_dw", Algorithms.RKCK45, ns, ups, ndo=ndo)
    for k in ("rtol", "atol", "edir", "options", "gPAR", "cIndex"):
        s[k] = base[k]
    for key in ("TD", "T", "sPAR", "sACC", "sACCi", "strength", "DOidx"):
        s[key] = np.ascontiguousarray(np.resize(base[key].T, (ns,) + base[key].T.shape[1:]).T)
    for key in ("X", "uPAR", "uACC", "uACCi"):
        s[key] = np.ascontiguousarray(np.resize(base[key].T, (ns * ups,) + base[key].T.shape[1:]).T)
    ring = np.zeros((ups, ups))
    for r in range(ups):
        ring[r, (r + 1) % ups] = ring[r, (r - 1) % ups] = 1.0
    s["cMat"] = np.concatenate([W.store_coupling(ring, 0, 0)] * 2)
    if ns > 100:
        s["TD"][1] = 2.0
    print(f"ring_dw {ns} x {ups}", flush=True)
    ref = pyoracle.run_pb("ring_dw", s)
    assert_pb_bitwise(run_pb_gpu(s), ref, "automatic")
    if ns < 100:
        assert (ref["uACCi"] == 2).any() and (ref["T"] < s["TD"][1]).any()


@pytest.mark.parametrize("ns,ups,off,K,alg", [(5, 1, 0, 3, Algorithms.RKCK45), (4, 13, 1, 5, Algorithms.RK4),
                                              (9, 100, 2, 64, Algorithms.RKCK45), (6, 131, 0, 7, Algorithms.RK4),
                                              (3, 256, 0, 9, Algorithms.RKCK45), (1027, 129, 3, 4, Algorithms.RKCK45),
                                              (2053, 113, 0, 6, Algorithms.RKCK45)])
def test_adjoint_equals_lane_form(ns, ups, off, K, alg):
    """Reverse pass at the same edges: gradients bit for bit those of the
    lane-per-pair form, a checkpoint interval that does not divide the steps."""
    s = W.config4_ring(ns=ns, ups=ups, periods=1, algorithm=alg, system="ring_duffing_q")
    end = 0.25 if ns > 100 else 1.0
    s["TD"][1] = np.linspace(0.5 * end, end, ns)
    s["n_active"] = ns - off
    if alg == Algorithms.RK4:
        s["options"]["dt0"] = 0.02
    w = W.Stream(W.SEED, 320).normal(3 * ns * ups).reshape(3, -1)
    print(f"adjoint {ns} x {ups} K={K} alg={int(alg)}", flush=True)
    outs = []
    for kernel in (1, 0):
        p = PBProblemSolver("ring_duffing_q", ns, ups, alg)
        try:
            W.load_pb(p, s)
            p.SolverOption(PBOption.CouplingKernel, kernel)
            outs.append([np.array(x) for x in p.adjoint(w, K, 400 // K + 2, 400)])
            p.SynchroniseFromDeviceToHost(PB.Status)
            p.InsertSynchronisationPoint()
            p.SynchroniseSolver()
            assert not (p.host_array(PB.Status) & 16).any()
        finally:
            p.close()
    for a, b in zip(*outs):
        a, b = (x.reshape(x.shape[0], ns, -1)[:, :ns - off] for x in (a, b))
        assert np.isfinite(a).all() and np.abs(a).max() > 0
        assert np.array_equal(a.view(np.uint64), b.view(np.uint64))


@pytest.mark.parametrize("kind", ["subnormal", "huge", "non-finite"])
def test_extreme_values(oracle, kind):
    """Subnormal and huge states, coupling terms and matrix entries, and systems
    with infinities and NaN beside ordinary ones in the same workgroup."""
    import pyoracle
    ns, ups = 9, 20
    rs = W.Stream(W.SEED, 330)
    s = W.new_pb_spec("pb_linear", Algorithms.RKCK45, ns, ups)
    s["cMat"] = rs.normal(ups * ups) * 0.1
    s["uPAR"][0] = rs.uniform(ns * ups, -1.0, 0.3)
    s["X"][0] = rs.uniform(ns * ups, -1.0, 1.0)
    s["strength"][0] = 1.0
    s["TD"][1] = 1.0
    s["rtol"] = s["atol"] = 1e-6
    if kind == "subnormal":
        s["X"][0] *= 1e-310
        s["cMat"][::7] *= 1e-309
    elif kind == "huge":
        s["X"][0] *= 1e150
        s["cMat"][::5] = -0.0
        s["strength"][0, 3] = 1e120
    else:
        s["X"][0, 2 * ups + 3] = np.inf
        s["X"][0, 5 * ups] = np.nan
        s["strength"][0, 7] = np.inf
    print(f"dense form {kind}", flush=True)
    ref = pyoracle.run_pb("pb_linear", s)
    assert_pb_bitwise(run_pb_gpu(s), ref, "automatic")
    assert_pb_bitwise(run_pb_gpu(s, kernel=1), ref, "lane per pair")
