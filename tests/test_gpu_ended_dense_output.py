"""Dense output of fixed-step Solves whose instances end before their time:
the buffers behind an instance's last point keep what was uploaded, whether a
wavefront shares its time (whole wavefronts) or not (workgroups of 100)."""
import os
import subprocess

import numpy as np
import pytest

from test_gpu_common_time import duffing
from mpgos import ListOfSolverOptions as O, ListOfVariables as V, ProblemSolver
from mpgos import workloads as W

pytestmark = pytest.mark.gpu

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "step_end")


@pytest.mark.parametrize("ndo,freq", [(40, 1), (40, 4), (300, 1)])
def test_non_finite(gpu, ndo, freq):
    spec = duffing(128, 200, ndo=ndo)
    spec["options"]["do_freq"] = freq
    spec["X"][0, 5] = 1e60
    spec["X"][0, 40] = 40.0
    spec["X"][1, 70] = 3e3
    got = []
    for block in (64, 100):
        s = ProblemSolver("duffing", 128, spec["algorithm"], ndo=ndo)
        W.load(s, spec)
        s.SolverOption(O.ThreadsPerBlock, block)
        for v in (V.DenseTime, V.DenseState):
            s.host_array(v)[...] = -7.0
        s.SynchroniseFromHostToDevice(V.All)
        s.solve_blocking()
        got.append({v: s.host_array(v).copy() for v in (V.DenseTime, V.DenseState, V.DenseIndex, V.AcceptedSteps, V.ActualState)})
        s.close()
    assert (got[0][V.AcceptedSteps] < 200).any()
    for v in got[0]:
        assert got[0][v].tobytes() == got[1][v].tobytes(), v


def test_step_action(gpu):
    assert os.path.exists(EXE), "build() compiles tests/cpp/step_end"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "same", (r.returncode, r.stdout, r.stderr)
