"""NaN tolerances of the adaptive stepper.  No error is below a tolerance that
is NaN on both sides, so every step is rejected and the Solve does not end
(looked at in launches of a bounded number of attempts); with one side NaN the
other one counts, bit for bit as in the oracle."""
import numpy as np
import pytest

import scenarios as S
from helpers import assert_bitwise, run_gpu
from mpgos import ListOfSolverOptions as O, Precision, ProblemSolver
from mpgos import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [Precision.DOUBLE, Precision.FLOAT, Precision.FLOAT_KAHAN])
@pytest.mark.parametrize("components", [(0,), (1,), (0, 1)])
def test_both_sides(gpu, precision, components):
    spec = S.affine(130, a01=1.0, a10=-1.0, x0=(1.0, 0.0), td=(0.0, 1.0))
    s = ProblemSolver("affine2", 130, spec["algorithm"], precision)
    W.load(s, spec)
    for i in range(2):
        tol = np.nan if i in components else 1e3
        s.SolverOption(O.RelativeTolerance, i, tol)
        s.SolverOption(O.AbsoluteTolerance, i, tol)
    for _ in range(3):
        assert s.solve_slice(40) == 130
    s.close()


@pytest.mark.parametrize("side", ["rtol", "atol"])
def test_one_side(gpu, oracle, side):
    spec = S.affine(130, a01=1.0, a10=-1.0, x0=(1.0, 0.5), td=(0.0, 3.0), rtol=1e-9, atol=1e-7)
    spec[side] = np.nan
    assert_bitwise(run_gpu(spec), oracle.run("affine2", spec), label=side)
