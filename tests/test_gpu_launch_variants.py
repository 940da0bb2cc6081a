"""Launch variants 2 and 3 (128 and 64 registers): their kernels are built apart
from those of variants 0 and 1 and treat the step's limits, the polynomials'
coefficients and, for compensated steps, the usual step in another manner.  In
every form, algorithm and precision their results are those of variant 1 bit for
bit, and in double precision the oracle's."""
import numpy as np
import pytest

from helpers import assert_bitwise, run_gpu
from mpgos import Algorithms, Precision
from mpgos import workloads as W

pytestmark = pytest.mark.gpu

KEYS = ("X", "T", "TD", "ACC", "ACCi", "nacc", "nrej", "status", "nev", "evlog", "evlogidx", "DOidx", "DOt", "DOx")
FORMS = {"plain": {}, "persistent": dict(kernel_mode=1), "sorted": dict(kernel_mode=3, relaunch_steps=5),
         "plain sliced": dict(slice_steps=7), "persistent sliced": dict(kernel_mode=1, slice_steps=7)}


def _spec(system, algorithm, precision, nt=333):
    # events of both directions, dense output, rejected steps; one instance each
    # with a state that is not finite, the smallest step and an empty interval
    r = np.random.RandomState(11)
    s = W.new_spec(system, algorithm, nt, ndo=12)
    s["TD"][1] = r.uniform(0.5, 4.0, nt)
    s["X"][0] = -0.5 + 0.1 * r.uniform(-1, 1, nt)
    if system == "lorenz":
        s["X"][:] = r.uniform(1.0, 5.0, s["X"].shape)
        s["cPAR"][0] = r.uniform(10.0, 28.0, nt)
    elif system == "duffing_dw":
        s["cPAR"][0] = W.linspace(0.2, 0.3, nt)
        s["sPAR"][0] = 0.3
        s["edir"] = np.array([-1, 0])
    s["X"][0][5] = np.nan
    s["X"][0][70] = 1e30
    s["TD"][1][130] = s["TD"][0][130]
    s["rtol"] = s["atol"] = 1e-9 if precision == Precision.DOUBLE else 1e-5
    s["dt0"] = 0.02
    return s


def _doubles(out):
    return {k: v.astype(np.float64) if isinstance(v, np.ndarray) and v.dtype == np.float32 else v for k, v in out.items()}


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("precision", [Precision.DOUBLE, Precision.FLOAT, Precision.FLOAT_KAHAN])
@pytest.mark.parametrize("algorithm", [Algorithms.RK4, Algorithms.RKCK45])
@pytest.mark.parametrize("system", ["lorenz", "duffing_dw"])
def test_few_registers(gpu, oracle, system, algorithm, precision, form):
    # variant 0: persistent RK4 kernels are built with those of few registers too
    s = _spec(system, algorithm, precision)
    ref = _doubles(run_gpu(s, precision, variant=1, **FORMS[form]))
    assert ref["nacc"].max() > 3 and (algorithm == Algorithms.RK4 or ref["nrej"].max() > 0)
    if precision == Precision.DOUBLE:
        assert_bitwise(ref, oracle.run(system, s), keys=KEYS, label="variant 1")
    for variant in (0, 2, 3):
        assert_bitwise(_doubles(run_gpu(s, precision, variant=variant, **FORMS[form])), ref, keys=KEYS, label=f"variant {variant}")
