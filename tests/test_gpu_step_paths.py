"""The adaptive step takes a short way while every lane of a wavefront has an
ordinary accepted step and a general one otherwise.  Wavefronts that mix
ordinary instances with each kind of unusual one, and options at which the
short way must not be taken, bit for bit against the oracle."""
import numpy as np
import pytest

import scenarios as S
from helpers import assert_bitwise, run_gpu
from mpgos import Algorithms
from mpgos import workloads as W

pytestmark = pytest.mark.gpu


def mixed(kind):
    """256 damped oscillators with an event function, some lanes of each wavefront unusual."""
    s = S.affine(256, a01=1.0, a10=-1.0, a11=-0.1, x0=(1.0, 0.0), td=(0.0, 6.0), rtol=1e-8, atol=1e-8, c=0.25, evcap=8)
    lanes = np.arange(256) % 64
    if kind == "non-finite":
        s["X"][0, lanes == 9] = np.inf
        s["X"][1, lanes == 10] = np.nan
        s["X"][0, lanes == 11] = 1e308
        s["cPAR"][0, lanes == 11] = 50.0
    elif kind == "stiff":
        s["cPAR"][0, lanes == 3] = -4000.0
    elif kind == "zero, backward and empty intervals":
        s["TD"][1, lanes == 5] = 0.0
        s["TD"][1, lanes == 6] = -1.0
        s["TD"][1, lanes == 7] = 1e-13
    elif kind == "no error":
        s["cPAR"][:4, lanes == 8] = 0.0
        s["X"][0, lanes == 8] = 0.25
    elif kind == "smallest step":
        s["options"]["dtmin"] = 0.02
        s["cPAR"][0, lanes == 20] = -90.0
    elif kind == "event at the start":
        s["X"][0, lanes == 30] = 0.25
        s["X"][0, lanes == 31] = 0.25 + 5e-7
    return s


@pytest.mark.parametrize("form", [0, 1, 2, 3])
@pytest.mark.parametrize("kind", ["ordinary", "non-finite", "stiff", "zero, backward and empty intervals", "no error", "smallest step",
                                  "event at the start"])
def test_mixed_wavefronts(gpu, oracle, kind, form):
    spec = mixed(kind)
    out = run_gpu(spec, kernel_mode=form, relaunch_steps=7, relaunch_launches=3)
    assert_bitwise(out, oracle.run("affine2", spec),
                   keys=("X", "T", "ACCi", "nacc", "nrej", "status", "nev", "evlog", "evlogidx"), label=f"{kind} form {form}")


@pytest.mark.parametrize("options", [{"etol": -1e-3, "c": 1e30}, {"etol": 0.0}, {"etol": np.nan}, {"shrink": 0.0}, {"shrink": 1e-80, "dt0": 500.0},
                                     {"grow": 1.0}, {"dtmax": 1e-2}, {"dtmin": 0.0}, {"rtol": 0.0, "atol": 0.0, "dtmin": 5e-2},
                                     {"rtol": 1e300, "atol": 1e300}, {"atol": 1e-300, "rtol": 1e-12, "dtmin": 1e-4}])
def test_options(gpu, oracle, options):
    spec = S.affine(130, a01=1.0, a10=-1.0, x0=(1.0, 0.0), td=(0.0, 3.0), c=options.get("c", 0.25), evcap=8)
    for k, v in options.items():
        if k in ("rtol", "atol", "etol"):
            spec[k] = v
        elif k != "c":
            spec["options"][k] = v
    assert_bitwise(run_gpu(spec), oracle.run("affine2", spec),
                   keys=("X", "T", "ACCi", "nacc", "nrej", "status", "nev", "evlog"), label=str(options))
