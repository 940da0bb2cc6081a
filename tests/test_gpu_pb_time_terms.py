"""A per-block system of one's own with time terms that depend on a parameter
(tests/cpp/pb_time_terms.cu)."""
import os
import subprocess

import pytest

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "pb_time_terms")


@pytest.mark.gpu
def test_gradient_without_a_time_term_vjp(gpu):
    assert os.path.exists(EXE), "build() compiles tests/cpp/pb_time_terms"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "same", (r.returncode, r.stdout, r.stderr)


def test_reverse_pass_that_exceeds_the_lds_runs_one_lane_per_unit():
    assert os.path.exists(EXE), "build() compiles tests/cpp/pb_time_terms"
    r = subprocess.run([EXE, "forms"], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "forms", (r.returncode, r.stdout, r.stderr)
