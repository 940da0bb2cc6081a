"""Of several buffers that a call allocates, any one may fail: the call says so,
and the next one allocates what is missing before it launches anything."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "allocation_fails")


def test_every_allocation_of_a_solve(gpu):
    assert os.path.exists(EXE), "build() compiles tests/cpp/allocation_fails"
    r = subprocess.run([EXE], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "same", (r.returncode, r.stdout, r.stderr)
