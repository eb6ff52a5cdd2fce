"""The library when a HIP call of its own fails on the host's side
(tests/capi/hip_faults.cpp): nothing abandoned may reach a later call."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "capi", "hip_faults")


@pytest.mark.parametrize("what", ["batch", "records"])
def test_failing_calls(what, cuda):
    res = subprocess.run([EXE, what], capture_output=True, text=True, timeout=100)
    print(res.stdout + res.stderr, flush=True)
    assert res.returncode == 0
