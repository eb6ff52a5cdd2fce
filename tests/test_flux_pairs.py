"""The two elements of a face see the same bits of Rusanov's flux: with the sides
exchanged and the normal turned it is the exact negative (tests/capi/flux_pairs.hip),
on the host in a build that may contract products into sums, and on the device."""
import os
import subprocess

import pytest

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "capi", "flux_pairs")


def _run(*args):
    res = subprocess.run([EXE, *args], capture_output=True, text=True, timeout=100)
    print(res.stdout + res.stderr, flush=True)
    if res.returncode == 77:
        pytest.skip("no fused multiply-add on this processor")
    rows = [line.split() for line in res.stdout.splitlines()]
    assert len(rows) == 8 and all(int(r[3]) == 1 << 16 and int(r[4]) == 0 for r in rows)
    assert res.returncode == 0


def test_host():
    _run()


@pytest.mark.gpu
def test_device(cuda):
    _run("--gpu")
