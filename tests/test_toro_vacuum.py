"""Toro's two-rarefaction speeds where the estimate has no positive base
(tests/capi/toro_base.hip): the acoustic speeds bit by bit, host and device."""
import os
import subprocess

import pytest

EXE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "capi", "toro_base")


def _run(*args):
    res = subprocess.run([EXE, *args], capture_output=True, text=True, timeout=100)
    print(res.stdout + res.stderr, flush=True)
    rows = [line.split() for line in res.stdout.splitlines()]
    assert len(rows) == 10 and all(int(r[2]) == 1 << 14 and int(r[3]) == 0 for r in rows)
    assert res.returncode == 0


def test_host():
    _run()


@pytest.mark.gpu
def test_device(cuda):
    _run("--gpu")
