"""Toro's two-rarefaction speeds in the solvers that use them, for gammas whose
1/z = 2 gamma / (gamma - 1) is an integer (1.4: 7, 5/3: 5, 1.2: 12, 2: 4) and for
others: the host build of the device code and the GPU kernels against the
oracle, which forms the estimate as written (physics.cpp:309-350). Bars: 1e-12
of the wave speed (each power carries a few ulp, raised to 1/z <= 24); on the
GPU the suite's parity bar, 1e-12 relative L-infinity per variable."""
import ctypes as C

import numpy as np
import pytest

from oracle import refcpu as R
from oracle.refcpu import RefSolver
from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, conservative, rel_linf, smooth_state

GAMMAS = [1.4, 5.0 / 3.0, 1.2, 2.0, 1.3, 1.09]


@pytest.mark.parametrize("gamma", GAMMAS)
def test_vacuum_speeds(gamma):
    """States that separate faster than their rarefactions: the base of the power
    1/z is negative. Where 1/z is an integer in double the reference's power is a
    number (positive for gamma = 2, 1/z = 4), elsewhere it is none and its
    comparisons take the acoustic speeds."""
    from rkdg_amd import capi

    sch = S.Scheme(riemann=S.HLL, gamma=gamma)
    sd = capi.scheme_desc(sch)
    pd = C.POINTER(C.c_double)
    n = np.array([1.0, 0.0])
    for speed in (8.0, 20.0):
        a = np.array(conservative(1.0, [-speed, 0.0], 0.4, gamma))
        b = np.array(conservative(1.1, [speed, 0.0], 0.5, gamma))
        f_ref, lam_ref = R.riemann_eval(sch, 2, a, b, n)
        f, lam = np.zeros(4), C.c_double()
        assert capi.lib().rkdg_riemann_eval(C.byref(sd), 2, *(v.ctypes.data_as(pd) for v in (a, b, n, f)),
                                            C.byref(lam)) == 0
        assert abs(lam.value - lam_ref) <= 1e-12 * lam_ref


@pytest.mark.gpu
@pytest.mark.parametrize("gamma", GAMMAS)
@pytest.mark.parametrize("riemann", [S.LLF, S.HLL, S.HLLC])
def test_gpu_rhs_matches_oracle(gamma, riemann, cuda):
    import torch

    from rkdg_amd.capi import Context

    for m, p, dense in ((M.structured_hex(3, 4, 3), 1, False), (M.structured_hex(3, 3, 3), 2, False),
                        (M.structured_quad(6, 5, periodic=(True, True)), 2, False),
                        (M.jittered_delaunay_tri(5, 4), 2, True)):
        sch = S.Scheme(riemann=riemann, gamma=gamma, bcs=all_outlet(m))
        ref = RefSolver(m, p, sch)
        x = smooth_state(ref.node_coords(), seed=3, amp=2e-2, gamma=gamma)
        y_ref, lam_ref = ref.mult(x)
        ctx = Context(m, p, sch)
        xd = torch.from_numpy(x).to(cuda)
        yd = torch.empty_like(xd)
        lam = ctx.rhs(xd, yd)
        assert rel_linf(yd.cpu().numpy(), y_ref, m.dim + 2) <= 1e-12
        assert abs(lam - lam_ref) <= 1e-13 * lam_ref
        ctx.close()
