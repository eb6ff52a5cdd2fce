"""A neighbour whose mean is not a number bounds nothing in the limiter's stencil
(the reference's comparisons skip it, indicator_bj.cpp:15-86): with one element of
NaN, the limited state of every other element against the oracle, 1e-12 of the
largest node value of each variable (the limited state combines node values). And a
node that is not finite leaves none of its variable finite in the multiplier's element,
mean + y (u - mean), also where y = 1 (limiter_multiplier.cpp:24-38): the same nodes
are finite as in the oracle."""
import numpy as np
import pytest

from oracle.refcpu import RefSolver
from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, smooth_state

pytestmark = pytest.mark.gpu

CASES = ["quad1", "quad3", "hex1", "hex2", "hex3", "tri2", "bilinear2"]


def _mesh(case):
    kind, order = case[:-1], int(case[-1])
    if kind == "hex":
        m = M.structured_hex(4, 4, 4, periodic=(False,) * 3)
    elif kind == "tri":
        m = M.jittered_delaunay_tri(4, 4)
    elif kind == "quad":
        m = M.structured_quad(4, 4)
    else:
        m = M.structured_quad(4, 4, warp=lambda X, Y: (X, Y * (1.0 + 0.2 * X)))
    return m, order


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("limiter", [S.LIM_MULTI, S.LIM_FINDIFF])
def test_stencil_skips_nan(case, limiter, cuda):
    import torch

    from rkdg_amd.capi import Context

    m, order = _mesh(case)
    sch = S.Scheme(riemann=S.HLL, indicator=S.IND_BJ, phi=S.PHI_BJ, limiter=limiter, bcs=all_outlet(m))
    ref = RefSolver(m, order, sch)
    xyz = ref.node_coords()
    U = smooth_state(xyz, seed=2, amp=1e-3).reshape(m.dim + 2, -1)
    j = 1.0 + 2.0 * (xyz[..., 0].ravel() > 0.4)
    U[0] *= j
    U[-1] *= j
    ne, nd = m.num_elements, ref.nd
    for bad in range(0, ne, 5):
        x = U.reshape(m.dim + 2, ne, nd).copy()
        x[:, bad] = np.nan
        x = x.reshape(-1)
        x_ref = ref.limit(x)[0].reshape(m.dim + 2, ne, nd)
        ctx = Context(m, order, sch)
        xd = torch.from_numpy(x).to(cuda)
        ctx.limit(xd)
        got = xd.cpu().numpy().reshape(m.dim + 2, ne, nd)
        rest = np.arange(ne) != bad
        scale = np.abs(U).max(axis=1)[:, None, None]
        assert np.all(np.isfinite(x_ref[:, rest]))
        assert np.all(np.abs(got[:, rest] - x_ref[:, rest]) <= 1e-12 * scale), bad
        ctx.close()


@pytest.mark.parametrize("case", CASES)
@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("indicator", [S.IND_BJ, S.IND_NOWHERE])
def test_nonfinite_node_spreads(case, value, indicator, cuda):
    import torch

    from rkdg_amd.capi import Context

    m, order = _mesh(case)
    sch = S.Scheme(riemann=S.HLL, indicator=indicator, phi=S.PHI_BJ, limiter=S.LIM_MULTI, last_hope=0,
                   bcs=all_outlet(m))
    ref = RefSolver(m, order, sch)
    ctx = Context(m, order, sch)
    ne, nd = m.num_elements, ref.nd
    # constant but for rounding: the indicator leaves every element alone
    U = np.array([1.0] + [0.3] * m.dim + [2.5])[:, None, None] * np.ones((1, ne, nd))
    for v in range(m.dim + 2):
        x = U.copy()
        x[v, ne // 2, nd - 1] = value
        x_ref = ref.limit(x.reshape(-1))[0]
        xd = torch.from_numpy(x.reshape(-1)).to(cuda)
        ctx.limit(xd)
        assert np.array_equal(np.isfinite(xd.cpu().numpy()), np.isfinite(x_ref)), v
    ctx.close()
