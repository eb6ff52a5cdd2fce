"""The Rusanov flux on hexahedra is taken outward from each element (its own side
first) up to order 2 and in the face's order above: rotated elements, walls and
periodic faces, against the oracle (relative L-infinity per variable <= 1e-12), and
conservation: on a periodic mesh the integral of the right-hand side is a sum of face
terms that cancel in pairs, so what is left is rounding of the sum, below 64 eps of
the sum of the magnitudes (each of up to 27 * 64 terms is rounded a few times, and
the errors of a sum of n terms grow like sqrt(n)). That the two elements see the same
bits is test_flux_pairs.py's."""
import numpy as np
import pytest

from oracle.refcpu import RefSolver
from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, rel_linf, scramble_orientations, smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", [1, 2, 3])
@pytest.mark.parametrize("periodic", [True, False])
def test_outward_flux(order, periodic, cuda):
    import torch

    from rkdg_amd.capi import Context

    m = scramble_orientations(M.structured_hex(3, 3, 3, periodic=(periodic,) * 3), seed=7)
    sch = S.Scheme(riemann=S.RUSANOV, bcs=all_outlet(m))
    ref = RefSolver(m, order, sch)
    x = smooth_state(ref.node_coords(), seed=5, amp=1e-2)
    y_ref, lam_ref = ref.mult(x)
    ctx = Context(m, order, sch)
    xd = torch.from_numpy(x).to(cuda)
    yd = torch.full_like(xd, float("nan"))
    lam = ctx.rhs(xd, yd)
    y = yd.cpu().numpy()
    assert rel_linf(y, y_ref, 5) <= 1e-12
    assert abs(lam - lam_ref) <= 1e-13 * lam_ref
    if periodic:
        t, w = np.polynomial.legendre.leggauss(order + 1)
        w3 = np.einsum("i,j,k->ijk", w, w, w).ravel() / 8.0  # equal elements: the volume drops out
        c = y.reshape(5, -1, w3.size) * w3
        assert np.all(np.abs(c.sum(axis=(1, 2))) <= 64 * np.finfo(float).eps * np.abs(c).sum(axis=(1, 2)))
    ctx.close()
