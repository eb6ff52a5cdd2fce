"""Non-conforming faces where one element carries many of them: the centre of a
3^dim mesh whose neighbours are all refined is the master of 2^(dim-1) slave
faces on each side (24 in 3D), more than the wavefronts that share an element's
faces. Every order, against the oracle; bar: relative L-infinity per variable
<= 1e-12 (the suite's parity bar), wave speed to 1e-13."""
import numpy as np
import pytest

from oracle.refcpu import RefSolver
from rkdg_amd import amr
from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, rel_linf, smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,order", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3)])
def test_surrounded_master(dim, order, cuda):
    import torch

    from rkdg_amd.capi import Context

    base = M.structured_hex(3, 3, 3, periodic=(False,) * 3) if dim == 3 else M.structured_quad(3, 3)
    tree = amr.NCMesh(base)
    tree.refine([e for e in range(base.num_elements) if e != base.num_elements // 2])
    m = tree.mesh()
    masters, count = np.unique(m.nc[:, 2], return_counts=True)
    assert count.max() == 2 * dim * 2 ** (dim - 1)
    sch = S.Scheme(riemann=S.RUSANOV, bcs=all_outlet(m))
    ref = RefSolver(m, order, sch)
    x = smooth_state(ref.node_coords(), seed=6, amp=1e-3)
    y_ref, lam_ref = ref.mult(x)
    ctx = Context(m, order, sch)
    xd = torch.from_numpy(x).to(cuda)
    yd = torch.empty_like(xd)
    lam = ctx.rhs(xd, yd)
    err = rel_linf(yd.cpu().numpy(), y_ref, dim + 2)
    print(f"[nc items dim {dim} p{order}] {err:.2e}", flush=True)
    assert err <= 1e-12
    assert abs(lam - lam_ref) <= 1e-13 * lam_ref
    ctx.close()
