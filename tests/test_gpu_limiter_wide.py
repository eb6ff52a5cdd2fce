"""The tensor limiter on either side of the size (256 workgroups of 8 hexahedra or 16
quadrilaterals) up to which a workgroup takes one wavefront per variable: a small mesh
alone and beside an unconnected large one, the same bits on the small one's elements
(the forms share their arithmetic; test_gpu_limiter_blocks compares it with the
oracle)."""
import numpy as np
import pytest

from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, smooth_state
from tests.test_gpu_limiter_blocks import KINDS

pytestmark = pytest.mark.gpu


def beside(a, b):
    shift = int(a.elem_verts.max()) + 1
    return M.Mesh(a.geom, np.concatenate([a.elem_coords, b.elem_coords]),
                  np.concatenate([a.elem_verts, b.elem_verts + shift]),
                  np.concatenate([a.bdr_verts, b.bdr_verts + shift]), np.concatenate([a.bdr_attr, b.bdr_attr]))


@pytest.mark.parametrize("kind", [*KINDS, "everywhere"])
@pytest.mark.parametrize("small,large,order", [((5, 4, 7), (683, 3, 1), 2), ((3, 3, 1), (16, 16, 8), 2),
                                               ((16, 16, 8), (1, 1, 1), 2), ((5, 4, 7), (683, 3, 1), 3),
                                               ((16, 16, 8), (1, 1, 1), 3), ((13, 10), (241, 17), 4),
                                               ((64, 64), (1, 1), 4), ((13, 10), (241, 17), 5),
                                               ((64, 64), (1, 1), 5)])
def test_both_forms(small, large, order, kind, cuda):
    import torch

    from rkdg_amd.capi import Context

    dim = len(small)

    def box(n):
        # extents that are powers of two times the spacing: exact parallelograms, the tensor path
        return (M.structured_quad(*n, x1=n[0] / 4.0, y1=n[1] / 4.0) if dim == 2 else
                M.structured_hex(*n, box=tuple((0.0, k / 4.0) for k in n), periodic=(False,) * 3))

    a, b = box(small), box(large)
    opts = dict(indicator=S.IND_BJ, **KINDS[kind]) if kind in KINDS else dict(
        indicator=S.IND_EVERYWHERE, phi=S.PHI_BJ, limiter=S.LIM_MULTI)
    got = []
    for m in (a, beside(a, b)):
        ctx = Context(m, order, S.Scheme(riemann=S.RUSANOV, bcs=all_outlet(m), **opts))
        xyz = ctx.node_coords()[:a.num_elements] / np.array([k / 4.0 for k in small])
        U = smooth_state(xyz, seed=9, amp=1e-4).reshape(dim + 2, -1)
        j = (xyz[..., 0].ravel() > 0.55).astype(float)  # a jump through some elements
        U[0] *= 1.0 + 1.5 * j
        U[-1] *= 1.0 + 2.5 * j
        n, rest = U.shape[1], ctx.info.num_dofs - U.shape[1]
        fill = np.array([1.0] + [0.1] * dim + [2.5])[:, None] * np.ones((1, rest))
        x = torch.from_numpy(np.concatenate([U, fill], axis=1).reshape(-1)).to(cuda)
        flags = torch.full((m.num_elements,), 7, dtype=torch.int8, device=cuda)
        ctx.limit(x, flags)
        got.append((x.cpu().numpy().reshape(dim + 2, -1)[:, :n], flags.cpu().numpy()[:a.num_elements]))
        ctx.close()
    assert np.all(np.isfinite(got[0][0])) and not np.array_equal(got[0][0], U)
    assert np.array_equal(got[0][0], got[1][0])
    assert np.array_equal(got[0][1], got[1][1])
