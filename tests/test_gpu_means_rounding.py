"""The rounding error of the tensor element means. One node's share is near 1 and each
of the others is 0.52 units in its last place, so a sum that adds them to it one by one
rounds up every time: (nodes - 1) * 0.48 units, up to 30. With at most 3 additions per
partial sum and 5 levels above them no share passes more than 8 additions, so the error
stays below 8 * 0.5 units = 8 eps/2, to which the division adds one rounding and the
weights below another: 12 * eps/2 is allowed. The weights are the kernel's own: the
means of states that are 1 at one node."""
import numpy as np
import pytest

from rkdg_amd import mesh as M
from rkdg_amd import scheme as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,order", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3)])
def test_means_are_short_sums(dim, order, cuda):
    import torch

    from rkdg_amd.capi import Context

    m = M.structured_quad(3, 3) if dim == 2 else M.structured_hex(3, 3, 3)
    ctx = Context(m, order, S.Scheme(riemann=S.RUSANOV))
    ne, neq, nd = m.num_elements, dim + 2, (order + 1) ** dim
    out = torch.empty(neq * ne, dtype=torch.float64, device=cuda)

    def means(u):
        """means of every element and variable for the node values u [nd]"""
        ctx.means(torch.from_numpy(np.tile(u, neq * ne)).to(cuda), out)
        return out.cpu().numpy()

    w = np.array([means(np.eye(nd)[k])[0] for k in range(nd)])
    assert abs(w.sum() - 1.0) < 1e-14
    for big in (0, nd // 2, nd - 1):
        u = 0.52 * 2.0 ** -52 / w
        u[big] = 1.0 / w[big]
        exact = (w.astype(np.longdouble) * u).sum()
        assert np.all(np.abs(means(u) - exact) <= 12 * 2.0 ** -53 * exact), big
    ctx.close()
