"""Q1 hexahedra at the edges of the right-hand side's work blocks (three elements
per wavefront, four idle lanes): element counts 1 to 5, 26 and 27, walls and
periodic, aligned and rotated elements, the two-colour form, every Riemann
solver, against the oracle. Bar: relative L-infinity per variable <= 1e-12."""
import numpy as np
import pytest

from oracle.refcpu import RefSolver
from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, rel_linf, scramble_orientations, smooth_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("riemann", [S.RUSANOV, S.LLF, S.HLL, S.HLLC])
@pytest.mark.parametrize("form", ["aligned", "rotated", "two_colour"])
def test_q1hex_block_edges(form, riemann, cuda):
    import torch

    from rkdg_amd.capi import Context

    walls = [(1, 1, 1), (2, 1, 1), (1, 3, 1), (2, 1, 2), (5, 1, 1), (13, 2, 1)]
    meshes = [M.structured_hex(*n, periodic=(False,) * 3) for n in walls] + [M.structured_hex(3, 3, 3)]
    if form == "two_colour":  # interior faces only, even extents
        meshes = [M.structured_hex(4, 4, 4), M.structured_hex(6, 4, 4)]
    for m in meshes:
        if form == "rotated":
            m = scramble_orientations(m, seed=4)
        sch = S.Scheme(riemann=riemann, bcs=all_outlet(m))
        ref = RefSolver(m, 1, sch)
        x = smooth_state(ref.node_coords(), seed=2, amp=1e-2)
        y_ref, lam_ref = ref.mult(x)
        ctx = Context(m, 1, sch, two_colour=form == "two_colour")
        assert ctx.info.two_colour == (form == "two_colour")
        xd = torch.from_numpy(x).to(cuda)
        yd = torch.full_like(xd, float("nan"))
        lam = ctx.rhs(xd, yd)
        assert rel_linf(yd.cpu().numpy(), y_ref, 5) <= 1e-12, (form, m.num_elements)
        assert abs(lam - lam_ref) <= 1e-13 * lam_ref
        ctx.close()
