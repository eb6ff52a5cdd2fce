"""The tensor limiter and means kernels at the edges of their work blocks (8
hexahedra or 16 quadrilaterals per wavefront; 16 to 128 elements per means
workgroup), every order, limiter function and limiter, with boundary faces and
elements the indicator leaves alone: the limited state, the flags and the means
against the oracle. Bar: 1e-12 of the largest node value of each variable (the
limited state combines node values; on the smallest meshes a momentum's mean may
cancel) and identical flags but within 1e-12 of the threshold."""
import numpy as np
import pytest

from oracle.refcpu import RefSolver
from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, smooth_state

pytestmark = pytest.mark.gpu

KINDS = {
    "michalak": dict(phi=S.PHI_MICHALAK, limiter=S.LIM_MULTI),
    "bj": dict(phi=S.PHI_BJ, limiter=S.LIM_MULTI, last_hope=0),
    "venkat": dict(phi=S.PHI_VENKAT, venkat_k=5.0, limiter=S.LIM_MULTI, pow_nd=0),
    "findiff": dict(phi=S.PHI_BJ, limiter=S.LIM_FINDIFF),
}
SIZES = {2: ((1, 1), (5, 3), (16, 1), (17, 1), (13, 10)), 3: ((1, 1, 1), (7, 1, 1), (2, 2, 2), (3, 3, 1), (5, 4, 7))}


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("dim,order", [(2, 1), (2, 2), (2, 3), (2, 4), (2, 5), (3, 1), (3, 2), (3, 3)])
def test_limiter_block_edges(dim, order, kind, cuda):
    import torch

    from rkdg_amd.capi import Context

    for n in SIZES[dim]:
        # extents that are powers of two times the spacing: exact parallelograms, the tensor path
        m = (M.structured_quad(*n, x1=n[0] / 4.0, y1=n[1] / 4.0) if dim == 2 else
             M.structured_hex(*n, box=tuple((0.0, k / 4.0) for k in n), periodic=(False,) * 3))
        sch = S.Scheme(riemann=S.RUSANOV, indicator=S.IND_BJ, bcs=all_outlet(m), **KINDS[kind])
        ref = RefSolver(m, order, sch)
        xyz = ref.node_coords()
        x = smooth_state(xyz / np.array([k / 4.0 for k in n]), seed=9, amp=1e-4)
        U = x.reshape(dim + 2, -1)
        j = (xyz[..., 0].ravel() > 0.55 * n[0] / 4.0).astype(float)  # a jump through some elements
        U[0] *= 1.0 + 1.5 * j
        U[-1] *= 1.0 + 2.5 * j
        x = np.ascontiguousarray(U.reshape(-1))
        x_ref, _, ymin = ref.limit(x)
        ctx = Context(m, order, sch)
        xd = torch.from_numpy(x).to(cuda)
        md = torch.full(((dim + 2) * m.num_elements,), float("nan"), dtype=torch.float64, device=cuda)
        ctx.means(xd, md)
        # a weighted sum of at most 64 node values: rounding is relative to them, not to a mean
        # that they may cancel to
        err = np.abs(md.cpu().numpy() - ref.means(x)).reshape(dim + 2, -1).max(axis=1)
        assert np.all(err <= 1e-13 * np.abs(U).max(axis=1))
        fd = torch.full((m.num_elements,), 7, dtype=torch.int8, device=cuda)
        ctx.limit(xd, fd)
        if m.num_elements == 1 and not sch.last_hope:
            # no interior face: the indicator keeps its start value 1e9, whose power overflows in
            # the reference and here alike; only the last hope gives such an element a result
            continue
        err = np.abs(xd.cpu().numpy() - x_ref).reshape(dim + 2, -1).max(axis=1)
        assert np.all(err <= 1e-12 * np.abs(U).max(axis=1))
        if KINDS[kind]["limiter"] == S.LIM_MULTI:
            flags = fd.cpu().numpy()
            assert np.all(((flags & 1) == (ymin < 1.0)) | (np.abs(ymin - 1.0) < 1e-12)), (n, kind)
        ctx.close()


@pytest.mark.parametrize("kind", list(KINDS))
@pytest.mark.parametrize("geom,order", [("tri", 1), ("tri", 2), ("tri", 3), ("quad", 1), ("quad", 2), ("quad", 3)])
def test_dense_limiter_block_edges(geom, order, kind, cuda):
    """The dense limiter holds 21 triangles or 16 quadrilaterals per wavefront."""
    import torch

    from rkdg_amd.capi import Context

    def bulge(X, Y):
        return X + 0.04 * np.sin(3 * X) * np.cos(2 * Y), Y + 0.05 * np.sin(2 * X + Y)

    sizes = ((2, 1), (5, 2), (7, 3), (3, 7), (9, 8)) if geom == "tri" else ((2, 1), (5, 3), (4, 4), (17, 1), (13, 9))
    for nx, ny in sizes:
        m = (M.jittered_delaunay_tri(nx, ny, 0.0, 1.0, 0.0, 1.0, seed=3) if geom == "tri"
             else M.structured_quad(nx, ny, warp=bulge))
        sch = S.Scheme(riemann=S.HLLC, indicator=S.IND_BJ, bcs=all_outlet(m), **KINDS[kind])
        ref = RefSolver(m, order, sch)
        xyz = ref.node_coords()
        U = smooth_state(xyz, seed=9, amp=1e-4).reshape(4, -1)
        j = (xyz[..., 0].ravel() > 0.55).astype(float)
        U[0] *= 1.0 + 1.5 * j
        U[-1] *= 1.0 + 2.5 * j
        x = np.ascontiguousarray(U.reshape(-1))
        x_ref, _, ymin = ref.limit(x)
        ctx = Context(m, order, sch, dense=geom == "quad")
        xd = torch.from_numpy(x).to(cuda)
        fd = torch.full((m.num_elements,), 7, dtype=torch.int8, device=cuda)
        ctx.limit(xd, fd)
        err = np.abs(xd.cpu().numpy() - x_ref).reshape(4, -1).max(axis=1)
        assert np.all(err <= 1e-12 * np.abs(U).max(axis=1)), (m.num_elements, kind)
        if KINDS[kind]["limiter"] == S.LIM_MULTI:
            flags = fd.cpu().numpy()
            assert np.all(((flags & 1) == (ymin < 1.0)) | (np.abs(ymin - 1.0) < 1e-12)), (m.num_elements, kind)
        ctx.close()
