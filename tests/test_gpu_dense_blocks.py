"""The dense right-hand side at the edges of its work blocks: element counts
around the number of elements a wavefront holds (64 / face points: 10, 7, 5 for
triangles, 8, 5, 4 for quadrilaterals of order 1, 2, 3), meshes whose shared
edges do and do not have exactly opposite normals (periodic seams), and batches
whose instances meet inside a wavefront. Bar: relative L-infinity per variable
<= 1e-12 against the oracle (the suite's parity bar), wave speeds to 1e-13."""
import numpy as np
import pytest

from oracle.refcpu import RefSolver
from rkdg_amd import mesh as M
from rkdg_amd import scheme as S
from tests.helpers import all_outlet, rel_linf, smooth_state

pytestmark = pytest.mark.gpu


def _bulge(X, Y):
    return X + 0.04 * np.sin(3 * X) * np.cos(2 * Y), Y + 0.05 * np.sin(2 * X + Y)


def _meshes(geom, order):
    if geom == "tri":
        return [M.jittered_delaunay_tri(nx, ny, 0.0, 1.0, 0.0, 1.0, seed=5)
                for nx, ny in ((1, 1), (2, 1), (2, 2), (1, 5), (7, 1), (3, 5))]
    out = [M.structured_quad(nx, ny, warp=_bulge) for nx, ny in ((1, 1), (2, 2), (5, 1), (3, 3), (7, 2), (4, 4))]
    # periodic with extents that are not binary fractions: seam normals differ in the last bit
    out.append(M.structured_quad(5, 3, 0.1, 0.8, -0.3, 1.1, periodic=(True, True)))
    return out


@pytest.mark.parametrize("riemann", [S.RUSANOV, S.HLLC])
@pytest.mark.parametrize("geom,order", [("tri", 1), ("tri", 2), ("tri", 3), ("quad", 1), ("quad", 2), ("quad", 3)])
def test_dense_rhs_block_edges(geom, order, riemann, cuda):
    import torch

    from rkdg_amd.capi import Context

    for m in _meshes(geom, order):
        sch = S.Scheme(riemann=riemann, bcs=all_outlet(m))
        ref = RefSolver(m, order, sch)
        x = smooth_state(ref.node_coords(), seed=8, amp=1e-2)
        y_ref, lam_ref = ref.mult(x)
        ctx = Context(m, order, sch, dense=geom == "quad")
        xd = torch.from_numpy(x).to(cuda)
        yd = torch.full_like(xd, float("nan"))
        lam = ctx.rhs(xd, yd)
        err = rel_linf(yd.cpu().numpy(), y_ref, 4)
        print(f"[dense {geom} p{order}] NE={m.num_elements} rel Linf {err:.2e}", flush=True)
        assert err <= 1e-12
        assert abs(lam - lam_ref) <= 1e-13 * lam_ref
        ctx.close()


@pytest.mark.parametrize("order", [1, 2, 3])
def test_batch_instances_inside_a_block(order, cuda):
    """Instances of 2 to 9 elements: several share a wavefront; states, times and
    wave-speed controlled steps equal the single solves bit for bit."""
    import torch

    from rkdg_amd import solver

    meshes = [M.structured_quad(nx, ny, 0.0, 1.0, 0.0, 0.7, warp=_bulge)
              for nx, ny in ((2, 1), (3, 1), (3, 3), (1, 2), (5, 1))]
    sch = [S.Scheme(riemann=S.HLL, indicator=S.IND_BJ, limiter=S.LIM_MULTI, bcs=all_outlet(m)) for m in meshes]
    ens = solver.Ensemble(meshes, order, sch)
    states = [smooth_state(xyz, seed=k, amp=1e-2) for k, xyz in enumerate(ens.node_coords())]
    x = torch.from_numpy(ens.pack(states)).to(cuda)
    t, dt, steps = solver.run_batch(ens, x, 10.0, 0.2, max_steps=3)
    got = ens.unpack(x.cpu().numpy())
    for k, m in enumerate(meshes):
        f = solver.FE_Evolution(m, order, sch[k], dense=True)
        lim = solver.Limiter(f)
        rk = solver.ExplicitRKLimitedSolver(*S.TABLEAUS["ssprk3"], limiter=lim)
        xs = torch.from_numpy(states[k]).to(cuda)
        st = solver.run(f, rk, lim, xs, 10.0, 0.2, max_steps=3)
        assert np.array_equal(xs.cpu().numpy(), got[k])
        assert st.t == t[k] and st.dt == dt[k] and steps[k] == 3
