"""rkdg_adjoint_solve with every choice of segments: all steps recorded (the
default where the records fit), one step per segment, segments that do not
divide the number of steps, a segment longer than the run. The steps and their
transposes are the same arithmetic whichever of them are recomputed, so the
objective, the gradient and the final state are the same bits; the boundary
parameters' adjoint is summed by atomics, compared to 1e-12 of its size."""
import numpy as np
import pytest

from rkdg_amd import scheme as S
from rkdg_amd.adjoint import FFSProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tableau", ["ssprk3", "ref_literal_rk2"])
def test_segments_agree(tableau, cuda):
    import torch

    P = FFSProblem(nx=20, ny=10, v_in=0.05)
    ctx, slot = P.prob.ctx, P.prob.obj_slot
    tab = S.TABLEAUS[tableau]
    x0 = P.prob.limit(P.initial_state(torch.tensor(3.0, dtype=torch.float64, device=cuda),
                                      torch.from_numpy(P.perturbation()).to(cuda)))
    dts = np.linspace(1.0, 1.3, 7) * 1e-3
    want = None
    for every in (0, 1, 2, 3, 4, 6, 7, 20):
        xbar, xN = torch.empty_like(x0), torch.empty_like(x0)
        J, pbar = ctx.adjoint_solve(x0, dts, tab, slot, xbar, every=every, xN=xN)
        if want is None:
            want = (J, xbar, xN, pbar)
            xf = x0.clone()
            assert ctx.forward_solve(xf, dts, tab, slot) == J
            assert torch.equal(xf, xN)
            assert float(xbar.abs().max()) > 0.0
        assert J == want[0], every
        assert torch.equal(xbar, want[1]), every
        assert torch.equal(xN, want[2]), every
        assert np.abs(pbar - want[3]).max() <= 1e-12 * np.abs(want[3]).max()
