"""What an adjoint solve leaves on the card: the records of all steps where they fit
2 GiB, else one segment's and the checkpoints, which stay below that too."""
import numpy as np
import pytest

from rkdg_amd.adjoint import FFSProblem

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("steps", [140, 200])
def test_held_memory(steps, cuda):
    import torch

    P = FFSProblem(nx=240, ny=80, v_in=0.05)
    x0 = P.prob.limit(P.initial_state(torch.tensor(3.0, dtype=torch.float64, device=cuda),
                                      torch.from_numpy(P.perturbation()).to(cuda)))
    record = 8 * 7 * x0.numel()  # a step of three stages: 14.45 MB
    P.prob.gradient(x0, np.full(1, 1e-5))
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    P.prob.gradient(x0, np.full(steps, 1e-5))
    torch.cuda.synchronize()
    held = before - torch.cuda.mem_get_info()[0]
    assert 0 <= held <= 2.2e9  # 2 GiB and the allocator's rounding
    assert (held > 100 * record) == (steps * record <= 2 << 30)
    P.prob.ctx.close()
