"""Steps and scales of the weight quantiser that are not plain numbers, runs without a GPU."""
import pytest
import torch

import lava_dl_amd.slayer as slayer

U = slayer.utils


@pytest.mark.parametrize('requires_grad', [False, True])
@pytest.mark.parametrize('step', [[[0.5], [0.25], [1.0]], [[1.0], [1.0], [1.0]], 0.25, 1.0])
@pytest.mark.parametrize('mode', [U.MODE.ROUND, U.MODE.FLOOR])
def test_step_is_a_tensor(requires_grad, step, mode):
    x = (torch.randn(3, 40, generator=torch.Generator().manual_seed(1)) * 3).requires_grad_(requires_grad)
    step = torch.tensor(step)
    out = U.quantize(x, step=step, mode=mode)
    snap = torch.round if mode == U.MODE.ROUND else torch.floor
    assert torch.equal(out.detach(), snap(x.detach() / step) * step)
    if requires_grad:
        out.sum().backward()
        assert torch.equal(x.grad, torch.ones(3, 40))
