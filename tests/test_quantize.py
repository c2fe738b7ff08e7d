"""Steps and scales of the weight quantiser that are not plain numbers, runs without a GPU."""
import numpy as np
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


def _chain(x, scale, descale):
    q = U.quantize(x, step=2 / scale).clamp(-512 / scale, 510 / scale)
    return q * scale if descale else q


DEVICES = ['cpu', pytest.param('cuda', marks=pytest.mark.gpu)]


@pytest.mark.parametrize('device', DEVICES)
@pytest.mark.parametrize('descale', [False, True])
@pytest.mark.parametrize('scale', [[[64.0], [32.0], [1.0]], [[64.0]], 50.0, 1.0])
def test_scale_is_a_tensor(device, descale, scale):
    """One scale per channel, a trained one: the operators, with their gradients."""
    x = torch.randn(3, 40, generator=torch.Generator().manual_seed(2)) * 5
    g = torch.randn(3, 40, generator=torch.Generator().manual_seed(3)).to(device)
    results = []
    for fx in (lambda v, s: U.quantize_hook_fx(v, scale=s, descale=descale), lambda v, s: _chain(v, s, descale)):
        v, s = x.to(device).requires_grad_(), torch.tensor(scale, device=device).requires_grad_()
        out = fx(v, s)
        results.append((out.detach(),) + torch.autograd.grad(out, (v, s), g))
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize('device', DEVICES)
@pytest.mark.parametrize('scale', [1e-30, 1e30, 2e38, float('inf'), 1, np.float64(64), np.int64(64), True])
def test_scale_beyond_what_one_launch_takes(device, scale):
    """Steps without a float32 reciprocal and limits beyond float32 do what the operators do, an error included."""
    x = torch.randn(3, 40, generator=torch.Generator().manual_seed(2)).to(device)

    def result(fx):
        try:
            return fx().cpu().view(torch.int32)
        except RuntimeError as e:
            return str(e)
    a, b = result(lambda: U.quantize_hook_fx(x, scale=scale)), result(lambda: _chain(x, scale, False))
    assert type(a) is type(b) and (torch.equal(a, b) if torch.is_tensor(a) else a == b)
