"""A fused neuron whose spikes get no gradient back (a later function returns None for them) hands zero gradients to its
input and parameters, as autograd's own zero filling does; the fused functions switch that off for their traces."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu


class _NoGradient(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x):
        return x.clone()

    @staticmethod
    def backward(ctx, grad):
        return None


@pytest.mark.parametrize('model', ['cuba', 'alif', 'rf'])
@pytest.mark.parametrize('learn', [False, True])
def test_no_gradient_for_the_spikes_is_a_zero_gradient(model, learn):
    import lava_dl_amd.slayer as slayer
    decays = {'cuba': dict(current_decay=0.25, voltage_decay=0.1), 'rf': dict(period=20, decay=0.1),
              'alif': dict(threshold_step=0.5, current_decay=0.25, voltage_decay=0.1, threshold_decay=0.2,
                           refractory_decay=0.3)}[model]
    neuron = getattr(slayer.neuron, model).Neuron(threshold=1.0, requires_grad=learn, **decays).to(dev())
    inputs = [torch.randn(2, 3, 21, device=dev(), requires_grad=True) for _ in range(2 if model == 'rf' else 1)]
    _NoGradient.apply(neuron(tuple(inputs) if len(inputs) > 1 else inputs[0])).sum().backward()
    for x in inputs:
        assert x.grad is not None and not x.grad.any()


def test_no_gradient_for_the_adaptive_resonator_is_a_zero_gradient():
    import lava_dl_amd.slayer as slayer
    shape, zero = (2, 3, 21), torch.zeros(1, device=dev())
    x = [torch.randn(shape, device=dev(), requires_grad=True) for _ in range(2)]
    sin, cos = (torch.full((1,), v, device=dev(), requires_grad=True) for v in (100.0, 2048.0))
    decay = torch.full((1,), 400.0, device=dev())
    dynamics = slayer.neuron.dynamics.adaptive_resonator.dynamics
    re, im, *_ = dynamics(*x, sin, cos, decay, decay, zero, zero, zero, zero, 1.0, 1.0, 64)
    (_NoGradient.apply(re) + _NoGradient.apply(im)).sum().backward()
    for t in x + [sin, cos]:
        assert t.grad is not None and not t.grad.any()
    # a gradient of one of the two is what a gradient of zeros beside it gives
    re, im, *_ = dynamics(*x, sin, cos, decay, decay, zero, zero, zero, zero, 1.0, 1.0, 64)
    g = torch.randn(shape, device=dev())
    one = torch.autograd.grad(re + _NoGradient.apply(im), x + [sin, cos], g, retain_graph=True)
    both = torch.autograd.grad([re, im], x + [sin, cos], [g, torch.zeros_like(g)])
    assert all(torch.equal(a, b) for a, b in zip(one, both))
