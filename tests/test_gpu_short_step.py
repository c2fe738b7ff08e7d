"""The short form of a fixed-point step (multipliers that are not negative) against the general one.  A wave takes it when
all of its 64 rows do, so one decay above 4096 among them puts the others on the general form: they must not change."""
import pytest
import torch

from oracle import slayer_oracle as O
from tests.util import dev, assert_exact

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def slayer():
    import lava_dl_amd.slayer as s
    return s


def _events(shape, seed):
    gen = torch.Generator().manual_seed(seed)
    return (torch.rand(shape, generator=gen) < 0.2).float() * torch.randn(shape, generator=gen) * 40


# whole quads and rows that are not; several chunks of 32 steps, so interior ones
@pytest.mark.parametrize('t', [300, 301, 1450])
@pytest.mark.parametrize('threshold', [0, 2.5])
def test_integrator_with_decays_on_either_side(slayer, t, threshold):
    c = 192
    decay = torch.randint(0, 4097, (c,), generator=torch.Generator().manual_seed(t)).float()
    decay[:4] = torch.tensor([0.0, 1.0, 4095.0, 4096.0])
    mixed = decay.clone()
    mixed[70], mixed[100] = 4146.0, 6000.0                                 # the second wave's rows take the general form
    x, zero = _events((2, c, t), t), torch.tensor([0.0])
    li = slayer.neuron.dynamics.leaky_integrator.dynamics
    args = (64, threshold) if threshold else (64,)
    for d in (decay, mixed):
        assert_exact(li(x.to(dev()), d.to(dev()), zero.to(dev()), *args), O.li_fwd(x, d, zero, *args), 'integrator')


@pytest.mark.parametrize('t', [300, 1450])
@pytest.mark.parametrize('model', ['cuba', 'alif'])
@pytest.mark.parametrize('shape', [(2, 64), (300, 64)])
def test_fused_neurons_in_both_forms(slayer, model, t, shape):
    c = shape[1]
    common = dict(threshold=1.0, current_decay=[0, 1], voltage_decay=[0, 1], shared_param=False)
    neuron = (slayer.neuron.cuba.Neuron(**common) if model == 'cuba' else
              slayer.neuron.alif.Neuron(threshold_step=0.5, threshold_decay=[0, 1], refractory_decay=[0, 1], **common)).to(dev())
    x = _events(shape + (t,), t).div(40).to(dev()).requires_grad_()
    neuron(x)
    names = [k for k, _ in neuron.named_parameters(recurse=False)]
    rows = [i for i in range(c) if i != 9]
    for name in names:                                                     # each of the multipliers by itself
        plain = neuron(x).detach()
        param = getattr(neuron, name)
        before = param.data.clone()
        param.data[9] = 5000.0
        mixed = neuron(x).detach()
        param.data.copy_(before)
        assert 0 < float(plain.mean()) < 1
        assert torch.equal(plain[:, rows], mixed[:, rows]), name
