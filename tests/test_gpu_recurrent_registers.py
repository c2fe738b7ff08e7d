"""Recurrent layers of up to 256 neurons keep their matrix in registers, sixteen columns in a row of lanes and four
neurons to a row: widths around the multiples of 16 and 64 the layout is cut at, and sample lengths around the four
steps a quad of lanes moves, against the CPU oracle.  Weights are quantised, so the forward pass is exact; a gradient
is a sum of at most 256 terms in another order, recursively over at most 9 steps (bar 1e-5, as in the other tests)."""
import pytest
import torch

from oracle import slayer_oracle as O
from tests.util import dev, assert_exact, assert_rel

pytestmark = pytest.mark.gpu

WIDTHS = [1, 15, 17, 64, 65, 128, 129, 192, 193, 255, 256]


class _Dense(torch.nn.Module):
    def __init__(self, weight):
        super().__init__()
        self.weight = torch.nn.Parameter(weight.reshape(weight.shape + (1, 1, 1)))
        self.pre_hook_fx = None


@pytest.mark.parametrize('c', WIDTHS)
@pytest.mark.parametrize('t', [1, 3, 4, 9])
@pytest.mark.parametrize('kind,graded', [('cuba', False), ('alif', False), ('alif', True)])
def test_register_kernels_match_the_oracle(c, t, kind, graded, monkeypatch):
    import lava_dl_amd.slayer as slayer
    monkeypatch.setattr(slayer.utils.recurrent, 'STEPS_FROM', 10 ** 9)
    gen = torch.Generator().manual_seed(1000 * c + 10 * t + graded)
    n = 3
    z = torch.randn(n, c, t, generator=gen) * 3
    # graded spikes feed voltages back: weights of 1/32 on a few inputs keep every product and sum exact
    w = torch.randint(-2, 3, (c, c), generator=gen).float() / 32
    w[torch.rand(c, c, generator=gen) > 4.0 / c] *= 0.0 if graded else 0.5
    syn = _Dense(w).to(dev())
    if kind == 'cuba':
        neuron = slayer.neuron.cuba.Neuron(threshold=1.25, current_decay=0.25, voltage_decay=0.25,
                                           persistent_state=True).to(dev())
        names, states = ('current', 'voltage'), [torch.zeros(1)] * 2
    else:
        neuron = slayer.neuron.alif.Neuron(threshold=1.0, threshold_step=0.5, current_decay=0.5, voltage_decay=0.5,
                                           threshold_decay=0.1, refractory_decay=0.2, persistent_state=True,
                                           graded_spike=graded).to(dev())
        names = ('current', 'voltage', 'threshold', 'refractory')
        states = [torch.zeros(1), torch.zeros(1), torch.tensor([neuron.threshold]), torch.zeros(1)]
    zg = z.to(dev()).requires_grad_()
    out = slayer.utils.recurrent.custom_recurrent(zg, neuron, syn)
    decays = [getattr(neuron, f'{k}_decay').detach().round().cpu() for k in names]
    if kind == 'cuba':
        theta = neuron.threshold + neuron.threshold_eps
        spk, vol, *last = O.recurrent_cuba_fwd(z, w, *decays, *states, 4096, theta)
    else:
        spk, vol, theta, last = O.recurrent_alif_fwd(z, w, decays, states, neuron.threshold_step, neuron.threshold,
                                                     4096, graded=graded)
    assert_exact(out, spk, 'spikes')
    for k, want in zip(names, last):
        assert_exact(getattr(neuron, f'{k}_state'), want, f'carried {k}')
    g = torch.rand(n, c, t, generator=gen)
    out.backward(g.to(dev()))
    gz, gw = O.recurrent_cuba_bwd(g, spk, vol, w, theta, neuron.tau_rho * 100, neuron.scale_rho * 0.1, graded=graded)
    assert_rel(zg.grad, gz, 'grad z')
    assert_rel(syn.weight.grad.reshape(c, c), gw, 'grad weight')


@pytest.mark.parametrize('graded', [False, True])
def test_large_batches_give_the_same_spikes_in_either_form(graded, monkeypatch):
    """193 neurons, 1023 and 1024 samples: the batch from which the forward pass takes the gathering form."""
    import lava_dl_amd.slayer as slayer
    monkeypatch.setattr(slayer.utils.recurrent, 'STEPS_FROM', 10 ** 9)
    gen = torch.Generator().manual_seed(7)
    z, c = torch.randn(1024, 193, 5, generator=gen) * 3, 193
    w = torch.randint(-2, 3, (c, c), generator=gen).float() / 32
    w[torch.rand(c, c, generator=gen) > 4.0 / c] = 0.0               # graded products and sums exact
    outs = []
    for n in (1023, 1024):
        neuron = slayer.neuron.alif.Neuron(threshold=1.0, threshold_step=0.5, current_decay=0.5, voltage_decay=0.5,
                                           threshold_decay=0.1, refractory_decay=0.2, persistent_state=True,
                                           graded_spike=graded).to(dev())
        outs.append(slayer.utils.recurrent.custom_recurrent(z[:n].to(dev()), neuron, _Dense(w).to(dev())))
    assert outs[0].any() and torch.equal(outs[0], outs[1][:1023])


@pytest.mark.parametrize('c', [5, 70, 140, 255])
@pytest.mark.parametrize('kind,graded', [('cuba', False), ('alif', False), ('alif', True)])
@pytest.mark.parametrize('value', [float('inf'), float('-inf'), float('nan')])
def test_a_weight_that_is_not_finite_counts_when_its_neuron_fires(c, kind, graded, value, monkeypatch):
    """A silent neuron feeds nothing back whatever its weights (0 * inf would be a NaN, which the fixed-point current takes
    as zero: the receiving neuron would lose its input); the wider layers' kernels gather the rows of the firing ones."""
    import lava_dl_amd.slayer as slayer
    monkeypatch.setattr(slayer.utils.recurrent, 'STEPS_FROM', 10 ** 9)
    gen = torch.Generator().manual_seed(c)
    z = torch.rand(2, c, 11, generator=gen) * 3
    silent, to = c // 2, c - 1
    z[:, silent] = -1.0
    w = torch.randint(-2, 3, (c, c), generator=gen).float() / 64
    w[silent] = 0.0
    outs = []
    for weight in (0.0, value):
        w[to, silent] = weight
        if kind == 'cuba':
            neuron = slayer.neuron.cuba.Neuron(threshold=1.25, current_decay=0.25, voltage_decay=0.25, persistent_state=True)
        else:
            neuron = slayer.neuron.alif.Neuron(threshold=1.0, threshold_step=0.5, current_decay=0.5, voltage_decay=0.5,
                                               threshold_decay=0.1, refractory_decay=0.2, persistent_state=True,
                                               graded_spike=graded)
        outs.append(slayer.utils.recurrent.custom_recurrent(z.to(dev()), neuron.to(dev()), _Dense(w).to(dev())).cpu())
    assert not outs[0][:, silent].any() and outs[0][:, to].any()
    assert torch.equal(*outs)
