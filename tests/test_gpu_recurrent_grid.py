"""Recurrent layers whose time loop is one launch spread over the chip (csrc/recurrent_grid.hip): at the edges of its
tiles -- one and two sample tiles per workgroup, units of 128 presynaptic neurons, chunks of 16 steps, the shortest
sequence it takes -- against the CPU oracle, and with weights that are not on a quantiser's grid."""
import os
import subprocess
import sys
import threading

import pytest
import torch

from oracle import slayer_oracle as O
from tests import test_gpu_recurrent as base
from tests.util import dev, assert_exact, assert_rel

pytestmark = pytest.mark.gpu

BINARY = os.path.join(os.path.dirname(os.path.abspath(__file__)), 'native', 'recurrent_solo_check')


@pytest.fixture(scope='module')
def slayer():
    import lava_dl_amd.slayer as s
    return s


# 16 and 17 samples; whole and partial tiles of 16 neurons; 8 steps (the fewest), 16 and 17; 33 samples of 2048 neurons
# and 129 of 516 take two sample tiles per workgroup
@pytest.mark.parametrize('n,c,t', [(16, 256, 8), (17, 260, 16), (1, 1028, 17), (5, 2036, 33), (33, 2048, 9), (129, 516, 18)])
def test_layer_matches_the_oracle(slayer, n, c, t):
    R = slayer.utils.recurrent
    gen = torch.Generator().manual_seed(1000 * c + n)
    z = torch.randn(n, c, t, generator=gen) * 1.5
    g = torch.rand(n, c, t, generator=gen)
    neuron = base._neuron(slayer)
    syn = base._Dense(c, torch.Generator().manual_seed(5)).to(dev())
    with torch.no_grad():
        syn.weight.mul_(6.0 / c ** 0.5)
    syn.pre_hook_fx = neuron.quantize_8bit
    zg = z.to(dev()).requires_grad_()
    out = R.custom_recurrent(zg, neuron, syn)
    assert 0.01 < float(out.detach().mean()) < 0.9
    rec = neuron.quantize_8bit(syn.weight.detach().reshape(c, c)).cpu()
    d_i, d_v = neuron.current_decay.detach().round().cpu(), neuron.voltage_decay.detach().round().cpu()
    thr, zero = neuron.threshold + neuron.threshold_eps, torch.tensor([0.0])
    r_spk, r_vol, r_cs, r_vs = O.recurrent_cuba_fwd(z, rec, d_i, d_v, zero, zero, 4096, thr)
    assert_exact(out, r_spk, 'spikes')
    assert_exact(neuron.current_state, r_cs, 'carried current')
    assert_exact(neuron.voltage_state, r_vs, 'carried voltage')
    out.backward(g.to(dev()))
    r_gz, _ = O.recurrent_cuba_bwd(g, r_spk, r_vol, rec, thr, neuron.tau_rho * 100, neuron.scale_rho * 0.1)
    assert_rel(zg.grad, r_gz, 'grad z')


@pytest.mark.parametrize('c', [260, 2048])
def test_feedback_of_weights_off_the_grid(slayer, c):
    """Weights with all their 24 bits: with decays of 4096 and a scale of 2^22 the voltage of step t is the feedback of the
    spikes of step t - 1 to 2^-24, compared with a float64 sum.  Bound: the three parts hold every bit of a weight, the
    sum of c terms is rounded about c / 32 + 16 times to 2^-24 of its running value, which stays below the sum of the
    magnitudes: c / 32 * 2^-24 of that sum, at most 5e-6 of it (measured: 3e-8)."""
    from lava_dl_amd.slayer import _native as N
    n, t = 20, 8
    gen = torch.Generator().manual_seed(c)
    rec = (torch.randn(c, c, generator=gen) * 3 / c ** 0.5).to(dev())
    z = torch.randn(n, c, t, generator=gen).mul(4)
    z[..., 1:] *= 1e-3
    z = z.to(dev())
    spk, vol = torch.empty_like(z), torch.empty_like(z)
    last = [torch.empty(n, c, device=dev()) for _ in range(2)]
    full, zero = torch.full((1,), 4096.0, device=dev()), torch.zeros(1, device=dev())
    floats = N.lib().slayer_recurrent_steps_workspace(n, c, t, 0)
    ws = torch.empty(floats, device=dev())
    N.check(N.lib().slayer_cuba_recurrent_steps_fwd(
        N.ptr(spk), N.ptr(vol), N.ptr(last[0]), N.ptr(last[1]), N.ptr(z), N.ptr(rec), N.ptr(full), N.ptr(full), N.ptr(zero),
        N.ptr(zero), 0.5, 0, 1.0, 1 << 22, n, c, 1, 1, 1, 1, t, N.ptr(ws), floats, N.stream_handle()))
    assert 0.05 < float(spk.mean()) < 0.95
    s, w = spk.cpu().double(), rec.cpu().double()
    for step in range(1, t):
        want = z[..., step].cpu().double() + s[..., step - 1] @ w.t()
        magnitude = s[..., step - 1] @ w.abs().t() + z[..., step].cpu().double().abs()
        err = ((vol[..., step].cpu().double() - want).abs() / (magnitude + 1)).max()
        assert float(err) <= 5e-6, float(err)


# 2048 neurons fill 32 workgroups of 64, 68 leave most of the second one empty; 33 samples of 1300 neurons do not fit the
# form for weights that are bfloat16 numbers, [4 samples] x [64 neurons] a workgroup; 18 steps are two chunks
@pytest.mark.parametrize('n,c,t', [(5, 68, 18), (32, 2048, 9), (33, 1300, 20), (7, 260, 33)])
@pytest.mark.parametrize('weights,scale', [('grid', 1.0), ('grid', 1e-34), ('grid', 1e27), ('real', 1.0), ('real', 1e-34),
                                           ('large', 1.0)])
def test_gradients_of_weights_on_and_off_the_grid(slayer, n, c, t, weights, scale):
    """The input gradient against a float64 evaluation, with weights that are bfloat16 numbers and others, among them one
    too large for the first form; gradients near both ends of float32's range.  Both forms keep 24 bits of either factor and sum
    in float32.  Bound: a step's float32 factor is off by the rounding of its exponent (of magnitude 2), of exp and of three
    products, 6 x 2^-24, and what comes back through all t steps carries t of them: 4e-7 t of the largest magnitude.  The
    surrogate's scale of 0.04 keeps a gradient from leaving float32 on its way (0.9 times a step without the large weight)."""
    from lava_dl_amd.slayer import _native as N
    gen = torch.Generator().manual_seed(c + n)
    rec = torch.randn(c, c, generator=gen) * 3 / c ** 0.5
    if weights != 'real':
        rec = (rec * 32).round().clamp(-128, 127) / 32
        if weights == 'large':
            rec[c // 2, c // 3] = 1024.0
    v = torch.randn(n, c, t, generator=gen) * 0.02 + 1.25
    g = torch.randn(n, c, t, generator=gen) * scale
    d = [x.to(dev()) for x in (g, v, rec)]
    gz = torch.empty_like(d[0])
    floats = N.lib().slayer_recurrent_steps_workspace(n, c, t, 0)
    ws = torch.empty(floats, device=dev())
    N.check(N.lib().slayer_recurrent_steps_bwd(N.ptr(gz), N.ptr(d[0]), N.ptr(d[1]), None, N.ptr(d[2]), 1.25, 0.05, 0.04, 0,
                                               n, c, t, N.ptr(ws), floats, N.stream_handle()))
    factor = (0.04 / 2 / 0.05) * torch.exp(-(v.double() - 1.25).abs() / 0.05)
    want, carry = torch.empty_like(factor), torch.zeros(n, c, dtype=torch.float64)
    for step in reversed(range(t)):
        want[..., step] = factor[..., step] * (g[..., step].double() + carry)
        carry = want[..., step] @ rec.double()
    err = (gz.cpu().double() - want).abs()
    if scale == 1e27:
        assert bool((want.abs() > 4e25).any())
    assert bool((err <= 4e-7 * t * want.abs().amax()).all()), float(err.max() / want.abs().max())


@pytest.mark.parametrize('where', [0, 1])
def test_gradients_in_place(slayer, where):
    """grad_z over grad_spikes or over the voltage, with gradients so large that the layer is computed a second time."""
    from lava_dl_amd.slayer import _native as N
    n, c, t = 5, 68, 18
    gen = torch.Generator().manual_seed(8)
    rec = (torch.randn(c, c, generator=gen) * 12 / c ** 0.5).round().to(dev()) / 4
    v = (torch.randn(n, c, t, generator=gen) * 0.02 + 1.25).to(dev())
    g = (torch.randn(n, c, t, generator=gen) * 1e27).to(dev())
    floats = N.lib().slayer_recurrent_steps_workspace(n, c, t, 0)
    ws = torch.empty(floats, device=dev())

    def run(gz, g, v):
        N.check(N.lib().slayer_recurrent_steps_bwd(N.ptr(gz), N.ptr(g), N.ptr(v), None, N.ptr(rec), 1.25, 0.05, 0.04, 0, n, c, t,
                                                   N.ptr(ws), floats, N.stream_handle()))
        return gz
    want = run(torch.empty_like(g), g, v)
    ins = [g.clone(), v.clone()]
    assert float(want.abs().max()) > 1e26
    assert_rel(run(ins[where], *ins), want.cpu(), 'grad z in place')


# 68 and 260 neurons leave twelve columns of a tile of 16 and sixty of a tile of 64 empty, in either form of the kernel
@pytest.mark.parametrize('c', [68, 260])
@pytest.mark.parametrize('weights', ['grid', 'real'])
@pytest.mark.parametrize('bad', [float('inf'), float('-inf'), float('nan')])
def test_gradients_that_are_not_finite(slayer, c, weights, bad):
    """Positive weights: an infinite gradient of one neuron leaves every earlier one of its sample infinite and of its sign, as in the
    float64 loop; a NaN makes them NaN; the other samples are untouched (bound as above)."""
    from lava_dl_amd.slayer import _native as N
    n, t = 5, 18
    gen = torch.Generator().manual_seed(c)
    rec = torch.rand(c, c, generator=gen) + 0.25
    if weights == 'grid':
        rec = (rec * 32).round() / 32
    rec /= 256
    v = torch.randn(n, c, t, generator=gen) * 0.02 + 1.25
    g = torch.randn(n, c, t, generator=gen)
    g[1, 3, t - 2] = bad
    d = [x.to(dev()) for x in (g, v, rec)]
    gz = torch.empty_like(d[0])
    floats = N.lib().slayer_recurrent_steps_workspace(n, c, t, 0)
    ws = torch.empty(floats, device=dev())
    N.check(N.lib().slayer_recurrent_steps_bwd(N.ptr(gz), N.ptr(d[0]), N.ptr(d[1]), None, N.ptr(d[2]), 1.25, 0.05, 0.04, 0,
                                               n, c, t, N.ptr(ws), floats, N.stream_handle()))
    factor = (0.04 / 2 / 0.05) * torch.exp(-(v.double() - 1.25).abs() / 0.05)
    want, carry = torch.empty_like(factor), torch.zeros(n, c, dtype=torch.float64)
    for step in reversed(range(t)):
        want[..., step] = factor[..., step] * (g[..., step].double() + carry)
        carry = want[..., step] @ rec.double()
    got = gz.cpu().double()
    assert not torch.isfinite(want[1, :, :t - 2]).any() and torch.isfinite(want).sum() == want.numel() - c * (t - 2) - 1
    finite = torch.isfinite(want)
    assert torch.equal(got[~finite].nan_to_num(5.0, 6.0, 7.0), want[~finite].nan_to_num(5.0, 6.0, 7.0))
    assert bool(((got - want)[finite].abs() <= 4e-7 * t * want[finite].abs().amax()).all())


def test_weights_that_are_not_finite(slayer, monkeypatch):
    """An infinite weight times a silent neuron is a NaN, and so is a NaN weight times any: what the two receiving neurons
    do is lost, the other neurons' feedback is untouched."""
    from lava_dl_amd.slayer import _native as N
    monkeypatch.setattr(N, '_range_policy', 'ignore')              # an infinite feedback leaves a state at its limit
    R = slayer.utils.recurrent
    n, c, t = 3, 300, 12
    gen = torch.Generator().manual_seed(3)
    z = (torch.randn(n, c, t, generator=gen) * 1.5).to(dev())
    weight = torch.round(torch.randn(c, c, generator=gen) * 12) / 64
    weight[:, 5] = weight[:, 9] = 0                                # what neurons 5 and 9 do reaches nobody
    results = []
    for bad in (0.0, float('inf'), float('nan')):
        neuron = base._neuron(slayer)
        weight[5, 7] = weight[9, 11] = bad
        with torch.no_grad():
            results.append(R._FusedRecurrent.apply(z, neuron, weight.to(dev())))
    assert 0.01 < float(results[0].mean()) < 0.9
    rows = [i for i in range(c) if i not in (5, 9)]
    for out in results[1:]:
        assert torch.equal(out[:, rows], results[0][:, rows])
        assert not torch.equal(out, results[0])
    torch.cuda.synchronize()
    N.clear_range_flag()


def test_workgroups_that_give_up_waiting():
    if not os.path.exists(BINARY):
        pytest.skip('tests/native/recurrent_solo_check has not been built (python -c "import __graft_entry__ as g; g.build()")')
    run = subprocess.run([BINARY], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout + run.stderr
    assert 'solo kernels agree' in run.stdout


def _layer(slayer, n, c, t, seed):
    gen = torch.Generator().manual_seed(seed)
    neuron = base._neuron(slayer)
    syn = base._Dense(c, gen).to(dev())
    with torch.no_grad():
        syn.weight.mul_(6.0 / c ** 0.5)
    syn.pre_hook_fx = neuron.quantize_8bit
    z = (torch.randn(n, c, t, generator=gen) * 1.5).to(dev()).requires_grad_()
    return neuron, syn, z, torch.rand(n, c, t, generator=gen).to(dev())


def _run_layer(slayer, neuron, syn, z, g):
    out = slayer.utils.recurrent.custom_recurrent(z, neuron, syn)
    grads = torch.autograd.grad(out, (z, syn.weight), g)
    return (out.detach(), neuron.current_state, neuron.voltage_state) + grads


def test_layers_on_two_streams_from_two_threads(slayer):
    """Both fill the chip, so they cannot run side by side: each gives what it gives alone."""
    sizes = [(32, 2048, 24), (40, 1028, 33)]
    wants = [_run_layer(slayer, *_layer(slayer, *size, 3)) for size in sizes]
    rounds = 4
    layers = [[_layer(slayer, *size, 3) for _ in range(rounds)] for size in sizes]
    torch.cuda.synchronize()
    results, errors = [[], []], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for layer in layers[i]:
                    results[i].append(_run_layer(slayer, *layer))
                torch.cuda.current_stream().synchronize()
        except Exception as e:                                     # shown by the main thread
            errors.append(e)
    threads = [threading.Thread(target=work, args=(i,)) for i in range(2)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    assert not errors, errors
    for got, want in zip(results, wants):
        assert len(got) == rounds and 0.01 < float(want[0].mean()) < 0.9
        for r in got:
            for k, what in enumerate(('spikes', 'current', 'voltage')):
                assert torch.equal(r[k], want[k]), what
            assert_rel(r[3], want[3].cpu(), 'grad z')
            assert_rel(r[4], want[4].cpu(), 'grad weight')


CHILD = """
import sys
import torch
import lava_dl_amd.slayer as slayer
from tests import test_gpu_recurrent_grid as T
torch.save([x.cpu() for x in T._run_layer(slayer, *T._layer(slayer, 5, 260, 20, 4))], sys.argv[1])
"""


def test_layer_in_a_process_beside_another(slayer, tmp_path):
    """The runtime grants cooperative launches to one process at a time (here this one): the other's layer takes a launch per
    step where it is refused, with the same spikes (quantised weights) and gradients."""
    want = _run_layer(slayer, *_layer(slayer, 5, 260, 20, 4))
    torch.cuda.synchronize()
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    path = str(tmp_path / 'child.pt')
    run = subprocess.run([sys.executable, '-c', CHILD, path], cwd=root, env=dict(os.environ, PYTHONPATH=root),
                         capture_output=True, text=True, timeout=100)
    assert run.returncode == 0, run.stdout + run.stderr
    got = torch.load(path, weights_only=True)
    for k, what in enumerate(('spikes', 'current', 'voltage')):
        assert torch.equal(got[k], want[k].cpu()), what
    assert_rel(got[3], want[3].cpu(), 'grad z')
    assert_rel(got[4], want[4].cpu(), 'grad weight')
