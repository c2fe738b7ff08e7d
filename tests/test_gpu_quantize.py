"""The weight quantiser's one launch (csrc/quantize.hip) against the operators it stands for, bit for bit."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu


@pytest.fixture(scope='module')
def slayer():
    import lava_dl_amd.slayer as s
    return s


def _chain(slayer, x, step, lo, hi, scale):
    q = slayer.utils.quantize(x, step=step).clamp(lo, hi)
    return q if scale == 1 else q * scale


# powers of two and scales whose step and reciprocal are rounded; ties, both limits, infinities, NaN, negative zero
@pytest.mark.parametrize('scale', [64, 1, 50, 3.7])
@pytest.mark.parametrize('descale', [False, True])
@pytest.mark.parametrize('shape', [(1,), (257,), (16, 8, 3, 3, 1)])
def test_quantizer_is_the_chain_of_operators(slayer, scale, descale, shape):
    gen = torch.Generator().manual_seed(int(scale * 10) + len(shape))
    x = torch.randn(shape, generator=gen) * 3 * 64 / scale
    flat = x.view(-1)
    special = [0.5 * 2 / scale, 1.5 * 2 / scale, -0.3 / scale, 254 / scale, 255 / scale, 256 / scale, -256 / scale, -257 / scale,
               float('inf'), float('-inf'), float('nan'), 1e-40]
    flat[:min(len(special), flat.numel())] = torch.tensor(special)[:flat.numel()]
    g = torch.randn(shape, generator=gen).to(dev())
    results = []
    for fused in (True, False):
        xg = x.to(dev()).requires_grad_()
        args = (xg, 2 / scale, -256 / scale, 254 / scale, scale if descale else 1)
        out = slayer.utils.limit(*args) if fused else _chain(slayer, *args)
        grad, = torch.autograd.grad(out, xg, g)
        with torch.no_grad():
            plain = slayer.utils.limit(*args) if fused else _chain(slayer, *args)
        results.append([t.detach().cpu().view(torch.int32) for t in (out, grad, plain)])
    for a, b in zip(*results):
        assert torch.equal(a, b)


def test_calls_that_keep_the_operators(slayer):
    """Layouts, types and devices the kernel does not take, and users of the single operations."""
    limit = slayer.utils.limit
    gen = torch.Generator().manual_seed(1)
    w = torch.randn(6, 10, generator=gen).to(dev())
    args = (2 / 64, -4.0, 254 / 64)
    want = _chain(slayer, w, *args, 1)
    assert torch.equal(limit(w.t(), *args), want.t())
    assert torch.equal(limit(w.cpu(), *args), want.cpu())
    assert limit(w.double(), *args).dtype == torch.float64
    assert limit(w[:0], *args).shape == (0, 10)
    assert torch.equal(torch.func.vmap(lambda r: limit(r, *args))(w), want)
    assert torch.equal(torch.jit.trace(lambda r: limit(r, *args), (w,))(w + 1), _chain(slayer, w + 1, *args, 1))
    with torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(w, torch.full_like(w, 0.75))
        primal, tangent = torch.autograd.forward_ad.unpack_dual(limit(dual, *args))
        want_tangent = torch.autograd.forward_ad.unpack_dual(_chain(slayer, dual, *args, 1)).tangent
        assert torch.equal(primal, want)
        assert (tangent is None) == (want_tangent is None) and (tangent is None or torch.equal(tangent, want_tangent))
    x = w.clone().requires_grad_()
    grad, = torch.autograd.grad((limit(x, *args) ** 2).sum(), x, create_graph=True)
    second, = torch.autograd.grad(grad.sum(), x)
    y = w.clone().requires_grad_()
    grad_y, = torch.autograd.grad((_chain(slayer, y, *args, 1) ** 2).sum(), y, create_graph=True)
    second_y, = torch.autograd.grad(grad_y.sum(), y)
    assert torch.equal(grad, grad_y) and torch.equal(second, second_y)


def test_more_weights_than_a_launch_has_threads(slayer):
    """2^32 + 300 entries through the C interface; looked at near both ends and in the middle, where a thread's second entry lies."""
    from lava_dl_amd.slayer import _native as N
    n, scale = (1 << 32) + 300, 64.0
    gen = torch.Generator().manual_seed(6)
    parts = [slice(0, 600), slice((1 << 31) - 300, (1 << 31) + 300), slice(n - 600, n)]
    x, out = (torch.empty(n, device=dev()) for _ in range(2))
    inside = torch.empty(n, dtype=torch.uint8, device=dev())
    for p in parts:
        x[p] = (torch.randn(600, generator=gen) * 3).to(dev())
    N.check(N.lib().slayer_quantize(N.ptr(out), N.ptr(inside), N.ptr(x), 2 / 64, -4.0, 254 / 64, scale, n, N.stream_handle()))
    wants = [_chain(slayer, x[p], 2 / 64, -4.0, 254 / 64, scale) for p in parts]
    for p, want in zip(parts, wants):
        assert torch.equal(out[p], want)
    N.check(N.lib().slayer_quantize_bwd(N.ptr(out), N.ptr(x), N.ptr(inside), scale, n, N.stream_handle()))
    for p in parts:
        q = slayer.utils.quantize(x[p], step=2 / 64)
        assert torch.equal(out[p], torch.where((q >= -4.0) & (q <= 254 / 64), x[p] * scale, 0.0))


def test_a_recorded_graph_holds_the_operators(slayer):
    from torch.fx.experimental.proxy_tensor import make_fx
    limit = slayer.utils.limit
    w = (torch.randn(6, 10, generator=torch.Generator().manual_seed(5)) * 3).to(dev())
    graph = make_fx(lambda r: limit(r, 2 / 64, -4.0, 254 / 64))(w)
    assert torch.equal(graph(w * 0.7), _chain(slayer, w * 0.7, 2 / 64, -4.0, 254 / 64, 1))


@pytest.mark.parametrize('form', ['is_grads_batched', 'vmap'])
def test_batched_gradients(slayer, form):
    """Gradients without memory of their own take the operators; what each entry of the batch gives alone is the kernel's."""
    gen = torch.Generator().manual_seed(4)
    w = (torch.randn(6, 10, generator=gen) * 3).to(dev()).requires_grad_()
    g = torch.randn(5, 6, 10, generator=gen).to(dev())
    out = slayer.utils.limit(w, 2 / 64, -4.0, 254 / 64, 64)
    single = torch.stack([torch.autograd.grad(out, w, r, retain_graph=True)[0] for r in g])
    if form == 'vmap':
        batched = torch.func.vmap(lambda r: torch.autograd.grad(out, w, r, retain_graph=True)[0])(g)
    else:
        batched, = torch.autograd.grad(out, w, g, is_grads_batched=True, retain_graph=True)
    assert torch.equal(single, batched)


def test_rotation_limits_are_the_chain_of_operators(slayer):
    """ResonatorNeuron.clamp in one launch: gains on either side of the limit, negative and vanishing parts, NaN, infinity."""
    gen = torch.Generator().manual_seed(3)
    neuron = slayer.neuron.rf.Neuron(threshold=1.0, period=[20, 200], decay=[0.01, 0.9], shared_param=False).to(dev())
    s, c = torch.randn(600, generator=gen) * 4000, torch.randn(600, generator=gen) * 4000
    s[:6] = torch.tensor([0.0, float('nan'), float('inf'), 4095.0, 1e-30, 3e38])
    c[:6] = torch.tensor([0.0, 1.0, 2.0, 0.0, -1e-30, 3e38])
    results = []
    for fused in (True, False):
        neuron.sin_decay.data, neuron.cos_decay.data = s.clone().to(dev()), c.clone().to(dev())
        if fused:
            neuron.clamp()
        else:
            with torch.no_grad():
                gain = torch.sqrt(neuron.sin_decay ** 2 + neuron.cos_decay ** 2)
                ratio = gain.clamp(0, 4095) / gain
                neuron.sin_decay.data.mul_(ratio).clamp_(1)
                neuron.cos_decay.data.mul_(ratio).clamp_(0)
        results.append([p.data.cpu().clone() for p in (neuron.sin_decay, neuron.cos_decay)])
    for a, b in zip(*results):
        assert torch.equal(torch.isnan(a), torch.isnan(b))
        ok = ~torch.isnan(a)
        assert torch.equal(a[ok].view(torch.int32), b[ok].view(torch.int32))
