"""The convolution kernels that run on the bfloat16 matrix instruction with operands split into three parts: spikes
(exact as they are), spikes with a few values in between that are not bfloat16 numbers, and real-valued inputs, against
float64; and inputs and gradients that are not finite, which give what IEEE arithmetic on the same sums gives.

Bar: 1e-5 of the sum of the magnitudes of an element's terms, as for the float32 kernels: what a split product leaves
out is below 2^-26 of it, and a float32 sum of n terms in one chain is within n * 2^-24 of their magnitudes (chains
here hold at most a few thousand)."""
import pytest
import torch
import torch.nn.functional as F

from tests.util import assert_sum, dev

pytestmark = pytest.mark.gpu

# (batch, Ci, H, W, T), Co, kernel, stride, padding, dilation
CASES = [
    ((1, 1, 3, 3, 4), 2, (1, 3), (1, 1), (0, 1), (1, 1)),
    ((2, 5, 6, 5, 31), 17, (3, 3), (1, 1), (1, 1), (1, 1)),          # 15 pairs: one tile
    ((1, 6, 5, 7, 33), 16, (3, 3), (1, 1), (0, 0), (1, 1)),          # 18 pairs: two tiles
    ((2, 11, 7, 4, 64), 33, (3, 3), (2, 1), (1, 1), (1, 1)),         # 33 pairs: two passes
    ((1, 16, 6, 9, 65), 48, (3, 3), (1, 1), (1, 1), (2, 1)),
    ((1, 4, 8, 8, 301), 8, (5, 5), (1, 1), (2, 2), (1, 1)),
    ((1, 13, 7, 6, 36), 20, (5, 5), (1, 1), (2, 2), (1, 1)),         # 65 pairs
    ((1, 32, 5, 6, 36), 8, (5, 5), (1, 1), (2, 2), (1, 1)),          # 160 pairs: the parts of the weights fill 75 KB
    ((2, 16, 5, 5, 44), 8, (2, 2), (1, 1), (1, 1), (1, 1)),
    ((1, 32, 4, 6, 300), 64, (3, 3), (1, 1), (1, 1), (1, 1)),
]


def _run(x, w, g, stride, padding, dilation):
    import lava_dl_amd.slayer as slayer
    xg, wg = x.to(dev()).requires_grad_(), w.to(dev()).requires_grad_()
    y = slayer.synapse.conv_synapse(xg, wg, stride, padding, dilation)
    y.backward(g.to(dev()))
    return y.detach(), xg.grad, wg.grad


def _reference(x, w, g, stride, padding, dilation):
    x, w = x.double().requires_grad_(), w.double().requires_grad_()
    y = F.conv3d(x, w, None, stride + (1,), padding + (0,), dilation + (1,))
    y.backward(g.double())
    return y.detach(), x.grad, w.grad


@pytest.mark.parametrize('case', CASES, ids=str)
@pytest.mark.parametrize('kind', ['spikes', 'mixed', 'real'])
@pytest.mark.parametrize('quantised', [True, False])
def test_split_products_match_float64(case, kind, quantised):
    shape, co, kernel, *geometry = case
    gen = torch.Generator().manual_seed(sum(shape) + co)
    x = (torch.rand(shape, generator=gen) < 0.2).float()
    if kind == 'mixed':                                              # some visits see more than bfloat16 holds
        x += (torch.rand(shape, generator=gen) < 0.002) * torch.randn(shape, generator=gen)
    elif kind == 'real':
        x = torch.randn(shape, generator=gen)
    w = torch.randn((co, shape[1]) + kernel + (1,), generator=gen)
    if quantised:
        w = (w * 32).round().clamp(-128, 127) / 64
    y_shape = F.conv3d(x[..., :1], w, None, *(v + (i,) for v, i in zip(geometry, (1, 0, 1)))).shape[:-1] + shape[-1:]
    g = torch.randn(y_shape, generator=gen)
    got, want = _run(x, w, g, *geometry), _reference(x, w, g, *geometry)
    size = _reference(x.abs(), w.abs(), g.abs(), *geometry)
    for name, a, b, m in zip(('output', 'grad input', 'grad weight'), got, want, size):
        assert_sum(a, b, m + 1e-30, f'{kind} {name}')
    if quantised and kind == 'spikes':
        assert torch.equal(got[0].cpu().double(), want[0]), 'sums of spikes times quantised weights are exact'


@pytest.mark.parametrize('where', ['input', 'gradient'])
@pytest.mark.parametrize('value', [float('inf'), float('-inf'), float('nan'), 3.4e38])
def test_values_that_are_not_finite_or_overflow_a_part(where, value):
    gen = torch.Generator().manual_seed(11)
    x = torch.randint(1, 3, (2, 8, 6, 6, 40), generator=gen).float()
    w = torch.randint(1, 5, (16, 8, 3, 3, 1), generator=gen).float() / 64
    g = torch.rand(2, 16, 4, 4, 40, generator=gen) + 0.5
    # an input pixel that every tap of its row meets inside the output
    {'input': x[0, 0, 2, 2], 'gradient': g[0, 0, 1, 1]}[where].view(-1)[0] = value
    geometry = (1, 1), (0, 0), (1, 1)
    got, want = _run(x, w, g, *geometry), _reference(x, w, g, *geometry)
    for name, a, b in zip(('output', 'grad input', 'grad weight'), got, want):
        a, b = a.cpu(), b.float()                                    # what overflows float32 is infinite in float32
        assert torch.equal(a.isnan(), b.isnan()), name
        assert torch.equal(a.isinf(), b.isinf()) and torch.equal(a[a.isinf()], b[b.isinf()]), name
        ok = a.isfinite()
        assert float((a[ok] - b[ok]).abs().max()) <= 1e-5 * float(b[ok].abs().max()), name


def _padded_sums(x, w, g, stride, padding, dilation):
    """The three passes in float64 as sums over every tap, taps outside the image as products with zero: what the float32
    matrix instruction gives for operands that are not finite (0 * inf among them).  Unit stride and dilation, or none."""
    x, w, g = x.double(), w.double()[..., 0], g.double()

    def correlate(a, b, pad):                                        # a [N, Ci, H, W, T], b [Co, Ci, kh, kw]
        kh, kw = b.shape[2:]
        a = F.pad(a, (0, 0, pad[1], pad[1], pad[0], pad[0])).unfold(2, kh, 1).unfold(3, kw, 1)
        return torch.stack([(a * b[co][None, :, None, None, None]).sum((1, 5, 6)) for co in range(b.shape[0])], 1)
    kh, kw = w.shape[2:]
    y = correlate(x, w, padding)
    gx = correlate(g, w.flip(2, 3).transpose(0, 1), (kh - 1 - padding[0], kw - 1 - padding[1]))
    taps = F.pad(x, (0, 0, padding[1], padding[1], padding[0], padding[0])).unfold(2, kh, 1).unfold(3, kw, 1)
    gw = torch.stack([(taps * g[:, co, None, ..., None, None]).sum((0, 2, 3, 4)) for co in range(w.shape[0])])
    return y, gx, gw[..., None]


# Layers whose two directions fill the split form's groups of 32 pairs (24, 26; 24, 51; 48, 24; 25, 50 pairs), rows that end inside
# a quad among them, and one with the float32 form forward (12 pairs).  It takes launches of 1024 waves and more, here
# by a batch that is zero but for one sample.
SPLIT = [((1, 12, 5, 5, 36), 13, (2, 2)), ((1, 8, 6, 5, 37), 17, (3, 3)), ((1, 16, 5, 6, 70), 8, (3, 3)), ((1, 5, 6, 6, 33), 10, (5, 5)),
         ((1, 4, 5, 6, 36), 16, (3, 3))]


def _run_in_large_batch(x, w, g, stride, padding, dilation):
    waves = g.shape[2] * ((g.shape[-1] + 63) // 64)
    batch = 1024 // min(waves, x.shape[2] * ((x.shape[-1] + 63) // 64)) + 1
    at = batch // 2

    def embed(v):
        return torch.zeros((batch,) + v.shape[1:]).index_copy(0, torch.tensor([at]), v)
    y, gx, gw = _run(embed(x), w, embed(g), stride, padding, dilation)
    return y[at:at + 1], gx[at:at + 1], gw


def _operands(case, kind='real'):
    shape, co, kernel = case
    gen = torch.Generator().manual_seed(sum(shape) + co)
    x = torch.randn(shape, generator=gen)
    if kind == 'spikes':
        x = (torch.rand(shape, generator=gen) < 0.5).float()
    elif kind == 'mixed':
        x = (x > 1).float() + (torch.rand(shape, generator=gen) < 0.002) * x
    w = torch.randn((co, shape[1]) + kernel + (1,), generator=gen)
    pad = (kernel[0] // 2, kernel[1] // 2)
    g = torch.randn((shape[0], co) + tuple(s + 2 * p - k + 1 for s, p, k in zip(shape[2:4], pad, kernel)) + shape[4:],
                    generator=gen)
    return x, w, g, ((1, 1), pad, (1, 1))


# ... and the ends of a group of 32 pairs, several blocks of channels, an image row cut into pieces
@pytest.mark.parametrize('case', SPLIT + [((1, 31, 4, 20, 64), 33, (1, 3)), ((1, 32, 4, 5, 65), 32, (1, 2)), ((1, 24, 5, 33, 301), 63, (1, 5)),
                                          ((1, 6, 6, 6, 40), 12, (5, 5))],
                         ids=str)
@pytest.mark.parametrize('kind', ['spikes', 'mixed', 'real'])
@pytest.mark.parametrize('quantised', [True, False])
def test_split_form_of_large_launches(case, kind, quantised):
    x, w, g, geometry = _operands(case, kind)
    if quantised:
        w = (w * 32).round().clamp(-128, 127) / 64
    got, want = _run_in_large_batch(x, w, g, *geometry), _reference(x, w, g, *geometry)
    size = _reference(x.abs(), w.abs(), g.abs(), *geometry)
    for name, a, b, m in zip(('output', 'grad input', 'grad weight'), got, want, size):
        assert_sum(a, b, m + 1e-30, f'{kind} {name}')
    if quantised and kind == 'spikes':
        assert torch.equal(got[0].cpu().double(), want[0]), 'sums of spikes times quantised weights are exact'


@pytest.mark.parametrize('case', SPLIT, ids=str)
@pytest.mark.parametrize('kind', ['spikes', 'real'])
@pytest.mark.parametrize('where', ['input', 'gradient', 'weight'])
@pytest.mark.parametrize('value', [float('inf'), float('-inf'), float('nan'), 3.4e38])
def test_not_finite_times_operands_of_several_parts(case, kind, where, value):
    """The parts of a split operand are zero or of either sign: inf times each of them is not inf times their sum."""
    x, w, g, geometry = _operands(case, kind)
    # a pixel whose taps all lie inside the image: the weight gradient does not visit columns outside it
    {'input': x[0, 1, 2, 3, 5:], 'gradient': g[0, 3, 2, 2, 9:], 'weight': w[2, 1, 1, 0]}[where].view(-1)[0] = value
    got, want = _run_in_large_batch(x, w, g, *geometry), _padded_sums(x, w, g, *geometry)
    size = _padded_sums(x.abs(), w.abs(), g.abs(), *geometry)
    for name, a, b, m in zip(('output', 'grad input', 'grad weight'), got, want, size):
        a, b32 = a.cpu(), b.float()                                  # what overflows float32 is infinite in float32
        assert torch.equal(a.isnan(), b32.isnan()), name
        assert torch.equal(a.isinf(), b32.isinf()) and torch.equal(a[a.isinf()], b32[b32.isinf()]), name
        ok = a.isfinite()
        assert bool(((a.double() - b).abs()[ok] <= 1e-5 * m[ok] + 1e-30).all()), name


@pytest.mark.parametrize('case', SPLIT[:4], ids=str)
@pytest.mark.parametrize('where', ['input', 'gradient', 'weight', 'input and weight', 'input and gradient'])
@pytest.mark.parametrize('scale', [2.0 ** -126, 1e-36, 1e-33, 1e-30, 1e-20, 1e20, 1e33])
def test_magnitudes_far_from_one(case, where, scale):
    """A value keeps its 24 bits whatever its magnitude (a part of a split operand must not fall below the smallest normal
    number), down to products and sums of float32's smallest numbers: the bar adds half a unit of these per term of a sum.
    Sums whose terms leave float32's range are infinite or NaN, by their order, and not looked at."""
    x, w, g, geometry = _operands(case)
    if 'input' in where:
        x *= scale
    if 'gradient' in where:
        g *= scale
    if 'weight' in where:
        w *= scale
    got, want = _run_in_large_batch(x, w, g, *geometry), _reference(x, w, g, *geometry)
    size = _reference(x.abs(), w.abs(), g.abs(), *geometry)
    taps = w.shape[2] * w.shape[3]
    terms = (x.shape[1] * taps, w.shape[0] * taps, g.numel() // w.shape[0])
    for name, n, a, b, m in zip(('output', 'grad input', 'grad weight'), terms, got, want, size):
        a, inside = a.cpu().double(), m < 2.0 ** 127                 # no order of the sum leaves the range
        assert bool(((a - b).abs() <= 1e-5 * m + n * 2.0 ** -150)[inside].all()), name


def test_filters_that_only_the_split_form_holds():
    """500 (channel, kernel row) pairs of two taps: too many for the float32 row form's 64 KB of LDS at any launch size."""
    from lava_dl_amd.slayer.synapse import layer
    gen = torch.Generator().manual_seed(3)
    x, w = torch.randn(1, 250, 2, 5, 8, generator=gen), torch.randn(250, 2, 4, 4, 1, generator=gen)
    y = layer._launch_input_grad(x.to(dev()), w[..., 0].transpose(0, 1).contiguous().to(dev()), (1, 2, 4, 10, 8), (2, 2), (1, 1), (1, 1))
    assert y is not None
    args = None, (2, 2, 1), (1, 1, 0)
    assert_sum(y, F.conv_transpose3d(x.double(), w.double(), *args), F.conv_transpose3d(x.double().abs(), w.double().abs(), *args), 'output')


@pytest.mark.parametrize('kind', ['graded', 'real'])
def test_products_of_the_lower_parts_do_not_round_the_sum(kind):
    """32 -> 64 channels, both operands of three parts: forward nine groups of 32 terms an output, the input gradient eighteen.
    A sum is rounded twice for each (the products of the lower parts, added up on their own, and the product of the first
    parts), each time by at most 2^-23 of it and its binade, evenly spread: a relative error of sqrt(2 groups / 2) *
    2^-23 / sqrt(3) * 0.72 in the 2-norm, half of the roundings weighing (the sum grows like a random walk).  With all six
    products into the one sum it was 2.1e-7 to 2.6e-7 and 3.7e-7, on the float32 instruction 1.2e-7 (graded), 2.9e-7 and 4.2e-7."""
    gen = torch.Generator().manual_seed(2)
    x = torch.randn(1, 32, 8, 8, 40, generator=gen)
    if kind == 'graded':
        x = (x > 1) * x
    w, g = torch.randn(64, 32, 3, 3, 1, generator=gen), torch.randn(1, 64, 8, 8, 40, generator=gen)
    geometry = (1, 1), (1, 1), (1, 1)
    got, want = _run_in_large_batch(x, w, g, *geometry), _reference(x, w, g, *geometry)
    for name, groups, a, b in zip(('output', 'grad input'), (9, 18), got, want):
        error = float((a.cpu().double() - b).norm() / b.norm())
        assert error <= groups ** 0.5 * 2.0 ** -23 / 3 ** 0.5 * 0.72, (name, error)


@pytest.mark.parametrize('batch', [204, 205])
@pytest.mark.parametrize('ci,kernel', [(43, 3), (85, 3), (86, 3), (32, 5), (33, 5)])
def test_workgroups_of_either_size(batch, ci, kernel):
    """Weights of which two workgroups share the LDS of a compute unit, and of which one fills it: four waves each, or eight
    from 1025 waves on (five rows an image, so the last workgroup of a sample has waves without work)."""
    from lava_dl_amd.slayer.synapse import layer
    gen = torch.Generator().manual_seed(ci + batch)
    x, w = torch.randn(batch, ci, 5, 8, 8, generator=gen), torch.randn(3, ci, kernel, kernel, 1, generator=gen)
    pad = kernel // 2
    y = layer._launch(x.to(dev()), w[..., 0].contiguous().to(dev()), (1, 1), (pad, pad), (1, 1))
    args = None, 1, (pad, pad, 0)
    assert_sum(y, F.conv3d(x.double(), w.double(), *args), F.conv3d(x.double().abs(), w.double().abs(), *args), 'output')
