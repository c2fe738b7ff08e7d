"""The walking kernels of the convolution synapse (csrc/synapse_walk.hip, synapse_wgrad_walk.hip) where they can go wrong: every number of taps along the
walk, strides along either axis, pixels that share a position, two blocks of channels, rows cut into pieces, residue classes of
a transposed convolution, and pixels whose steps are not whole quads.  The operands are small integers, so every sum is exact
in float32 whatever its order and the results equal float64's, bit for bit.

The layers are small, and for such the library takes few pixels to a position, one block of channels and many pieces: the tests
below that give the cut themselves take every layer through the others too."""
import pytest
import torch
import torch.nn.functional as F

from tests.util import dev

pytestmark = pytest.mark.gpu

# (batch, Ci, H, W, T), Co, kernel, stride, padding, dilation
FORMS = [
    ((1, 1, 1, 1, 4), 1, (1, 2), (1, 1), (0, 1), (1, 1)),
    ((2, 3, 4, 5, 5), 2, (3, 3), (1, 1), (1, 1), (1, 1)),            # five pixels: with two or three to a position some are alone
    ((1, 2, 7, 9, 6), 1, (3, 3), (1, 1), (1, 1), (1, 1)),
    ((1, 8, 33, 6, 7), 8, (3, 3), (1, 1), (1, 1), (1, 1)),
    ((1, 8, 6, 33, 11), 3, (5, 5), (1, 1), (2, 2), (1, 1)),
    ((1, 5, 6, 7, 64), 17, (3, 3), (1, 1), (0, 2), (1, 1)),          # two blocks of channels, the second of one channel
    ((1, 32, 5, 5, 300), 64, (3, 3), (1, 1), (1, 1), (1, 1)),
    ((300, 17, 4, 4, 9), 40, (2, 2), (1, 1), (1, 1), (1, 1)),        # many samples
    ((1, 4, 9, 8, 13), 6, (4, 4), (1, 1), (1, 2), (1, 1)),           # four taps
    ((2, 4, 9, 10, 10), 8, (3, 3), (2, 2), (1, 1), (1, 1)),          # rows of a step outside the image on one side
    ((2, 3, 10, 9, 50), 4, (5, 5), (2, 3), (2, 1), (1, 1)),
    ((1, 2, 11, 12, 8), 5, (4, 3), (3, 2), (0, 0), (1, 1)),
    ((1, 3, 8, 9, 20), 16, (3, 3), (1, 1), (2, 2), (1, 2)),          # taps along the line that lie apart
    ((1, 3, 9, 8, 20), 16, (3, 3), (1, 1), (2, 2), (2, 1)),          # walked along the other axis
    ((1, 3, 9, 8, 20), 4, (3, 3), (1, 1), (2, 2), (2, 2)),           # not one that it takes
    ((1, 3, 9, 9, 20), 4, (7, 7), (1, 1), (3, 3), (1, 1)),
    ((1, 3, 3, 12, 21), 4, (1, 5), (1, 1), (0, 2), (1, 1)),
    ((1, 20, 4, 5, 31), 20, (1, 1), (1, 1), (0, 0), (1, 1)),
    ((2, 4, 9, 7, 17), 4, (2, 2), (3, 3), (0, 0), (1, 1)),           # transposed: classes without taps
    ((2, 3, 36, 5, 9), 4, (33, 3), (1, 1), (2, 1), (1, 1)),          # more rows than a line has taps
]


def _integers(gen, shape, most):
    return torch.randint(-most, most + 1, shape, generator=gen).float()


@pytest.mark.parametrize('form', FORMS, ids=str)
@pytest.mark.parametrize('parts', [1, 3])
def test_integers_equal_float64(form, parts):
    """parts = 1: both operands are bfloat16 numbers; 3: neither is (up to 2^11 times 2^9, a few hundred terms: below 2^31,
    held exactly where a sum stays below 2^24, which few taps of sparse inputs do)."""
    import lava_dl_amd.slayer as slayer
    shape, co, kernel, stride, padding, dilation = form
    gen = torch.Generator().manual_seed(sum(shape) + co)
    x = _integers(gen, shape, 3 if parts == 1 else 1025)
    w = _integers(gen, (co, shape[1]) + kernel + (1,), 5 if parts == 1 else 517)
    if parts == 3:                                                   # at most 2^24 / (1025 * 517) = 31 terms of one sum
        x *= torch.rand(shape, generator=gen) < 0.5
        w *= torch.rand(w.shape, generator=gen) < min(1.0, 16 / (shape[1] * kernel[0] * kernel[1]))
        assert float((w != 0).sum((1, 2, 3, 4)).max()) <= 31
    cfg = (stride + (1,), padding + (0,), dilation + (1,))
    want = F.conv3d(x.double(), w.double(), None, *cfg)
    got = slayer.synapse.conv_synapse(x.to(dev()), w.to(dev()), stride, padding, dilation)
    assert torch.equal(got.cpu().double(), want), 'convolution'
    up = [(shape[2 + i] - 1) * stride[i] - 2 * padding[i] + dilation[i] * (kernel[i] - 1) + 1 for i in (0, 1)]
    if min(up) < 1:
        return
    wt = w.transpose(0, 1).contiguous()[:, :31]                      # [Ci, Co, ...]: sums over Ci
    if parts == 3:
        wt = wt * (torch.rand(wt.shape, generator=gen) < min(1.0, 16 / float((wt != 0).sum((0, 2, 3, 4)).max())))
        if float((wt != 0).sum((0, 2, 3, 4)).max()) > 31:
            return
    want = F.conv_transpose3d(x.double(), wt.double(), None, cfg[0], cfg[1], 0, 1, cfg[2])
    got = slayer.synapse.conv_transpose_synapse(x.to(dev()), wt.to(dev()), stride, padding, dilation)
    assert torch.equal(got.cpu().double(), want), 'transposed convolution'


@pytest.mark.parametrize('form', FORMS + [((1, 3, 33, 3, 12), 16, (3, 3), (1, 1), (1, 1), (1, 1)),          # rows in four pieces
                                          ((1, 2, 9, 4, 70), 4, (3, 3), (1, 1), (1, 1), (1, 1)),            # ... of two or three
                                          ((3, 2, 6, 5, 9), 20, (3, 3), (1, 1), (1, 1), (1, 1)),            # few sets, two blocks of channels
                                          ((1, 2, 12, 16, 40), 3, (2, 2), (1, 1), (0, 0), (1, 1)),
                                          ((330, 17, 4, 4, 9), 80, (2, 2), (1, 1), (0, 0), (1, 1)),         # a set of sums to a wave
                                          ((40, 8, 8, 8, 300), 16, (3, 3), (1, 1), (1, 1), (1, 1))], ids=str)   # whole rows
@pytest.mark.parametrize('split', ['neither', 'gradient', 'input'])
def test_weight_gradient_of_integers_equals_float64(form, split):
    """Up to 2^18 terms of at most 3 * 3, or at most 31 of an operand that takes several parts: below 2^24."""
    from lava_dl_amd.slayer.synapse import layer
    shape, co, kernel, stride, padding, dilation = form
    gen = torch.Generator().manual_seed(sum(shape) + co + 1)
    out = [(shape[2 + i] + 2 * padding[i] - dilation[i] * (kernel[i] - 1) - 1) // stride[i] + 1 for i in (0, 1)]
    x, g = _integers(gen, shape, 3), _integers(gen, (shape[0], co, *out, shape[4]), 3)
    if split != 'neither':
        big = g if split == 'gradient' else x
        keep = torch.rand(big.shape, generator=gen) < 16 / (big.numel() / big.shape[1])
        big.copy_(_integers(gen, big.shape, 60001) * keep)
        assert float((big != 0).sum((0, 2, 3, 4)).max()) <= 31       # 31 * 60001 * 3 < 2^24
    wd = torch.zeros((co, shape[1]) + kernel + (1,), dtype=torch.float64).requires_grad_()
    F.conv3d(x.double(), wd, None, stride + (1,), padding + (0,), dilation + (1,)).backward(g.double())
    got = layer._weight_gradient(x.to(dev()), wd.shape, g.to(dev()), stride, padding, dilation)
    assert torch.equal(got.cpu().double(), wd.grad)


@pytest.mark.parametrize('sets', [1, 5, 38])
def test_a_smaller_workspace_is_cut_to(sets):
    """[1,1,16,15,168] -> 32 channels, 2x2: tiles of 256 floats for `sets` sums of each block of 16 channels, beside 64 for the
    reduction.  At most 17 * 16 * 168 terms of 9."""
    from lava_dl_amd.slayer import _native as N
    gen = torch.Generator().manual_seed(sets)
    x, g = _integers(gen, (1, 1, 16, 15, 168), 3), _integers(gen, (1, 32, 17, 16, 168), 3)
    wd = torch.zeros((32, 1, 2, 2, 1), dtype=torch.float64).requires_grad_()
    F.conv3d(x.double(), wd, None, 1, (1, 1, 0)).backward(g.double())
    floats = (sets + 64) * 2 * 256 * 2
    assert floats < N.lib().slayer_conv_synapse_wgrad_workspace(1, 1, 32, 16, 15, 168, 2, 2, 1, 1, 1)
    x, g, workspace = x.to(dev()), g.to(dev()), torch.empty(floats, device=dev())
    got = torch.empty(32, 1, 2, 2, 1, device=dev())
    with N.device_guard(x.device):
        N.check(N.lib().slayer_conv_synapse_wgrad(N.ptr(got), N.ptr(g), N.ptr(x), 1, 1, 32, 16, 15, 168, 2, 2, 1, 1, 1, 1, 1, 1,
                                                  N.ptr(workspace), floats, N.stream_handle()))
    assert torch.equal(got.cpu().double(), wd.grad)


@pytest.mark.parametrize('value', [float('inf'), float('-inf'), float('nan')])
@pytest.mark.parametrize('form', [FORMS[i] for i in (1, 3, 9, 10, 11, 18)], ids=str)
def test_a_value_that_is_not_finite_reaches_the_outputs_whose_taps_meet_it_and_no_others(form, value):
    import lava_dl_amd.slayer as slayer
    shape, co, kernel, stride, padding, dilation = form
    gen = torch.Generator().manual_seed(5)
    x = torch.randint(1, 4, shape, generator=gen).float()
    x[0, 0, shape[2] // 2, shape[3] // 2, 1] = value
    cfg = (stride + (1,), padding + (0,), dilation + (1,))
    for transposed in (False, True):
        w = torch.randint(1, 5, ((shape[1], co) if transposed else (co, shape[1])) + kernel + (1,), generator=gen).float()
        op = slayer.synapse.conv_transpose_synapse if transposed else slayer.synapse.conv_synapse
        met = torch.zeros(shape).masked_fill_(~x.isfinite(), 1.0)
        if transposed:
            reach = F.conv_transpose3d(met, w, None, cfg[0], cfg[1], 0, 1, cfg[2]) > 0
            want = F.conv_transpose3d(torch.where(x.isfinite(), x, 0.0), w, None, cfg[0], cfg[1], 0, 1, cfg[2])
        else:
            reach = F.conv3d(met, w, None, *cfg) > 0
            want = F.conv3d(torch.where(x.isfinite(), x, 0.0), w, None, *cfg)
        got = op(x.to(dev()), w.to(dev()), stride, padding, dilation).cpu()
        want = torch.where(reach, torch.full_like(want, value), want)
        assert torch.equal(got.isnan(), want.isnan()) and torch.equal(got.nan_to_num(7.0), want.nan_to_num(7.0))


# (batch, Ci, H, W, T) -> Co, kernel, stride, padding, dilation: a launch per residue class, pixels together, classes of one tap
CLASSES = [((16, 4, 16, 16, 50), 1, (5, 5), (5, 5), (0, 0), (1, 1)),         # as many taps as the stride
           ((16, 4, 16, 16, 50), 1, (8, 8), (8, 8), (0, 0), (1, 1)),
           ((64, 4, 16, 16, 12), 1, (7, 7), (5, 5), (0, 0), (1, 1)),         # classes of one tap and of two
           ((64, 4, 16, 16, 12), 1, (3, 3), (2, 2), (1, 1), (2, 1)),
           ((64, 4, 16, 16, 13), 2, (2, 2), (2, 2), (0, 0), (3, 3)),
           ((64, 4, 16, 16, 12), 1, (5, 3), (5, 2), (0, 0), (1, 1)),
           ((8, 16, 16, 16, 100), 2, (3, 3), (2, 2), (1, 1), (2, 1))]


@pytest.mark.parametrize('form', CLASSES, ids=str)
def test_a_pixel_meets_the_taps_of_its_own_class(form):
    """Terms of at most 15 in a sum of at most 16 * 9 of them."""
    import lava_dl_amd.slayer as slayer
    shape, co, kernel, stride, padding, dilation = form
    gen = torch.Generator().manual_seed(sum(shape) + co)
    x, w = _integers(gen, shape, 3), _integers(gen, (shape[1], co) + kernel + (1,), 5)
    cfg = (stride + (1,), padding + (0,), dilation + (1,))
    want = F.conv_transpose3d(x, w, None, cfg[0], cfg[1], 0, 1, cfg[2])
    got = slayer.synapse.conv_transpose_synapse(x.to(dev()), w.to(dev()), stride, padding, dilation)
    assert torch.equal(got.cpu(), want), 'transposed convolution'
    image = torch.zeros(want.shape, device=dev()).requires_grad_()
    slayer.synapse.conv_synapse(image, w.to(dev()), stride, padding, dilation).backward(x.to(dev()))
    assert torch.equal(image.grad.cpu(), want), 'input gradient'


@pytest.mark.parametrize('transposed', [False, True])
@pytest.mark.parametrize('steps', [66, 67, 131])
@pytest.mark.parametrize('cut', [None, (1, 1, 2, False), (2, 2, 2, False), (1, 1, 2, True)], ids=str)
def test_finite_results_are_those_of_the_call_without_the_infinite_value(transposed, steps, cut):
    """The last two quads of a pixel share steps and may lie in two waves: 17 or 33 quads of a pixel, 16 in a wave."""
    import lava_dl_amd.slayer as slayer
    gen = torch.Generator().manual_seed(steps)
    x = torch.randn(2, 3, 5, 4, steps, generator=gen)
    w = torch.randn(*((3, 18) if transposed else (18, 3)), 3, 3, 1, generator=gen)
    op = slayer.synapse.conv_transpose_synapse if transposed else slayer.synapse.conv_synapse
    if cut is not None:
        def op(x, w, *_):
            w = (w.transpose(0, 1) if transposed else w)[..., 0].contiguous()
            return _cut(transposed, x, w, (2, 18, 5, 4, steps), (1, 1), (1, 1), (1, 1), False, *cut)
    want = op(x.to(dev()), w.to(dev()), 1, 1, 1)
    x[0, 1, 2, 1, 10] = float('inf')
    x[1, 0, 0, 0, steps - 3] = float('inf')
    got = [op(x.to(dev()), w.to(dev()), 1, 1, 1) for _ in range(2)]
    finite = got[0].isfinite()
    met = torch.zeros_like(x).masked_fill_(~x.isfinite(), 1.0)
    conv = F.conv_transpose3d if transposed else F.conv3d
    assert torch.equal(finite.cpu(), conv(met, torch.ones_like(w), None, 1, (1, 1, 0)) == 0)
    assert not finite.all() and finite.sum() > finite.numel() // 4
    if cut is None or cut[0] == 1:
        assert torch.equal(got[0][finite], want[finite])
    else:       # pixels together have each other's taps as products with zero: a result beside it may be a float32 sum of 27 terms, too
        terms = conv(x.nan_to_num(0.0, 0.0, 0.0).abs(), w.abs(), None, 1, (1, 1, 0)).to(dev())       # and each sum within 28 * 2^-24 of these
        assert bool(((got[0] - want).abs() <= 2 * 28 * 2.0 ** -24 * terms)[finite].all())
    assert torch.equal(got[0].nan_to_num(7.0, 8.0, 9.0), got[1].nan_to_num(7.0, 8.0, 9.0))


# ------------------------------------------------------------------ the cut given
def _cut(input_grad, x, w, out_shape, stride, padding, dilation, by_class, pixels, blocks, pieces, whole=False):
    """The call with the cut given, or None where there is no such cut.  w: [Co, Ci, kh, kw], Co the channels of the result."""
    from lava_dl_amd.slayer import _native as N
    out = torch.full(out_shape, -12345.0, device=dev())
    big, small = (out_shape, x.shape) if input_grad else (x.shape, out_shape)            # of the plain convolution
    with N.device_guard(x.device):
        code = N.lib().slayer_conv_synapse_cut(N.ptr(out), N.ptr(x), N.ptr(w), big[0], big[1], small[1], *big[2:], *w.shape[2:], *stride,
                                               *padding, *dilation, int(input_grad), int(by_class), pixels, blocks, pieces, int(whole),
                                               N.stream_handle())
    if code == -3:
        return None
    N.check(code)
    return out


@pytest.mark.parametrize('form', FORMS + CLASSES[3:5], ids=str)
def test_every_cut_of_a_layer_gives_the_same(form):
    """Terms of at most 15, a few hundred of them."""
    shape, co, kernel, stride, padding, dilation = form
    shape = (min(shape[0], 3),) + shape[1:]
    gen = torch.Generator().manual_seed(sum(shape) + co + 2)
    x, w = _integers(gen, shape, 3), _integers(gen, (co, shape[1]) + kernel, 5)
    cfg = (stride + (1,), padding + (0,), dilation + (1,))
    want = F.conv3d(x, w[..., None], None, *cfg)
    up = [(shape[2 + i] - 1) * stride[i] - 2 * padding[i] + dilation[i] * (kernel[i] - 1) + 1 for i in (0, 1)]
    cases = [(False, False, x.to(dev()), w.to(dev()), want)]
    if min(up) >= 1:
        want = F.conv_transpose3d(x, w.transpose(0, 1)[..., None], None, cfg[0], cfg[1], 0, 1, cfg[2])
        cases += [(True, by_class, x.to(dev()), w.to(dev()), want) for by_class in (False, True)]
    taken = [0, 0]
    for input_grad, by_class, xd, wd, want in cases:
        for pixels in (1, 2, 3, 4, 6, 8):
            for blocks in (1, 2):
                for pieces, whole in ((1, False), (2, False), (3, False), (16, False), (1, True), (3, True), (16, True)):
                    got = _cut(input_grad, xd, wd, want.shape, stride, padding, dilation, by_class, pixels, blocks, pieces, whole)
                    assert got is None or torch.equal(got.cpu(), want), (input_grad, by_class, pixels, blocks, pieces, whole)
                    taken[pixels > 1] += got is not None
    if max(kernel) < 6 and 1 in dilation:
        assert taken[0]
    if max(kernel) < 6 and dilation == (1, 1):
        assert taken[1]


@pytest.mark.parametrize('split', ['input', 'neither'])
@pytest.mark.parametrize('blocks', [1, 2])
@pytest.mark.parametrize('channels', [5, 12, 20, 30, 70])            # two, four, six, eight loads to a lane; more groups than one
@pytest.mark.parametrize('taps', [1, 2, 3, 4, 5])
def test_every_form_of_the_walking_kernel(taps, channels, blocks, split):
    """`taps` along the walk and one along the line: as many triples as channels.  At most 5 * 70 terms of 1025 * 5: below 2^24."""
    gen = torch.Generator().manual_seed(100 * taps + channels)
    x, w = _integers(gen, (2, channels, 7, 3, 18), 3), _integers(gen, (40, channels, taps, 1), 5)
    if split == 'input':
        x = _integers(gen, x.shape, 1025)
    want = F.conv3d(x.double(), w[..., None].double(), None, 1, (taps // 2, 0, 0))
    got = _cut(False, x.to(dev()), w.to(dev()), want.shape, (1, 1), (taps // 2, 0), (1, 1), False, 1, blocks, 2)
    assert got is not None and torch.equal(got.cpu().double(), want)    # five taps and two blocks: walked along the other axis


@pytest.mark.parametrize('form', [((2, 56, 16, 9, 9), 16, (9, 2), (8, 1), (0, 0), (1, 1)),      # weights beyond LDS along the rows
                                  ((2, 16, 45, 8, 9), 8, (32, 2), (1, 1), (0, 0), (1, 1)),      # 1024 taps on the one-pixel kernel
                                  ((2, 12, 45, 8, 9), 8, (16, 5), (1, 1), (0, 0), (1, 1))], ids=str)
def test_filters_of_the_most_taps(form):
    import lava_dl_amd.slayer as slayer
    shape, co, kernel, stride, padding, dilation = form
    gen = torch.Generator().manual_seed(shape[1])
    x, w = _integers(gen, shape, 3), _integers(gen, (co, shape[1]) + kernel, 5)
    want = F.conv3d(x, w[..., None], None, stride + (1,), padding + (0,), dilation + (1,))
    assert torch.equal(slayer.synapse.layer._launch(x.to(dev()), w.to(dev()), stride, padding, dilation).cpu(), want)
    if stride == (8, 1):
        got = _cut(False, x.to(dev()), w.to(dev()), want.shape, stride, padding, dilation, False, 1, 1, 4)
        assert got is not None and torch.equal(got.cpu(), want)
