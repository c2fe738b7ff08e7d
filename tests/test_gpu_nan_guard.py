"""The NaN guard of the resonator family's backward pass (resonator.py:421-439 in the reference): the kernels report on
their way, the tensors are searched only when they have something to report.  Step-by-step passes, scans of whole-quad
rows and of any-length rows; a NaN in the first, an inner and the last sample; infinities of both signs are no NaN."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(2, 8, 50), (1, 3, 4), (8, 32, 4100), (64, 64, 301)]       # the last two have 2^20 elements and more


def _pass(shape, grad, learn, delayed=False):
    import lava_dl_amd.slayer as slayer
    gen = torch.Generator().manual_seed(5)
    x = [torch.randn(shape, generator=gen).cuda().requires_grad_() for _ in range(2)]
    neuron = slayer.neuron.rf.Neuron(threshold=1.0, period=10, decay=0.1, requires_grad=learn).cuda()
    delays = None
    if delayed:
        delays = slayer.neuron.dynamics.delays.Delays(output_delay=torch.full((shape[1],), 3.0).cuda())
    neuron(tuple(x), delays=delays).backward(grad)
    return x


@pytest.mark.parametrize('learn', [False, True])
@pytest.mark.parametrize('shape', SHAPES)
def test_nan_anywhere_in_the_gradient_raises(shape, learn):
    numel = shape[0] * shape[1] * shape[2]
    for at in (0, numel // 2 + 1, numel - 1):
        grad = torch.ones(shape).cuda()
        grad.view(-1)[at] = float('nan')
        with pytest.raises(Exception, match='grad_spikes has NaN'):
            _pass(shape, grad, learn)
    grad = torch.ones(shape).cuda()
    assert torch.isfinite(_pass(shape, grad, learn)[0].grad).all()


@pytest.mark.parametrize('shape', SHAPES)
def test_nan_that_a_delay_shifts_out_of_its_row_raises(shape):
    grad = torch.ones(shape).cuda()
    grad[..., 0] = float('nan')                  # read back at t = -3: no result ever sees it
    with pytest.raises(Exception, match='grad_spikes has NaN'):
        _pass(shape, grad, False, delayed=True)


@pytest.mark.parametrize('shape', SHAPES)
def test_infinities_of_both_signs_are_not_reported(shape):
    import lava_dl_amd.slayer as slayer
    zero = torch.zeros(1).cuda()
    sin, cos = torch.full((1,), 0.0).cuda(), torch.full((1,), 2048.0).cuda()
    x = torch.zeros(shape).cuda().requires_grad_()
    re, im = slayer.neuron.dynamics.resonator.dynamics(x, torch.zeros(shape).cuda(), sin, cos, zero, zero, 64)
    grad = torch.zeros(shape).cuda()
    grad[0, 0, 0], grad[0, -1, 0] = float('inf'), float('-inf')     # step 0: no earlier step takes them up
    g, = torch.autograd.grad(slayer.neuron.dynamics.resonator.dynamics(
        x, torch.zeros(shape).cuda(), sin, cos, zero, zero, 64), x, [grad, torch.zeros(shape).cuda()])
    assert torch.equal(g, grad)


@pytest.mark.parametrize('model', ['rf', 'resonator', 'adaptive'])
def test_a_call_that_fails_waits_for_its_launches(model, monkeypatch):
    """The word the kernels report NaN in goes back to torch's pinned-memory cache when the call ends: a call that raises
    after its launches (a raised range flag of an earlier call does) must not let go of it while they are still to run."""
    import lava_dl_amd.slayer as slayer
    from lava_dl_amd.slayer import _native
    D, zero = slayer.neuron.dynamics, torch.zeros(1).cuda()
    sin, cos = torch.full((1,), 100.0).cuda(), torch.full((1,), 2048.0).cuda()
    x = [torch.randn(2, 3, 21).cuda().requires_grad_() for _ in range(2)]
    if model == 'rf':
        y = slayer.neuron.rf.Neuron(threshold=1.0, period=10, decay=0.1).cuda()(tuple(x))
    elif model == 'resonator':
        y = sum(D.resonator.dynamics(*x, sin, cos, zero, zero, 64))
    else:
        y = sum(D.adaptive_resonator.dynamics(*x, sin, cos, sin, sin, zero, zero, zero, zero, 1.0, 1.0, 64)[:2])

    class Failed(Exception):
        pass

    def check(code):
        assert code == 0
        raise Failed()
    grad = torch.ones_like(y)
    torch.cuda.synchronize()
    monkeypatch.setattr(_native, 'check', check)
    torch.cuda._sleep(200_000_000)                                   # the launches queue up behind this
    with pytest.raises(Failed):
        y.backward(grad)
    assert torch.cuda.current_stream().query()
