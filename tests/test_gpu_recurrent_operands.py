"""The operands of the recurrent weight gradient in one launch (csrc/recurrent_wgrad.hip), at the edges of its tiles of 64 neurons
x 64 steps, against the operators it stands for: copies, so equal; and who still gets the operators."""
import pytest
import torch

from tests.util import dev

pytestmark = pytest.mark.gpu


def _operators(grad, x):
    return (grad[..., 1:].transpose(0, 1).reshape(grad.shape[1], -1), x[..., :-1].transpose(1, 2).reshape(-1, x.shape[1]))


@pytest.mark.parametrize('n,c,t', [(1, 1, 2), (2, 64, 64), (3, 65, 65), (1, 63, 66), (5, 130, 129), (2, 4, 300)])
def test_operands_equal_the_operators(n, c, t):
    from lava_dl_amd.slayer.utils import recurrent as R
    gen = torch.Generator().manual_seed(n + c + t)
    grad, x = (torch.randn(n, c, t, generator=gen).to(dev()) for _ in range(2))
    for got, want in zip(R._operands(grad, x), _operators(grad, x)):
        assert got.shape == want.shape and torch.equal(got, want)


def test_calls_that_keep_the_operators():
    from lava_dl_amd.slayer.utils import recurrent as R
    grad, x = torch.randn(2, 5, 7, device=dev()), torch.randn(2, 5, 7, device=dev())
    assert R._operands(grad[..., :1], x[..., :1]) is None                       # no step before the first
    assert R._operands(grad.transpose(0, 1), x.transpose(0, 1)) is None         # not as they lie in memory
    assert R._operands(grad.double(), x.double()) is None
    assert R._operands(grad.cpu(), x.cpu()) is None
    assert R._operands(grad, x.requires_grad_()) is None                        # a graph of the gradient is wanted
    with torch.no_grad():
        assert R._operands(grad, x) is not None
    want = torch.matmul(*_operators(grad, x.detach()))
    assert torch.equal(torch.func.vmap(R._weight_gradient)(grad[None], x.detach()[None])[0], want)
