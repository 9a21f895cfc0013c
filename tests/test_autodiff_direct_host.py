"""Which form of an autograd Function a recorded call takes (CPU)."""
from types import SimpleNamespace

import pytest
import torch

from brainstate_amd.nn import _event


@_event._with_direct
class _Square(torch.autograd.Function):
    @staticmethod
    def forward(x):
        return x * x

    @staticmethod
    def setup_context(ctx, inputs, output):
        ctx.save_for_backward(inputs[0])
        ctx.save_for_forward(inputs[0])

    @staticmethod
    def backward(ctx, g):
        return 2 * ctx.saved_tensors[0] * g

    @staticmethod
    def jvp(ctx, t):
        return 2 * ctx.saved_tensors[0] * t


@pytest.mark.parametrize('known', [True, False])
def test_recorded_form(monkeypatch, known):
    """Outside transforms the direct form; inside them, and on a torch without the query for
    active transforms, the form with its own setup_context."""
    if not known:
        monkeypatch.setattr(_event, 'torch', SimpleNamespace(_C=SimpleNamespace()))
    x = torch.tensor([1.0, -3.0], requires_grad=True)
    y = _event._record(_Square, x)
    assert type(y.grad_fn).__name__ == ('_SquareDirectBackward' if known else '_SquareBackward')
    g, = torch.autograd.grad(y.sum(), x)
    assert torch.equal(g, 2 * x)
    v = torch.func.grad(lambda a: _event._record(_Square, a).sum())(x.detach())
    assert torch.equal(v, g.detach())
