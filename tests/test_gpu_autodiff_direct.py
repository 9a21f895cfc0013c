"""GPU: the event operators record the same derivatives inside torch.func transforms and
outside them (reverse mode, forward-mode duals, saved-tensor hooks)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('layer', ['conn', 'conn_batch', 'linear', 'homo'])
def test_derivatives_equal_torch_func(layer):
    import torch
    import torch.autograd.forward_ad as fa
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    import brainstate_amd as bs
    rs = np.random.RandomState(3)
    f = lambda *s: torch.as_tensor(np.float32(rs.randn(*s)), device='cuda')  # noqa: E731
    n_in, n_out = 40, 30
    x = (f(n_in) > 0.5).float() if layer != 'conn_batch' else (f(5, n_in) > 0.5).float()
    if layer.startswith('conn'):
        m, w = bs.nn.EventFixedProb(n_in, n_out, 6, f(n_in, 6), seed=1), f(n_in, 6)
    elif layer == 'linear':
        m, w = bs.nn.EventLinear(n_in, n_out, f(n_in, n_out)), f(n_in, n_out)
    else:
        m, w = bs.nn.EventLinear(n_in, n_out, 0.3), torch.tensor(0.3, device='cuda')
    dx, dw = f(*x.shape), f(*w.shape)

    def fun(x, w):
        m.weight.restore_value(w)
        return m(x)

    want, want_t = torch.func.jvp(fun, (x, w), (dx, dw))
    with fa.dual_level():
        out = fa.unpack_dual(fun(fa.make_dual(x, dx), fa.make_dual(w, dw)))
    close = lambda a, b: torch.allclose(a, b, rtol=1e-5, atol=1e-5)  # noqa: E731
    assert close(out.primal, want) and close(out.tangent, want_t)
    g = f(*want.shape)
    wx, ww = torch.func.vjp(fun, x, w)[1](g)
    xa, wa = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
    seen = []
    with torch.autograd.graph.saved_tensors_hooks(lambda t: seen.append(t) or t, lambda t: t):
        y = fun(xa, wa)
    gx, gw = torch.autograd.grad(y, (xa, wa), g)
    assert close(y, want) and close(gx, wx) and close(gw, ww)
    assert any(t.shape == x.shape for t in seen)
    with torch.no_grad():
        assert not fun(xa, wa).requires_grad
