"""GPU: gradients of a batch through the transposed form against the per-row kernel, bit for bit
(grad_spk, and grad_w as the per-row gradients added in row order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 16 and 64 batch lanes, one lane group past each, batches that end inside a group; rows of less
# than one, one, and several chunks; tiles of the transposition cut on both sides
@pytest.mark.parametrize('B,n_pre,n_post,k', [(3, 7000, 63, 65), (8, 50, 64, 64), (16, 300, 65, 17),
                                              (17, 200, 1000, 80), (64, 129, 127, 128),
                                              (65, 40, 1, 200), (130, 33, 500, 1), (9, 4, 4000, 1000)])
@pytest.mark.parametrize('het', [True, False])
@pytest.mark.parametrize('csr', [True, False])
@pytest.mark.parametrize('odd', [True, False])
def test_transposed_vjp_equals_rows(B, n_pre, n_post, k, het, csr, odd):
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import _native as N
    from brainstate_amd import ops
    print('[case] vjp batch', B, n_pre, n_post, k, het, csr, odd, flush=True)
    assert N.lib().bs_event_matvec_vjp_batch_workspace_size(B, n_pre, n_post) > 0
    rs = np.random.RandomState(B + k)
    t = lambda a: torch.as_tensor(a, device='cuda')  # noqa: E731
    idx = rs.randint(-2, n_post + 2, (n_pre, k)).astype(np.int32)
    indptr = None
    if csr:
        lens = rs.randint(0, k + 1, n_pre)
        indptr = t(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
        idx = idx.reshape(-1)[:int(lens.sum())]
    idx = t(idx)
    w = t(rs.randn(*idx.shape).astype(np.float32)) if het else 0.7
    x = t(np.where(rs.rand(B, n_pre) < 0.2, rs.rand(B, n_pre) + 0.1, 0).astype(np.float32))
    g = rs.randn(B, n_post).astype(np.float32)
    if odd:
        g[B // 2, n_post // 2] = np.inf
        g[0, 0] = np.nan
    g = t(g)
    gs, gw = ops.event_matvec_vjp_batch(x, idx, w, n_post, g, indptr=indptr)
    same = lambda a, b: torch.equal(torch.nan_to_num(a, nan=7e30), torch.nan_to_num(b, nan=7e30))  # noqa: E731
    total, absum = None, 0.0
    for b in range(B):
        a, c = ops.event_matvec_vjp(x[b], idx, w, n_post, g[b].contiguous(), indptr=indptr)
        assert same(gs[b], a), b
        total = c if total is None else total + c
        absum += float(x[b].sum()) * k * float(g[b].abs().max())
    if het:
        assert same(gw, total)
    elif not odd:
        # n fp32 terms of one sum in another order: n 2^-24 of their absolute sum at most
        assert abs(float(gw) - float(total)) <= 1e-5 * absum
    only = ops.event_matvec_vjp_batch(x, idx, w, n_post, g, indptr=indptr, need_w=False)[0]
    assert same(only, gs)


# calls that take the transposed form and calls that keep one wave per row for the whole batch
# (its launch and the transposition of a wide g cost more than the gathers of few synapses)
@pytest.mark.parametrize('B,n_pre,n_post,k,transposed', [
    (2, 20_000, 300, 9, False), (3, 700, 200_003, 20, False), (5, 3000, 400, 80, False),
    (8, 51, 100_001, 33, False), (17, 70, 100_001, 20, False), (3, 7000, 63, 65, False),
    (64, 320, 400, 80, True), (16, 500, 1000, 200, True), (3, 40_000, 500, 130, True)])
@pytest.mark.parametrize('het', [True, False])
@pytest.mark.parametrize('csr', [True, False])
def test_route_and_bits_of_the_two_entry_points(B, n_pre, n_post, k, transposed, het, csr):
    import ctypes
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import _native as N
    print('[case] vjp batch route', B, n_pre, n_post, k, het, csr, flush=True)
    rs = np.random.RandomState(B + k)
    t = lambda a: torch.as_tensor(a, device='cuda')  # noqa: E731
    idx = rs.randint(-2, n_post + 2, (n_pre, k)).astype(np.int32)
    indptr, per = None, k
    if csr:
        lens = rs.randint(0, k + 1, n_pre)
        indptr = t(np.concatenate([[0], np.cumsum(lens)]).astype(np.int32))
        idx = idx.reshape(-1)[:int(lens.sum())]
        per = k // 2
    idx = t(idx)
    w = t(rs.randn(*idx.shape).astype(np.float32)) if het else None
    # small integers: the shared weight's gradient is exact in every order
    x = t((rs.randint(1, 4, (B, n_pre)) * (rs.rand(B, n_pre) < 0.3)).astype(np.float32))
    g = t((rs.randn(B, n_post) if het else rs.randint(-3, 4, (B, n_post))).astype(np.float32))
    got = []
    nbytes = int(N.lib().bs_event_matvec_vjp_batch_workspace_size(B, n_pre, n_post))
    ws = torch.full((max(nbytes, 8),), 0xA5, dtype=torch.uint8, device='cuda')
    for with_ws in (False, True):
        gs = torch.empty(B, n_pre, device='cuda')
        gw = torch.empty(idx.shape if het else (), device='cuda')
        args = (N.ptr(x), N.BS_SPK_F32, B, n_pre, N.ptr(indptr), N.ptr(idx), per, N.ptr(w), 0.5,
                n_post, N.ptr(g), N.ptr(gs), N.ptr(gw))
        sh = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        if with_ws:
            N.check(N.lib().bs_event_matvec_vjp_batch_ws_f32(*args, N.ptr(ws), nbytes, sh), 'ws')
        else:
            N.check(N.lib().bs_event_matvec_vjp_batch_f32(*args, sh), 'per row')
        got.append((gs, gw))
    assert bool((ws != 0xA5).any()) == transposed
    (gs, gw), (gs2, gw2) = got
    assert torch.equal(gs, gs2) and torch.equal(gw, gw2)
    from brainstate_amd import ops
    total = None
    for b in range(B):
        a, c = ops.event_matvec_vjp(x[b], idx, w if het else 0.5, n_post, g[b].contiguous(),
                                    indptr=indptr)
        assert torch.equal(gs[b], a), b
        total = c if total is None else total + c
    assert torch.equal(gw, total)


def test_more_batch_rows_than_a_grid_has_in_y():
    """65,537 tiles of 64 batch rows, one past a grid's y limit here: gradients of the few rows that carry any equal the per-row
    calls, the others are zero."""
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import ops
    B, n_pre, n_post, k = 65_536 * 64 + 1, 2, 3, 5
    print('[case] vjp batch rows', B, flush=True)
    rs = np.random.RandomState(4)
    t = lambda a: torch.as_tensor(np.asarray(a), device='cuda')  # noqa: E731
    idx = t(rs.randint(0, n_post, (n_pre, k)).astype(np.int32))
    w = t(rs.randn(n_pre, k).astype(np.float32))
    x = torch.zeros(B, n_pre, device='cuda')
    g = torch.zeros(B, n_post, device='cuda')
    at = [0, 63, 64, 70_000, B // 2, B - 2, B - 1]
    for b in at:
        x[b] = t(rs.rand(n_pre).astype(np.float32) + 0.5)
        g[b] = t(rs.randn(n_post).astype(np.float32))
    gs, gw = ops.event_matvec_vjp_batch(x, idx, w, n_post, g)
    total = None
    for b in at:
        a, c = ops.event_matvec_vjp(x[b], idx, w, n_post, g[b].contiguous())
        assert torch.equal(gs[b], a), b
        total = c if total is None else total + c
    assert torch.equal(gw, total)
    gs[at] = 0
    assert int(torch.count_nonzero(gs)) == 0
