"""GPU: the shared weight's gradient, one sum over every synapse of every active row, is carried
past the row sums in 64 bits in each kernel that forms it.

Rows in groups of four have row sums 2^26, 1, -2^26, 1: exact in fp32, as is every group's total
of 2.  The kernels add groups of whole rows (4 waves take 4 neighbouring rows, or a wave a multiple of 4), so a
64-bit sum over a workgroup is exact and so are the fp32 sums of the workgroups' small integers:
equality is required, and one row dropped, doubled or added in fp32 to 2^26 breaks it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rows(torch, n_pre, n_post, k, csr):
    """(indices, indptr, g): the row sums above, from three posts far apart; g is 0 elsewhere."""
    rs = np.random.RandomState(n_pre)
    at = [0, n_post // 2, n_post - 1]                       # posts worth 2^26, 1, -2^26
    lens = rs.randint(1, k + 1, n_pre) if csr else np.full(n_pre, k)
    ptr = np.concatenate([[0], np.cumsum(lens)])
    idx = rs.randint(1, n_post // 2, int(ptr[-1]))          # g = 0
    idx[ptr[:-1] + rs.randint(0, lens)] = np.asarray([at[0], at[1], at[2], at[1]])[
        np.arange(n_pre) % 4]
    g = torch.zeros(n_post, device='cuda')
    for j, v in zip(at, (2.0 ** 26, 1.0, -2.0 ** 26)):
        g[j] = v
    t = lambda a: torch.as_tensor(a.astype(np.int32), device='cuda')  # noqa: E731
    return t(idx if csr else idx.reshape(n_pre, k)), t(ptr) if csr else None, g


# a wave per row with g read from L2, and g passing through LDS: one range, two, and more, rows of
# one chunk up to several blocks.  There a wave owns neighbouring rows: n_pre is a multiple that
# starts every wave's rows at a group of four (16 waves per compute unit own rows, 12 with more
# than two ranges)
@pytest.mark.parametrize('per_wave,n_post,k', [(None, 5000, 30), (None, 100_000, 64), (4, 300, 100),
                                               (8, 20_417, 60), (4, 40_000, 130),
                                               (8, 60_000, 128), (4, 100_003, 2000)])
@pytest.mark.parametrize('sdt', ['u8', 'f32'])
def test_single_vectors(per_wave, n_post, k, sdt):
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import ops
    print('[case] shared gradient', per_wave, n_post, k, sdt, flush=True)
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    n_pre = 6004 if per_wave is None else cus * (12 if n_post > 2 * 20_416 else 16) * per_wave
    idx, _, g = _rows(torch, n_pre, n_post, k, False)
    x = torch.ones(n_pre, device='cuda', dtype=torch.uint8 if sdt == 'u8' else torch.float32)
    gs, gw = ops.event_matvec_vjp(x, idx, 0.5, n_post, g)
    assert float(gw) == n_pre // 2
    assert torch.equal(gs[:4], torch.tensor([2.0 ** 25, 0.5, -2.0 ** 25, 0.5], device='cuda'))
    assert float(ops.event_matvec_vjp(x, idx, 0.5, n_post, g, need_spk=False)[1]) == n_pre // 2


# batches with g transposed: 16 lanes and 64, one lane group and more
@pytest.mark.parametrize('B,n_pre,k', [(16, 500, 200), (64, 3200, 80), (130, 400, 33)])
@pytest.mark.parametrize('csr', [False, True])
def test_transposed(B, n_pre, k, csr):
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import ops
    print('[case] shared gradient, transposed', B, n_pre, k, csr, flush=True)
    n_post = 700
    idx, indptr, g = _rows(torch, n_pre, n_post, k, csr)
    x = torch.ones(B, n_pre, device='cuda')
    _, gw = ops.event_matvec_vjp_batch(x, idx, 0.5, n_post, g.expand(B, n_post), indptr=indptr)
    assert float(gw) == B * n_pre // 2


# batches of two, and of a few on a small layer: one wave per row for all of them
@pytest.mark.parametrize('B,n_pre,k', [(2, 100_000, 70), (2, 36, 3), (5, 3000, 80), (7, 2000, 64)])
@pytest.mark.parametrize('csr', [False, True])
@pytest.mark.parametrize('sdt', ['u8', 'f32'])
def test_batched_rows(B, n_pre, k, csr, sdt):
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import ops
    print('[case] shared gradient, batch', B, n_pre, k, csr, sdt, flush=True)
    n_post = 5000
    idx, indptr, g = _rows(torch, n_pre, n_post, k, csr)
    x = torch.ones(B, n_pre, device='cuda', dtype=torch.uint8 if sdt == 'u8' else torch.float32)
    gs, gw = ops.event_matvec_vjp_batch(x, idx, 0.5, n_post, g.expand(B, n_post), indptr=indptr)
    assert float(gw) == B * n_pre // 2
    if sdt == 'f32':
        x[:, ::4] = -0.0
        x[:, 2::4] = 0.0
        gw = ops.event_matvec_vjp_batch(x, idx, 0.5, n_post, g.expand(B, n_post),
                                        indptr=indptr, need_spk=False)[1]
        assert float(gw) == B * n_pre // 2                  # the rows of 1 alone
    assert torch.equal(gs[0, :4], torch.tensor([2.0 ** 25, 0.5, -2.0 ** 25, 0.5], device='cuda'))
