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
