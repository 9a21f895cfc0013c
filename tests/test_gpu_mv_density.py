"""GPU: the event and value mat-vec chooses between atomics and sums in LDS from the density of the
spikes (word 0 of a batch row's workspace header: 0 row groups for atomics); both ways against
float64 sums."""
import ctypes

import pytest

pytestmark = pytest.mark.gpu


# single vectors: rows past the sample, and fewer rows than it; batches: several row groups and
# rows of odd length, then one row group of many spans (the workspace is its header alone)
@pytest.mark.parametrize('B,n_pre,n_post,k,kind', [
    (1, 100_003, 20_001, 201, 'value'), (1, 3001, 9000, 7001, 'event'),
    (1, 250_001, 20_001, 201, 'event_shared'), (9, 5001, 6000, 100, 'value'),
    (9, 5003, 6000, 100, 'event'), (260, 40_001, 300, 30, 'value_shared')])
@pytest.mark.parametrize('p', [0.0, 2e-4, 0.5])
@pytest.mark.parametrize('sdt', ['u8', 'f32'])
def test_way_follows_density(B, n_pre, n_post, k, kind, p, sdt):
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import _native as N
    value, shared = kind.startswith('value'), kind.endswith('shared')
    if value and sdt == 'u8':
        pytest.skip('values are fp32')
    print('[case] mv density', B, n_pre, n_post, k, kind, p, sdt, flush=True)
    gen = torch.Generator(device='cuda').manual_seed(n_pre)
    rand = lambda *s: torch.rand(s, device='cuda', generator=gen)  # noqa: E731
    idx = torch.randint(-1, n_post + 1, (n_pre, k), device='cuda', generator=gen,
                        dtype=torch.int32)
    w = None if shared else rand(n_pre, k) - 0.3
    x = rand(B, n_pre)
    act = x < p
    x = act.to(torch.uint8) if sdt == 'u8' else torch.where(act, x - 0.9 * p,
                                                            torch.zeros_like(x))
    base = rand(B, n_post)
    nbytes = int(N.lib().bs_matvec_workspace_size(B, n_pre, k, n_post,
                                                  1 if kind == 'event_shared' else 0))
    assert nbytes % (4 * B) == 0 and nbytes >= 256 * B
    outs = []
    for acc in (0, 1):
        ws = torch.full((nbytes // 4,), 77, dtype=torch.int32, device='cuda')
        out = base.clone()
        N.check(N.lib().bs_matvec_ws_f32(
            N.ptr(x), N.BS_SPK_U8 if sdt == 'u8' else N.BS_SPK_F32, 1 if value else 0, B, n_pre,
            N.ptr(idx), k, N.ptr(w), 0.37, n_post, N.ptr(out), acc, N.ptr(ws), nbytes,
            ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)), 'bs_matvec_ws_f32')
        groups = ws.reshape(B, -1)[:, 0]
        assert bool((groups == 0).all()) if p < 0.1 else bool((groups >= 1).all())
        outs.append(out)
    for b in sorted({0, B // 2, B - 1}):
        rows = x[b].nonzero().reshape(-1)
        j = idx[rows].long()
        v = (x[b][rows].double() if value else torch.ones_like(rows).double())[:, None] * \
            (0.37 if shared else w[rows].double())
        v = torch.where((j >= 0) & (j < n_post), v.expand(j.shape), torch.zeros_like(v))
        j = j.clamp(0, n_post - 1).reshape(-1)
        want = torch.zeros(n_post, dtype=torch.float64, device='cuda').index_add_(
            0, j, v.reshape(-1))
        # an fp32 sum of n terms in any order: n 2^-24 of the terms' absolute sum at most (and
        # the products' and the weight's rounding, one each)
        size = torch.zeros_like(want).index_add_(0, j, v.reshape(-1).abs())
        n = torch.zeros_like(want).index_add_(0, j, (v.reshape(-1) != 0).double())
        bound = (n + 2) * 2.0 ** -24 * (size + base[b].double().abs()) + 1e-30
        assert bool(((outs[0][b].double() - want).abs() <= bound).all()), b
        assert bool(((outs[1][b].double() - want - base[b].double()).abs() <= bound).all()), b


def test_few_long_rows_take_lds():
    """60 rows of 50,000 synapses in 8 batch rows: one workgroup per batch row could add them by
    atomics (1,007 us at p = 0.1), so the outputs are summed in LDS (109), with the same sums."""
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import ops
    print('[case] mv long rows', flush=True)
    gen = torch.Generator(device='cuda').manual_seed(2)
    B, n_pre, n_post, k = 8, 60, 5000, 50_000
    idx = torch.randint(0, n_post, (n_pre, k), device='cuda', generator=gen, dtype=torch.int32)
    x = (torch.rand(B, n_pre, device='cuda', generator=gen) < 0.2).float()
    # integer weights: every sum is exact
    w = torch.randint(-3, 4, (n_pre, k), device='cuda', generator=gen).float()
    out = ops.value_matvec(x, idx, w, n_post)
    for b in range(B):
        want = torch.zeros(n_post, device='cuda')
        for r in x[b].nonzero().reshape(-1):
            want.index_add_(0, idx[r].long(), w[r])
        assert torch.equal(out[b], want), b
