"""GPU: the event and value mat-vec on sizes whose sums are formed in LDS, against float64 sums
and, for events of one shared weight, bit for bit against the bucketed operator (both add the
weight once per event in one chain)."""
import pytest

pytestmark = pytest.mark.gpu


# single vectors: one range, the most ranges, a last range cut to nothing, many rows per group,
# one row group; batches: a few row groups each, one, and posts in slices of a few outputs (small
# ones stay with k_matvec)
@pytest.mark.parametrize('B,n_pre,n_post,k,p', [
    (0, 400_000, 17, 125, 0.01), (0, 50_001, 128_000, 1001, 0.03), (0, 50_000, 16_001, 1000, 0.002),
    (0, 100_003, 3, 500, 0.0), (0, 60, 90_000, 900_000, 0.5), (8, 4097, 16_000, 33, 0.3),
    (33, 1000, 300, 64, 0.5), (64, 3200, 4000, 80, 0.05), (9, 8200, 20_003, 65, 1.0),
    (130, 5, 1, 3, 0.6), (260, 2000, 5, 40, 0.3)])
@pytest.mark.parametrize('kind', ['event', 'value', 'event_shared', 'value_shared'])
@pytest.mark.parametrize('sdt', ['u8', 'f32'])
def test_matvec_lds(B, n_pre, n_post, k, p, kind, sdt):
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    from brainstate_amd import ops
    print('[case] mv lds', B, n_pre, n_post, k, p, kind, sdt, flush=True)
    value, shared = kind.startswith('value'), kind.endswith('shared')
    if value and sdt == 'u8':
        pytest.skip('values are fp32')
    gen = torch.Generator(device='cuda').manual_seed(n_pre + k)
    rand = lambda *s: torch.rand(s, device='cuda', generator=gen)  # noqa: E731
    idx = torch.randint(-1, n_post + 1, (n_pre, k), device='cuda', generator=gen,
                        dtype=torch.int32)
    w = 0.37 if shared else rand(n_pre, k) - 0.3
    lead = (B,) if B else ()
    x = rand(*lead, n_pre)
    act = x < p
    x = act.to(torch.uint8) if sdt == 'u8' else torch.where(act, x - 0.9 * p, torch.zeros_like(x))
    f = ops.value_matvec if value else ops.event_matvec
    out = f(x, idx, w, n_post)
    base = rand(*lead, n_post)
    acc = f(x, idx, w, n_post, out=base.clone(), accumulate=True)
    xs, os, bs_, as_ = (t.reshape(-1, t.shape[-1]) for t in (x, out, base, acc))
    L = ops.build_buckets(idx, n_post, w_homo=0.37) if kind == 'event_shared' else None
    for b in sorted({0, xs.shape[0] // 2, xs.shape[0] - 1}):
        rows = xs[b].nonzero().reshape(-1)
        j = idx[rows].long()
        v = (xs[b][rows].double() if value else torch.ones_like(rows).double())[:, None] * \
            (0.37 if shared else w[rows].double())
        v = torch.where((j >= 0) & (j < n_post), v.expand(j.shape), torch.zeros_like(v))
        j = j.clamp(0, n_post - 1).reshape(-1)
        want = torch.zeros(n_post, dtype=torch.float64, device='cuda').index_add_(
            0, j, v.reshape(-1))
        # an fp32 sum of n terms in any order: n 2^-24 of the terms' absolute sum at most
        size = torch.zeros_like(want).index_add_(0, j, v.reshape(-1).abs())
        n = torch.zeros_like(want).index_add_(0, j, (v.reshape(-1) != 0).double())
        bound = (n + 2) * 2.0 ** -24 * (size + bs_[b].double().abs()) + 1e-30
        assert bool(((os[b].double() - want).abs() <= bound).all()), b
        assert bool(((as_[b].double() - want - bs_[b].double()).abs() <= bound).all()), b
        if L is not None:
            assert torch.equal(os[b], ops.event_bucket(xs[b], L, mode='split')), b
