"""GPU: the reverse mode of the event mat-vec on sizes that take the LDS kernel, against the same
rows in calls small enough for the L2 kernel (each row's sum and each synapse's gradient are
formed by the same operations in the same order: bit for bit)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
R = 20416          # posts per LDS range


@pytest.fixture(scope='module')
def torch_cuda():
    import torch
    if not torch.cuda.is_available():
        pytest.fail('GPU tests need a ROCm GPU')
    return torch


# row lengths around one, two, four, eight and sixteen 64-synapse chunks and past 1,024;
# g of one range, two, three (the last cut short, not a multiple of 4) and five
@pytest.mark.parametrize('n_pre,k,n_post', [(40_000, 64, 1), (23_501, 65, R), (12_000, 128, R + 1),
                                            (6_100, 250, 2 * R), (4_099, 1000, 2 * R + 1),
                                            (1_600, 2049, 3 * R - 1), (3_500, 1024, 100_003),
                                            (30_001, 127, 2 * R + 5), (800, 4000, 50_000)])
@pytest.mark.parametrize('het', [True, False])
@pytest.mark.parametrize('sdt', ['u8', 'f32'])
def test_vjp_lds_equals_row_subsets(torch_cuda, n_pre, k, n_post, het, sdt):
    torch = torch_cuda
    from brainstate_amd import ops
    print('[case] vjp lds', n_pre, k, n_post, het, sdt, flush=True)
    gen = torch.Generator(device='cuda').manual_seed(n_pre + k)
    idx = torch.randint(-2, n_post + 2, (n_pre, k), device='cuda', generator=gen,
                        dtype=torch.int32)
    w = torch.randn(n_pre, k, device='cuda', generator=gen) if het else 0.37
    x = (torch.rand(n_pre, device='cuda', generator=gen) < 0.3).to(
        torch.uint8 if sdt == 'u8' else torch.float32)
    if sdt == 'f32':
        x = x * (torch.rand(n_pre, device='cuda', generator=gen) + 0.5)
    g = torch.randn(n_post + 1, device='cuda', generator=gen)
    if n_post > 8:
        g[3] = float('inf')
    g = g[1:] if k % 2 else g[:n_post]          # 4-byte and 16-byte aligned gradients
    gs, gw = ops.event_matvec_vjp(x, idx, w, n_post, g)
    same = lambda a, b: torch.equal(torch.nan_to_num(a, nan=7e30), torch.nan_to_num(b, nan=7e30))  # noqa: E731
    m = max(1, 400_000 // k)                    # rows per call: below every LDS rule
    gw_sum = 0.0
    for lo in range(0, n_pre, m):
        sl = slice(lo, min(lo + m, n_pre))
        a, b = ops.event_matvec_vjp(x[sl], idx[sl], w[sl] if het else w, n_post, g)
        assert same(gs[sl], a), lo
        if het:
            assert same(gw[sl], b), lo
        else:
            gw_sum += float(b)
    if not het and n_post <= 8:
        # one sum over n_pre * k terms of magnitude up to |g| x: fp32 rounding of its partials
        scale = float((x.float().sum() * k * g.abs().max()))
        assert abs(float(gw) - gw_sum) <= 1e-5 * max(scale, 1.0)
    only = ops.event_matvec_vjp(x, idx, w, n_post, g, need_w=False)
    assert only[1] is None and same(only[0], gs)
    if het:
        only = ops.event_matvec_vjp(x, idx, w, n_post, g, need_spk=False)
        assert only[0] is None and same(only[1], gw)


def test_shared_weight_gradient_over_many_active_rows(torch_cuda):
    """Every row active: the shared weight's gradient against float64.  A row's sum is added in
    fp32 (ceil(k / 64) + 6 roundings, each at most 2^-24 of its absolute sum), the rows of a
    workgroup in 64 bits, and at most 4,096 workgroups meet in fp32, each rounding at most 2^-24
    of the running sum, which stays below 6 root sums of squares of the rows.  Less than a typical
    row adds, so a row left out or added twice shows."""
    torch = torch_cuda
    from brainstate_amd import ops
    for n_pre, k, n_post in ((30_000, 100, 30_000), (3_000, 30, 500), (40_000, 128, 60_000)):
        gen = torch.Generator(device='cuda').manual_seed(k)
        idx = torch.randint(0, n_post, (n_pre, k), device='cuda', generator=gen, dtype=torch.int32)
        x = torch.rand(n_pre, device='cuda', generator=gen) + 0.5
        g = torch.randn(n_post, device='cuda', generator=gen)
        _, gw = ops.event_matvec_vjp(x, idx, 0.5, n_post, g)
        t = x.double()[:, None] * g.double()[idx.long()]
        rows = t.sum(1)
        bound = 2.0 ** -24 * ((-(-k // 64) + 6) * float(t.abs().sum()) +
                              4096 * 6 * float(rows.square().sum().sqrt()))
        assert bound < float(rows.abs().median())
        assert abs(float(gw) - float(t.sum())) <= bound
