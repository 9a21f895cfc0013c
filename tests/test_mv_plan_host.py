"""Which mat-vec calls may sum in LDS, seen from the workspace they ask for (CPU: the size query
needs no device; a single-launch plan asks for none and is not listed)."""
import pytest

from brainstate_amd import _native as N


@pytest.mark.parametrize('batch,n_pre,k,n_post,count,planned', [
    (1, 100_000, 1000, 100_000, 0, True), (1, 250_000, 100, 4000, 0, True),
    (1, 10_000, 100, 10_000, 0, False),            # few synapses: atomics
    (1, 100_000, 250, 100_000, 1, False),          # ... of a shared weight up to 5e7
    (1, 250_000, 250, 100_000, 1, True),
    (1, 100_000, 1000, 128_001, 0, False),         # more than 8 ranges
    (8, 20_000, 100, 20_000, 0, True), (16, 2000, 20, 128_000, 0, False),
    (8, 20_000, 20, 100_000, 0, False),            # LDS would not win at any density
    (128, 200_000, 100, 20_000, 0, True),          # one row group, many spans: a header each
    # few long rows: few workgroups to add them by atomics
    (1, 200, 200_000, 50_000, 0, True), (1, 4000, 10_000, 100_000, 0, True),
    (1, 1, (1 << 30) - 1, 100, 0, False), (0, 5, 5, 5, 0, False), (1, 0, 5, 5, 0, False)])
def test_planned_calls(batch, n_pre, k, n_post, count, planned):
    size = N.lib().bs_matvec_workspace_size(batch, n_pre, k, n_post, count)
    assert (size > 0) == planned
    assert size % 256 == 0 or n_post % 64
    assert size <= batch * 256 + 512 * n_post * 4   # partial sums of at most 512 workgroups
