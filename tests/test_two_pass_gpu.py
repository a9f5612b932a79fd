"""Tables of the two-pass way home (build_two_pass): counted up to 7680 tiles of 160 KiB of results,
sorted beyond."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,entries", [
    (np.float64, lambda t: 2 * t),            # the fewest
    (np.float32, lambda t: 2 * t + 1),        # a last tile of one entry
    (np.float64, lambda t: 3 * t - 1),
    (np.float32, lambda t: 1100 * t + 5),     # more tiles than threads of a block
    (np.float64, lambda t: 7680 * t),         # the last size with counters
    (np.float64, lambda t: 7680 * t + 1),     # the first with sorts
])
def test_every_result_lands_on_its_entry(ctx, dtype, entries):
    """Rows of ones: result e is value e to the bit, wherever the plan's order put the entry."""
    n = entries((160 << 10) // np.dtype(dtype).itemsize)
    rng = np.random.default_rng(n)
    rows, cols = max(300, n // 20), 512
    ii = rng.integers(0, rows, n, dtype=np.uint32)
    jj = rng.integers(0, cols, n, dtype=np.uint32)
    vv = rng.random(n, dtype=dtype)
    S = ctx.plan(rows, cols, ii, jj, vv, two_pass_min=1)
    assert S.info.two_pass_results == 1
    dA, dB = ctx.panel_from(np.ones((rows, 1), dtype)), ctx.panel_from(np.ones((cols, 1), dtype))
    dC = ctx.vals(n, dtype)
    ctx.sddmm(S, dA, dB, dC)
    assert np.array_equal(dC.download(), vv)
    for h in (S, dA, dB, dC):
        h.close()
