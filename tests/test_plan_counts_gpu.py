"""Column and row counts, and the order of staged results, as the device builder makes them, at the edges of
their buckets, parts and tiles, against the host builder and against unstaged stores."""
import ctypes

import numpy as np
import pytest

from spcomm3d_amd import device
from tests.test_plan_device_gpu import both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with device.Context(0) as c:
        yield c


# columns: up to 2^14 of them are counted without a digit of a sort, up to 2^22 after one; entries: a
# part holds 2^16, or a 64th where that is more
@pytest.mark.parametrize("ncols,nnz", [(1, 70000), (2, 65537), ((1 << 14) - 1, 65536), (1 << 14, 65535),
                                       ((1 << 14) + 1, 131073), (1 << 15, 200001), ((1 << 22) - 1, 66000),
                                       (1 << 22, 140000), ((1 << 22) + 1, 140001), (1 << 26, 65537),
                                       (5000, (1 << 22) + 67), ((1 << 20) + 7, (1 << 22) + 64 * 65)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_counts(ctx, ncols, nnz, shuffled):
    rng = np.random.default_rng(nnz)
    nrows = max(3, ncols // 3) if shuffled else 900
    ii = rng.integers(0, nrows, nnz).astype(np.uint32)
    # half of them in a few columns; the last column is there
    jj = np.where(rng.random(nnz) < 0.5, rng.integers(0, min(ncols, 40), nnz) * (ncols // 40 + 1) % ncols,
                  rng.integers(0, ncols, nnz)).astype(np.uint32)
    jj[nnz // 2] = ncols - 1
    if not shuffled:
        o = np.argsort(ii, kind="stable")
        ii, jj = ii[o], jj[o]
    P = both(ctx, nrows, ncols, ii, jj, xcd_slices=8, l2_hot_bytes=2048, hub_min=64, k_hint=16,
             keep_entry_order=shuffled)
    assert P["info"].cols_touched == np.unique(jj).size and P["info"].max_row_nnz == np.bincount(ii).max()


# a tile holds 4096 entries; rows of 300 are hub rows, whose entries are regrouped and staged, rows of 7 are not
@pytest.mark.parametrize("nnz", [600, 4095, 4096, 4097, 8191, 8192, 8193, 1 << 18, (1 << 18) + 1])
def test_staged_results_come_home(ctx, nnz):
    rng = np.random.default_rng(nnz)
    ii = np.repeat(np.arange(nnz, dtype=np.uint32), np.where(np.arange(nnz) % 2 == 0, 300, 7))[:nnz].copy()
    m, n, k = int(ii[-1]) + 1, 4000, 4
    jj = np.minimum(rng.pareto(0.6, nnz) * 4, n - 1).astype(np.uint32)
    vv = rng.uniform(0.5, 1, nnz)
    A, B = rng.uniform(-1, 1, (m, k)), rng.uniform(-1, 1, (n, k))
    dA, dB, dC, got = ctx.panel_from(A), ctx.panel_from(B), ctx.vals(nnz, np.float64), []
    for staged in (None, False):
        S = ctx.plan(m, n, ii, jj, vv, xcd_slices=8, l2_hot_bytes=256, hub_min=32, k_hint=k, staged_stores=staged)
        assert S.info.nqueues == 8
        assert (S.info.staged_entries > 0) == (staged is None)
        dC.fill(np.nan)
        ctx.sddmm(S, dA, dB, dC)
        got.append(dC.download())
        S.close()
    assert np.array_equal(got[0], got[1]) and not np.isnan(got[0]).any()


# entries that come in the order of their rows, 1024 of them to a wavefront, 64 at a time: rows that end where
# those do or next to it, go over several, and the whole pattern; hub rows from 1 entry on and from 64
@pytest.mark.parametrize("lengths", [[1024] * 5, [1023, 1, 1024, 1025, 1], [64] * 40, [63, 65, 2, 0, 300] * 30,
                                     [5000, 3, 9000, 1, 1], [20000], [1] * 500 + [2048, 7, 4096] + [2] * 300,
                                     [1, 70000, 1], [130] * 600])
@pytest.mark.parametrize("hub_min", [1, 64])
def test_rows_in_order(ctx, lengths, hub_min):
    rng = np.random.default_rng(len(lengths))
    ii = np.repeat(np.arange(len(lengths), dtype=np.uint32), lengths)
    n = 4000
    jj = np.minimum(rng.pareto(0.6, ii.size) * 4, n - 1).astype(np.uint32)
    P = both(ctx, len(lengths), n, ii, jj, xcd_slices=8, l2_hot_bytes=256, hub_min=hub_min, k_hint=4, seg_max=500)
    assert P["info"].nqueues == 8 and P["info"].hub_rows == sum(v >= hub_min for v in lengths)
    both(ctx, len(lengths), n, ii, jj, xcd_slices=1)


# the longest row that is placed without a sort, and the shortest that makes the plan sort its entries
@pytest.mark.parametrize("longest", [1 << 24, (1 << 24) + 1])
def test_longest_row_in_order(ctx, longest):
    lengths = [3, 700, longest, 1, 200000, 64]
    ii = np.repeat(np.arange(len(lengths), dtype=np.uint32), lengths)
    n = 4000
    jj = np.minimum(np.random.default_rng(5).pareto(0.6, ii.size) * 4, n - 1).astype(np.uint32)
    P = both(ctx, len(lengths), n, ii, jj, xcd_slices=8, l2_hot_bytes=256, hub_min=64, k_hint=4)
    assert P["info"].nqueues == 8 and P["info"].hub_rows == 4


def test_scratch_of_a_pattern_in_order():
    # The pool of a fresh context keeps what making a plan took.  Per entry that is the ids and the scratch of one
    # digit of their sort (8 bytes), half a byte for the primitives, and the kernel order, which is the caller's and
    # goes back (4): less than 14.  Rows, columns and counters: under 64 MiB.
    n, deg = 1 << 17, 512
    jj = np.random.default_rng(0).integers(0, n, n * deg, dtype=np.uint32)
    with device.Context(0) as c:
        free, total = ctypes.c_size_t(), ctypes.c_size_t()

        def used():
            c.sync()
            assert c._lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
            return total.value - free.value

        dii, djj = c.vals(jj.size, np.float32), c.vals(jj.size, np.float32)
        dii.upload(np.repeat(np.arange(n, dtype=np.uint32), deg).view(np.float32))
        djj.upload(jj.view(np.float32))
        small = device.Plan.from_device(c, n, n, dii, djj, 1000, np.float32)
        before = used()
        S = device.Plan.from_device(c, n, n, dii, djj, jj.size, np.float32, col_blocks=1, sweep=False)
        assert S.info.order_is_identity and S.info.nqueues == 1
        assert used() - before - S.info.device_bytes <= jj.size * 14 + (64 << 20)
        for h in (S, small, dii, djj):
            h.close()
