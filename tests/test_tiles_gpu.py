"""Row tiles beside an ordinary plan: which calls run over them, at the edge of the rule, in both
element types, with rows left over, in arbitrary order, and under every call a plan takes."""
import numpy as np
import pytest

from spcomm3d_amd import device
from tests.test_parity_gpu import check_sddmm, check_spmm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with device.Context(0) as c:
        yield c


def pattern(lengths, n, shuffled, seed=3):
    rng = np.random.default_rng(seed)
    ii = np.repeat(np.arange(len(lengths), dtype=np.uint32), lengths)
    jj = rng.integers(0, n, ii.size).astype(np.uint32)
    if shuffled:
        o = rng.permutation(ii.size)
        ii, jj = ii[o], jj[o]
    return np.ascontiguousarray(ii), np.ascontiguousarray(jj)


# lengths of the rows, columns; 1 KB dense rows: 4 blocks of 3.25 MiB from 9985 touched columns on
ROWS_80 = [80] * 7000
MIXED = [90] * 6000 + [7] * 3000 + [0] * 10 + [300] * 30
ROWS_20 = [20] * 27000      # SDDMM only
@pytest.mark.parametrize("dtype,k", [(np.float32, 256), (np.float64, 128)])
@pytest.mark.parametrize("lengths,n,tiled", [(ROWS_80, 11000, True), (MIXED, 12001, True),
                                             (ROWS_20, 12000, True), (ROWS_80, 9000, False),
                                             ([80] * 6500, 11000, False)])
@pytest.mark.parametrize("shuffled", [False, True])
def test_calls_over_the_tiles(ctx, dtype, k, lengths, n, tiled, shuffled):
    m = len(lengths)
    ii, jj = pattern(lengths, n, shuffled)
    rng = np.random.default_rng(k)
    vv, v2 = (rng.uniform(0, 1, ii.size).astype(dtype) for _ in range(2))
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)).astype(dtype) for r in (m, n, m))
    S = ctx.plan(m, n, ii, jj, vv, k_hint=k)
    plain = ctx.plan(m, n, ii, jj, vv, k_hint=k, sweep=False)
    assert (S.info.device_bytes > plain.info.device_bytes) == tiled
    assert S.info.nsegments == plain.info.nsegments and S.info.sweep_entries == 0
    dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(ii.size, dtype)
    S.set_values(v2)
    S.set_values(vv)
    for again in range(2):  # eagerly, then recorded and replayed
        dC.fill(-5.0)
        dY.upload(Y0)
        if again:
            ctx.capture_begin()
        ctx.sddmm(S, dA, dB, dC)
        ctx.spmm(S, dB, dY)
        if again:
            g = ctx.capture_end()
            g.launch()
            ctx.sync()
            dC.fill(-5.0)
            dY.upload(Y0)
            g.launch()
        C, Y = dC.download(), dY.download()
        if again:
            assert np.array_equal(C, C1) and np.array_equal(Y, Y1)
            g.close()
        C1, Y1 = C, Y
    check_sddmm(A, B, ii, jj, vv, C)
    check_spmm(B, ii, jj, vv, Y0, Y)
    dY.upload(Y0)
    ctx.spmm_noalloc(S, dB, dY)
    assert np.array_equal(dY.download(), Y)
    dY.upload(Y0)
    ctx.sddmm_spmm(S, dA, dB, dC, dY, chained=True)
    check_sddmm(A, B, ii, jj, vv, dC.download())
    check_spmm(B, ii, jj, dC.download(), Y0, dY.download())
    w = 3  # another width
    a, b = np.ascontiguousarray(A[:, :w]), np.ascontiguousarray(B[:, :w])
    ctx.sddmm(S, ctx.panel_from(a), ctx.panel_from(b), dC)
    check_sddmm(a, b, ii, jj, vv, dC.download())
    S.close()
    plain.close()


@pytest.mark.parametrize("shuffled", [False, True])
def test_the_callers_order_is_kept_where_it_is_asked_for(ctx, shuffled):
    # SPC3D_PLAN_KEEP_ENTRY_ORDER: no tiles, which add block after block; and tiles show in the info
    k, n, m = 128, 11000, len(ROWS_80)
    ii, jj = pattern(ROWS_80, n, shuffled)
    rng = np.random.default_rng(1)
    vv = rng.uniform(0, 1, ii.size)
    B, Y0 = rng.uniform(-1, 1, (n, k)), rng.uniform(-1, 1, (m, k))
    dB, got = ctx.panel_from(B), []
    for opts in ({"keep_entry_order": True}, {"keep_entry_order": True, "sweep": False}, {}):
        S, dY = ctx.plan(m, n, ii, jj, vv, k_hint=k, **opts), ctx.panel_from(Y0)
        ctx.spmm(S, dB, dY)
        got.append((S.info, dY.download()))
        S.close()
    (kept, Y), (plain, Y_plain), (tiled, _) = got
    assert np.array_equal(Y, Y_plain) and kept.device_bytes == plain.device_bytes
    assert kept.sweep_tiles == kept.sweep_k == 0
    assert tiled.sweep_tiles > 0 and tiled.sweep_k == k and tiled.sweep_entries == 0


def test_a_plan_for_one_call_has_no_tiles(ctx):
    # one-shot calls that keep nothing: SpMM adds in the order of the ordinary plan, not by blocks
    k, n, m = 128, 11000, len(ROWS_80)
    ii, jj = pattern(ROWS_80, n, False)
    rng = np.random.default_rng(2)
    vv = rng.uniform(0, 1, ii.size)
    B, Y0 = rng.uniform(-1, 1, (n, k)), rng.uniform(-1, 1, (m, k))
    S, dY = ctx.plan(m, n, ii, jj, vv, k_hint=k, sweep=False), ctx.panel_from(Y0)
    ctx.spmm(S, ctx.panel_from(B), dY)
    S.close()
    with device.Context(0, host_cache=False) as c:
        Y = Y0.copy()
        c.spmm_host(B, ii, jj, vv, Y)
    assert np.array_equal(Y, dY.download())


# widths that leave lanes of the tiles idle or end inside a 16-byte unit, at the edges of each lane
# count (16 lanes to 256 bytes, 32 to 512, 64 to 1024), and widths that fill them
@pytest.mark.parametrize("dtype,k", [(np.float32, k) for k in (33, 36, 50, 63, 64, 65, 67, 96, 127, 128, 129,
                                                               131, 175, 252, 255)] +
                                    [(np.float64, k) for k in (17, 31, 33, 50, 63, 65, 100, 127)])
@pytest.mark.parametrize("by_column", [False, True])  # results staged, or straight to their places
def test_tiles_of_any_width(ctx, dtype, k, by_column):
    row_bytes = k * np.dtype(dtype).itemsize
    n = 11 * (13 << 18) // (3 * row_bytes)              # 4 blocks of 3.25 MiB
    nnz = max(13 * n, (545 << 20) // row_bytes)
    lengths = [80] * (nnz // 80) + [7] * 500 + [0] * 9 + [211] * 40
    lengths = np.random.default_rng(5).permutation(lengths)
    m = len(lengths)
    ii, jj = pattern(lengths, n, False)
    if by_column:
        o = np.lexsort((jj, ii))
        ii, jj = ii[o], jj[o]
    rng = np.random.default_rng(k)
    vv = rng.uniform(0, 1, ii.size).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)).astype(dtype) for r in (m, n, m))
    S = ctx.plan(m, n, ii, jj, vv, k_hint=k)
    assert S.info.sweep_tiles > 0 and S.info.sweep_entries == 0
    dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(ii.size, dtype)
    dC.fill(-5.0)
    ctx.sddmm(S, dA, dB, dC)
    ctx.spmm(S, dB, dY)
    C, Y = dC.download(), dY.download()
    check_sddmm(A, B, ii, jj, vv, C)
    check_spmm(B, ii, jj, vv, Y0, Y)
    dY.upload(Y0)
    ctx.spmm(S, dB, dY)
    assert np.array_equal(dY.download(), Y)
    # an infinity in the part of a row that two lanes load and one counts goes where it belongs only
    at, c = k - 2, int(jj[0])
    B[c, at] = np.inf
    dB.upload(B)
    dY.upload(Y0)
    ctx.sddmm(S, dA, dB, dC)
    ctx.spmm(S, dB, dY)
    C, Y = dC.download(), dY.download()
    assert not np.isnan(C).any() and np.array_equal(np.isinf(C), (jj == c) & (vv != 0))
    assert not np.isnan(Y).any()
    want = np.zeros((m, k), dtype=bool)
    want[ii[(jj == c) & (vv != 0)], at] = True
    assert np.array_equal(np.isinf(Y), want)
    for h in (S, dA, dB, dY, dC):
        h.close()
