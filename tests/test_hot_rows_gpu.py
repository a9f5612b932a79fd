"""Hot dense rows whose numbers crowd (a power of two apart, few low bits): calls that gather them
from a copy side by side give the bits of calls that gather them where they lie."""
import numpy as np
import pytest

from spcomm3d_amd import device
from tests._launches import launches
from tests.test_parity_gpu import check_sddmm, check_spmm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with device.Context(0) as c:
        yield c


def pattern(m, n, nnz, order, crowded=True, seed=5):
    """Half of the entries in every 32nd row and column (or in as many that do not crowd), skewed."""
    rng = np.random.default_rng(seed)

    def ids(size):
        hot = (size // 32 * rng.random(nnz) ** 2).astype(np.uint32)
        hot = hot * 32 if crowded else hot * 31 % np.uint32(size)
        return np.where(rng.random(nnz) < 0.6, hot, rng.integers(0, size, nnz)).astype(np.uint32)

    ii, jj = ids(m), ids(n)
    o = np.lexsort((jj, ii)) if order == "sorted" else (
        np.lexsort((ii, jj)) if order == "column" else rng.permutation(nnz))
    return np.ascontiguousarray(ii[o]), np.ascontiguousarray(jj[o])


# 256-byte rows need 12.6 M entries, wider ones 1.5 GiB of gathers
CASES = [(np.float32, 64, 4000, 240000, 12700000, "sorted"), (np.float64, 64, 9000, 130000, 3200000, "sorted"),
         (np.float64, 64, 100000, 130000, 3200000, "shuffled"), (np.float64, 64, 120000, 130000, 3200000, "column"),
         (np.float32, 256, 3000, 70000, 1600000, "sorted"), (np.float64, 256, 3000, 36000, 800000, "sorted"),
         (np.float64, 512, 2500, 18000, 400000, "sorted")]


@pytest.mark.parametrize("dtype,k,m,n,nnz,order", CASES)
def test_copied_rows_give_the_bits_of_rows_in_place(ctx, dtype, k, m, n, nnz, order):
    ii, jj = pattern(m, n, nnz, order)
    rng = np.random.default_rng(k)
    w = np.dtype(dtype).itemsize
    vv = rng.uniform(0, 1, nnz).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)).astype(dtype) for r in (m, n, m))
    S = ctx.plan(m, n, ii, jj, vv, k_hint=k, seg_max=512)
    # the same layout, planned for rows that are no power of two
    plain = ctx.plan(m, n, ii, jj, vv, k_hint=k * 3 // 2, l2_hot_bytes=3 << 20, seg_max=512)
    sums = plain.info.npartial_slots * (k // 2) * w
    assert S.info.nsegments == plain.info.nsegments and S.info.hot_cols == plain.info.hot_cols > 0
    assert S.info.device_bytes + sums >= plain.info.device_bytes + 4 * nnz
    dA, dY, dC = ctx.panel_from(A), ctx.panel_from(Y0), ctx.vals(nnz, dtype)
    raw = ctx.panel_from(np.vstack([np.full((1, k), np.nan, dtype), B, np.full((1, k), np.nan, dtype)]))
    for off in (0, 16):  # the operand on whole lines, and 16 bytes past one
        dB = device.Panel(ctx, n, k, dtype, dev=raw.device_ptr() + k * w - off)
        if off:
            dB.upload(B)
        out = []
        for plan in (plain, S):
            dC.fill(-5.0)
            dY.upload(Y0)
            ctx.sddmm(plan, dA, dB, dC)
            C = dC.download()
            ctx.spmm(plan, dB, dY)
            Y = dY.download()
            ctx.sddmm_spmm(plan, dA, dB, dC, dY, chained=True)
            out.append((C, Y, dC.download(), dY.download()))
        for want, got in zip(*out):
            assert np.array_equal(want, got)
    check_sddmm(A, B, ii, jj, vv, out[1][0])
    check_spmm(B, ii, jj, vv, Y0, out[1][1])


# (planned for 64 columns no other width repays the copy; for 128 columns 64 do, out of the same buffer)
@pytest.mark.parametrize("k,widths", [(64, (32, 60, 128)), (128, (64, 128))])
def test_other_widths_recordings_and_the_call_without_allocations(ctx, k, widths):
    dtype, m, n, nnz, order = np.float64, 3000, 130000, 3200000, "sorted"
    ii, jj = pattern(m, n, nnz, order)
    rng = np.random.default_rng(1)
    vv = rng.uniform(0, 1, nnz).astype(dtype)
    S = ctx.plan(m, n, ii, jj, vv, k_hint=k)
    for kk in widths:
        A, B, Y0 = (rng.uniform(-1, 1, (r, kk)).astype(dtype) for r in (m, n, m))
        dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(nnz, dtype)
        ctx.sddmm(S, dA, dB, dC)
        ctx.spmm(S, dB, dY)
        C, Y = dC.download(), dY.download()
        check_sddmm(A, B, ii, jj, vv, C)
        check_spmm(B, ii, jj, vv, Y0, Y)
        dC.fill(-5.0)
        dY.upload(Y0)
        ctx.capture_begin()
        ctx.sddmm(S, dA, dB, dC)
        ctx.spmm(S, dB, dY)
        g = ctx.capture_end()
        for _ in range(2):
            dB.upload(B)
            dY.upload(Y0)
            g.launch()
            ctx.sync()
            assert np.array_equal(dC.download(), C) and np.array_equal(dY.download(), Y)
        # what a replay gathers is the operand as it is then
        dB.upload(B * 2)
        dY.upload(Y0)
        g.launch()
        assert np.array_equal(dC.download(), C * 2)
        check_spmm(B * 2, ii, jj, vv, Y0, dY.download())
        g.close()
        dB.upload(B)
        dY.upload(Y0)
        ctx.spmm_noalloc(S, dB, dY)
        assert np.array_equal(dY.download(), Y)


@pytest.mark.parametrize("k,nnz,crowded,taken", [(64, 3200000, True, True), (64, 3000000, True, False),
                                                 (64, 3200000, False, False), (62, 3400000, True, False)])
def test_where_the_line_lies(ctx, k, nnz, crowded, taken):
    m, n = 9000, 130000
    ii, jj = pattern(m, n, nnz, "sorted", crowded)
    opts = dict(seg_max=512, dtype=np.float64)
    S = ctx.plan(m, n, ii, jj, k_hint=k, l2_hot_bytes=k * 8 * 4096, **opts)
    plain = ctx.plan(m, n, ii, jj, k_hint=96, l2_hot_bytes=96 * 8 * 4096, **opts)
    assert S.info.hot_cols == plain.info.hot_cols > 0
    more = S.info.device_bytes - (plain.info.device_bytes - plain.info.npartial_slots * (96 - k) * 8)
    assert (more >= 4 * nnz) == taken


@pytest.mark.parametrize("hint,nnz,widths", [(512, 400000, {32: 0, 64: 0, 256: 0, 512: 1}),
                                             (128, 3200000, {32: 0, 64: 1, 128: 1, 256: 0})])
def test_the_copy_is_made_where_the_call_repays_it(ctx, hint, nnz, widths):
    """widths: columns of a call and how many kernels more than without hot rows it launches."""
    m, n = 2500, 130000 if hint == 128 else 18000
    ii, jj = pattern(m, n, nnz, "sorted")
    vv = np.ones(nnz)
    S = ctx.plan(m, n, ii, jj, vv, k_hint=hint, seg_max=512)
    plain = ctx.plan(m, n, ii, jj, vv, k_hint=hint * 3 // 2, l2_hot_bytes=3 << 20, seg_max=512)
    assert S.info.nsegments == plain.info.nsegments and S.info.hot_cols == plain.info.hot_cols > 0
    for k, more in widths.items():
        dA, dB, dY = (ctx.panel(r, k, np.float64) for r in (m, n, m))
        dC = ctx.vals(nnz, np.float64)
        for call in (lambda P: ctx.sddmm(P, dA, dB, dC), lambda P: ctx.spmm(P, dB, dY),
                     lambda P: ctx.sddmm_spmm(P, dA, dB, dC, dY)):
            call(S), call(plain)
            with_copy, without = (launches(ctx, lambda: call(P)) for P in (S, plain))
            assert len(with_copy) == len(without) + more, (k, with_copy, without)


@pytest.mark.parametrize("mode,order", [("all_hit", "sorted"), ("all_miss", "sorted"), ("all_hit", "column")])
def test_probed_columns_keep_the_copy(ctx, mode, order):
    """spc3d_plan_probe_columns on a plan with copied hot rows: its calls launch what they launched, hold
    the memory they held and give the bits of a plan without, probed the same way."""
    k, m, n, nnz = 64, 120000, 130000, 3200000
    ii, jj = pattern(m, n, nnz, order)
    rng = np.random.default_rng(7)
    vv = rng.uniform(0, 1, nnz)
    S = ctx.plan(m, n, ii, jj, vv, k_hint=k, seg_max=512)
    plain = ctx.plan(m, n, ii, jj, vv, k_hint=k * 3 // 2, l2_hot_bytes=3 << 20, seg_max=512)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)) for r in (m, n, m))
    dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(nnz, np.float64)
    calls = (lambda P: ctx.sddmm(P, dA, dB, dC), lambda P: ctx.spmm(P, dB, dY))
    for call in calls:
        call(S), call(plain)
    before = [launches(ctx, lambda: call(S)) for call in calls]
    assert [len(b) for b in before] == [len(launches(ctx, lambda: call(plain))) + 1 for call in calls]
    held = S.info.device_bytes
    out = []
    for plan in (plain, S):
        plan.probe_columns(mode, 2048)
        dY.upload(Y0)
        for call in calls:
            call(plan)
        out.append((dC.download(), dY.download()))
    assert all(np.array_equal(a, b) for a, b in zip(*out))
    assert [launches(ctx, lambda: call(S)) for call in calls] == before
    assert S.info.device_bytes == held


def test_plans_that_never_copy_hot_rows_hold_no_list_of_them(ctx):
    """Column blocks whose hot rows crowd: the memory of the same blocks planned for a width without."""
    m, n, nnz = 9000, 130000, 5500000
    ii, jj = pattern(m, n, nnz, "sorted")
    # no row is cut: the only memory that depends on the width would be the hot rows'
    opts = dict(seg_max=1 << 20, hub_min=1 << 20, dtype=np.float64)
    S, plain = (ctx.plan(m, n, ii, jj, k_hint=k, l2_hot_bytes=k * 8 * 1024, col_blocks=2, **opts) for k in (64, 96))
    assert S.info.ncol_blocks == plain.info.ncol_blocks == 2 and S.info.nqueues == plain.info.nqueues == 8
    assert S.info.npartial_slots == plain.info.npartial_slots == 0
    assert S.info.device_bytes == plain.info.device_bytes
    whole, plain = (ctx.plan(m, n, ii, jj, k_hint=k, l2_hot_bytes=k * 8 * 1024, **opts) for k in (64, 96))
    assert whole.info.device_bytes > plain.info.device_bytes + 4 * nnz  # (they do crowd)


def test_a_plan_without_a_width_is_for_64_columns(ctx):
    k, m, n, nnz = 64, 9000, 130000, 3200000
    ii, jj = pattern(m, n, nnz, "sorted")
    vv = np.random.default_rng(3).uniform(0, 1, nnz)
    opts = dict(seg_max=512, dtype=np.float64)
    S, hinted = ctx.plan(m, n, ii, jj, vv, **opts), ctx.plan(m, n, ii, jj, vv, k_hint=k, **opts)
    assert S.info.device_bytes == hinted.info.device_bytes > ctx.plan(m, n, ii, jj, vv, k_hint=60, l2_hot_bytes=15 << 17,
                                                                      **opts).info.device_bytes + 4 * nnz
    rng = np.random.default_rng(4)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)) for r in (m, n, m))
    dA, dB, dC, dY = ctx.panel_from(A), ctx.panel_from(B), ctx.vals(nnz, np.float64), ctx.panel_from(Y0)
    ctx.sddmm(S, dA, dB, dC)
    check_sddmm(A, B, ii, jj, vv, dC.download())
    ctx.spmm(S, dB, dY)
    check_spmm(B, ii, jj, vv, Y0, dY.download())
