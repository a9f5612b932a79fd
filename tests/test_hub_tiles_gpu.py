"""Tiles of the longest rows beside a sliced plan: skewed patterns just large enough for them, in every order of the
entries, in widths that fill the tiles' lanes and that do not, against the oracle and the plan without tiles."""
import numpy as np
import pytest

from spcomm3d_amd import _capi as capi
from spcomm3d_amd import device
from spcomm3d_amd import workloads as W
from tests._launches import launches
from tests.test_parity_gpu import check_sddmm, check_spmm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with device.Context(0) as c:
        yield c


@pytest.fixture(scope="module")
def patterns():
    made = {}

    def get(scale, edges, order):
        if (scale, edges) not in made:
            made.clear()
            made[scale, edges] = W.rmat(scale, edges, 1)
        w = made[scale, edges]
        ii, jj = w.ii, w.jj
        rng = np.random.default_rng(scale)
        if order == "runs":      # every row's entries lie together, rows and columns renumbered
            ii = rng.permutation(w.nrows).astype(np.uint32)[ii]
            jj = rng.permutation(w.ncols).astype(np.uint32)[jj]
        elif order != "sorted":
            o = rng.permutation(ii.size) if order == "shuffled" else np.lexsort((ii, jj))
            ii, jj = ii[o], jj[o]
        return w.nrows, np.ascontiguousarray(ii), np.ascontiguousarray(jj)

    return get


def some_rows(ii, m):
    """The entries of the longest rows, of 300 others and of short ones, and those rows' new numbers."""
    deg = np.bincount(ii, minlength=m)
    rng = np.random.default_rng(0)
    rows = np.unique(np.concatenate([np.argsort(deg)[-6:], rng.integers(0, m, 300),
                                     np.flatnonzero((deg > 0) & (deg < 9))[:300]]))
    at = np.flatnonzero(np.isin(ii, rows))
    return rows, at, np.searchsorted(rows, ii[at]).astype(np.uint32)


CASES = [(np.float64, 128, 17, 28), (np.float32, 250, 17, 28), (np.float64, 67, 18, 32), (np.float32, 100, 18, 32),
         (np.float32, 64, 19, 24)]


@pytest.mark.parametrize("order", ["sorted", "shuffled", "runs", "column"])
@pytest.mark.parametrize("dtype,k,scale,edges", CASES)
def test_calls_over_tiles_of_the_longest_rows(ctx, patterns, dtype, k, scale, edges, order):
    m, ii, jj = patterns(scale, edges, order)
    nnz, w = ii.size, np.dtype(dtype).itemsize
    assert nnz * k * w >= 5 << 29
    rng = np.random.default_rng(k)
    vv = rng.uniform(0.5, 1, nnz).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (m, k)).astype(dtype) for _ in range(3))
    S, plain = ctx.plan(m, m, ii, jj, vv, k_hint=k), ctx.plan(m, m, ii, jj, vv, k_hint=k, sweep=False)
    assert S.info.nqueues == 8 and S.info.nsegments == plain.info.nsegments
    assert S.info.device_bytes > plain.info.device_bytes + nnz * (10 + w // 2)
    dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(nnz, dtype)

    def step(P, chained=None):
        dC.fill(-5.0)
        dY.upload(Y0)
        if chained is not None:
            ctx.sddmm_spmm(P, dA, dB, dC, dY, chained=chained)
        else:
            ctx.sddmm(P, dA, dB, dC)
            ctx.spmm(P, dB, dY)
        return dC.download(), dY.download()

    C, Y = step(S)
    C0, Y1 = step(plain)
    rows, at, sub = some_rows(ii, m)
    assert (np.bincount(ii).max() > max(64, nnz // 8192))  # one is cut
    check_sddmm(A[rows], B, sub, jj[at], vv[at], C[at])
    check_spmm(B, sub, jj[at], vv[at], Y0[rows], Y[rows])
    # all of it: either side is within (terms) eps of the exact sum of terms below 1 and the start below 1
    eps = np.finfo(dtype).eps
    assert np.abs(C - C0).max() <= 2 * (k + 1) * eps * k
    terms = np.bincount(ii, minlength=m)[:, None] + 1
    assert (np.abs(Y - Y1) <= 2 * terms * terms * eps).all()
    # the same bits call after call, recorded and replayed, and without an allocation (refused where the
    # ordinary plan's partial sums are too many, as without tiles)
    ctx.capture_begin()
    ctx.sddmm(S, dA, dB, dC)
    ctx.spmm(S, dB, dY)
    g = ctx.capture_end()
    for _ in range(3):
        dC.fill(-5.0)
        dY.upload(Y0)
        g.launch()
        assert np.array_equal(dC.download(), C) and np.array_equal(dY.download(), Y)
    g.close()
    refused = []
    for P, want in ((S, Y), (plain, Y1)):
        dY.upload(Y0)
        try:
            ctx.spmm_noalloc(P, dB, dY)
            refused.append(False)
            assert np.array_equal(dY.download(), want)
        except capi.Spc3dError as e:
            assert "NOALLOC_SCRATCH" in str(e)
            refused.append(True)
    assert refused[0] == refused[1]
    # calls that do not run over the tiles: in one pass, and of another width
    for a, b in zip(step(S, chained=True), step(plain, chained=True)):
        assert np.array_equal(a, b)
    # other values
    vv2 = (vv * 0.5 + 1).astype(dtype)
    S.set_values(vv2)
    C, Y = step(S)
    check_sddmm(A[rows], B, sub, jj[at], vv2[at], C[at])
    check_spmm(B, sub, jj[at], vv2[at], Y0[rows], Y[rows])
    # an infinity, in the part of a row that two lanes load and one counts, goes where it belongs only
    c, x = int(jj[at[0]]), k - 2
    B[c, x] = np.inf
    dB.upload(B)
    C, Y = step(S)
    assert not np.isnan(C).any() and np.array_equal(np.isinf(C), jj == c)
    want = np.zeros((m, k), dtype=bool)
    want[ii[jj == c], x] = True
    assert not np.isnan(Y).any() and np.array_equal(np.isinf(Y), want)
    v = 3  # another width
    a, b = ctx.panel_from(np.ascontiguousarray(A[:, :v])), ctx.panel_from(np.ascontiguousarray(A[:, 1:v + 1]))
    plain.set_values(vv2)
    got = []
    for P in (S, plain):
        y = ctx.panel_from(np.ascontiguousarray(Y0[:, :v]))
        ctx.sddmm(P, a, b, dC)
        ctx.spmm(P, b, y)
        got.append((dC.download(), y.download()))
    assert np.array_equal(got[0][0], got[1][0]) and np.array_equal(got[0][1], got[1][1])
    for h in (S, plain, dA, dB, dY, dC, a, b):
        h.close()


def test_where_there_are_none(ctx, patterns):
    # a few too few bytes of gathers, an order to be kept, or segments of a given length
    m, ii, jj = patterns(17, 28, "shuffled")
    vv = np.ones(ii.size)
    k = -(-(5 << 29) // (ii.size * 8))
    size = {}
    for name, opts in {"none": dict(k_hint=k, sweep=False), "tiles": dict(k_hint=k), "less": dict(k_hint=k - 1),
                       "less_none": dict(k_hint=k - 1, sweep=False), "kept": dict(k_hint=k, keep_entry_order=True),
                       "kept_none": dict(k_hint=k, keep_entry_order=True, sweep=False),
                       "cut": dict(k_hint=k, seg_max=512), "cut_none": dict(k_hint=k, seg_max=512, sweep=False)}.items():
        S = ctx.plan(m, m, ii, jj, vv, **opts)
        size[name] = S.info.device_bytes
        S.close()
    assert size["tiles"] > size["none"]
    assert size["less"] == size["less_none"] and size["kept"] == size["kept_none"]
    assert size["cut"] == size["cut_none"]


# Which calls run over the tiles, on either side of every line of the rule: few blocks of columns, rows that leave a
# third of their lanes idle, rows of up to 256 bytes, results of two passes, and plans that have them for one call only
# (A: SDDMM, B: SpMM).
RULE = [(np.float64, 80, 16, 120, {o: "" for o in ("sorted", "runs", "shuffled", "column")}),
        (np.float64, 100, 17, 40, {"sorted": "AB", "runs": "AB", "shuffled": "B", "column": "AB"}),
        (np.float64, 120, 17, 40, {"shuffled": "AB"}),
        (np.float32, 200, 17, 40, {"sorted": "AB", "shuffled": "AB"}),
        (np.float64, 67, 18, 32, {"sorted": "AB", "runs": "AB", "shuffled": "B", "column": "AB"}),
        (np.float32, 134, 18, 32, {"runs": "AB", "shuffled": "B"}),
        (np.float64, 80, 18, 20, {"sorted": "", "shuffled": ""}),  # gathers of less than 3 GiB
        (np.float32, 168, 19, 20, {"shuffled": "AB"}),             # blocks enough for results of two passes
        (np.float64, 42, 19, 24, {"sorted": "A", "runs": "", "shuffled": "", "column": "A"}),
        (np.float64, 43, 19, 24, {"sorted": "AB", "runs": "AB", "shuffled": ""}),
        (np.float64, 64, 19, 28, {"shuffled": "AB"}),
        (np.float32, 85, 19, 24, {"sorted": "A", "runs": "", "shuffled": "", "column": "A"}),
        (np.float32, 86, 19, 24, {"runs": "AB", "shuffled": "AB", "column": "A"}),
        (np.float64, 32, 19, 24, {"sorted": "AB", "runs": "", "shuffled": "", "column": "A"}),
        (np.float32, 64, 19, 24, {"runs": "AB", "column": "A"}),
        (np.float64, 32, 19, 28, {"sorted": "A"}),  # from 3 GiB on hot rows are copied
        (np.float32, 64, 19, 28, {"sorted": "AB"}),
        (np.float32, 128, 20, 12, {"column": "AB"}),  # blocks enough for one call alone
        (np.float32, 85, 20, 26, {"runs": "A"}),
        # 512 and 1024 bytes, hot rows copied and (their numbers drawn anew) not
        (np.float64, 64, 19, 28, {"sorted": "AB", "runs": "AB"}),
        (np.float32, 128, 19, 28, {"sorted": "AB", "runs": "AB"}),
        (np.float64, 128, 18, 28, {"runs": "AB"}),
        (np.float32, 256, 18, 28, {"sorted": "AB", "runs": "AB"}),
        # the workload of the benchmark, planned for its width
        (np.float64, 64, 20, 16, {"sorted": "AB", "runs": "AB", "shuffled": "AB", "column": "AB"}),
        (np.float32, 64, 20, 16, {"sorted": "AB", "shuffled": "AB", "column": "A"})]


@pytest.mark.parametrize("dtype,k,scale,edges,order,over", [(*c, o, over) for *c, orders in RULE
                                                            for o, over in orders.items()])
def test_calls_that_run_over_tiles(ctx, patterns, dtype, k, scale, edges, order, over):
    m, ii, jj = patterns(scale, edges, order)
    nnz = ii.size
    assert nnz * k * np.dtype(dtype).itemsize >= 5 << 29
    rng = np.random.default_rng(k)
    vv = rng.uniform(0.5, 1, nnz).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (m, k)).astype(dtype) for _ in range(3))
    S, plain = ctx.plan(m, m, ii, jj, vv, k_hint=k), ctx.plan(m, m, ii, jj, vv, k_hint=k, sweep=False)
    assert (S.info.device_bytes > plain.info.device_bytes) == (over != "")
    dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(nnz, dtype)
    dC.fill(-5.0)
    ctx.sddmm(S, dA, dB, dC)
    ctx.spmm(S, dB, dY)
    rows, at, sub = some_rows(ii, m)
    check_sddmm(A[rows], B, sub, jj[at], vv[at], dC.download()[at])
    check_spmm(B, sub, jj[at], vv[at], Y0[rows], dY.download()[rows])
    ctx.sddmm(plain, dA, dB, dC)
    ctx.spmm(plain, dB, dY)
    for name, call in (("A", lambda P: ctx.sddmm(P, dA, dB, dC)), ("B", lambda P: ctx.spmm(P, dB, dY))):
        assert (launches(ctx, lambda: call(S)) != launches(ctx, lambda: call(plain))) == (name in over), name
    for h in (S, plain, dA, dB, dY, dC):
        h.close()


@pytest.mark.parametrize("dtype,k,scale,edges,order", [(np.float64, 64, 19, 28, "sorted"), (np.float32, 128, 19, 28, "shuffled"),
                                                       (np.float32, 64, 19, 24, "runs"), (np.float64, 64, 19, 24, "column")])
def test_probed_columns(ctx, patterns, dtype, k, scale, edges, order):
    """spc3d_plan_probe_columns on a plan that holds tiles, hot rows copied and not: its calls run over them as before,
    and compute the pattern (ii, jj % modulus), or one of columns that are all there."""
    m, ii, jj = patterns(scale, edges, order)
    nnz, modulus = ii.size, 997
    rng = np.random.default_rng(5)
    vv = rng.uniform(0.5, 1, nnz).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (m, k)).astype(dtype) for _ in range(3))
    S = ctx.plan(m, m, ii, jj, vv, k_hint=k)
    dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(nnz, dtype)
    calls = (lambda: ctx.sddmm(S, dA, dB, dC), lambda: ctx.spmm(S, dB, dY))
    for call in calls:
        call()
    before, held = [launches(ctx, call) for call in calls], S.info.device_bytes
    rows, at, sub = some_rows(ii, m)
    for again in range(2):
        S.probe_columns("all_hit", modulus)
        dY.upload(Y0)
        for call in calls:
            call()
        if order != "column":
            check_sddmm(A[rows], B, sub, (jj[at] % modulus).astype(np.uint32), vv[at], dC.download()[at])
        else:  # SDDMM exchanges rows and columns: it is the rows that are taken modulo
            check_sddmm(A, B[jj[at]], (ii[at] % modulus).astype(np.uint32), np.arange(at.size, dtype=np.uint32), vv[at],
                        dC.download()[at])
        check_spmm(B, sub, (jj[at] % modulus).astype(np.uint32), vv[at], Y0[rows], dY.download()[rows])
        assert [launches(ctx, call) for call in calls] == before and S.info.device_bytes == held
    S.probe_columns("all_miss")
    dY.upload(Y0)
    for call in calls:
        call()
    assert np.isfinite(dC.download()).all() and np.isfinite(dY.download()).all()
    for h in (S, dA, dB, dY, dC):
        h.close()
