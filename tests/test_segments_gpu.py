"""The default longest segment by rows and width, the fix-up's runs of slots, and rows just
below and at the length from which a pattern of short segments takes the wide launch."""
import numpy as np
import pytest

from spcomm3d_amd import device
from tests._launches import launches
from tests.test_parity_gpu import check_sddmm, check_spmm, gpu_sddmm, gpu_spmm, rand_case
from tests.test_plan_device_gpu import both

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with device.Context(0) as c:
        yield c


def rows_of(lengths, n, seed):
    rng = np.random.default_rng(seed)
    ii = np.repeat(np.arange(len(lengths), dtype=np.uint32), lengths)
    return ii, rng.integers(0, n, ii.size).astype(np.uint32)


@pytest.mark.parametrize("k_hint", [1, 16, 17, 64, 400])
@pytest.mark.parametrize("lengths,whole", [([25] * 400, True), ([128] * 80, True), ([129] * 80, False),
                                           ([3] * 300 + [90] * 2, False)])
def test_even_short_rows_stay_whole(ctx, k_hint, lengths, whole):
    ii, jj = rows_of(lengths, 500, 1)
    plan = both(ctx, len(lengths), 500, ii, jj, k_hint=k_hint)
    assert (plan["info"].nsplit_rows == 0) == whole


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("k", [1, 8, 17, 64, 150, 600])
@pytest.mark.parametrize("seg_max,hub", [(1, 5), (1, 900), (7, 900), (16, 2500)])
def test_rows_of_few_and_of_many_slots(ctx, dtype, k, seg_max, hub):
    ii, jj, vv, A, B, Y0 = rand_case(31 + k, 50, 200, k, 3000, dtype, hub=hub)
    check_spmm(B, ii, jj, vv, Y0, gpu_spmm(ctx, 50, 200, ii, jj, vv, B, Y0, seg_max=seg_max))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("k", [2, 16, 33, 64, 130])
@pytest.mark.parametrize("length", [4, 9, 11, 12, 13, 15])
def test_uniform_short_rows(ctx, dtype, k, length):
    m, n = 203, 150
    ii, jj = rows_of([length] * m, n, length)
    rng = np.random.default_rng(k)
    vv = rng.uniform(0, 1, ii.size).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)).astype(dtype) for r in (m, n, m))
    check_sddmm(A, B, ii, jj, vv, gpu_sddmm(ctx, m, n, ii, jj, vv, A, B))
    check_spmm(B, ii, jj, vv, Y0, gpu_spmm(ctx, m, n, ii, jj, vv, B, Y0))


# even rows over a panel of 64 MiB, a workgroup either side of the launch that is kept to fewer
# workgroups per CU, and with a chunk of segments left over; rows that fill 32 lanes and 64, that end
# inside their last vector, and that leave lanes of 64 idle
@pytest.mark.parametrize("dtype,k,n", [(np.float64, 64, 132000), (np.float32, 127, 133000),
                                       (np.float64, 100, 84000), (np.float64, 128, 66000)])
@pytest.mark.parametrize("m,length", [(32767, 16), (32768, 16), (32771, 17), (32768, 6), (32768, 24),
                                      (200001, 16)])
def test_even_rows_over_a_large_panel(ctx, dtype, k, n, m, length):
    ii, jj = rows_of([length] * m, n, length)
    jj[:n] = np.arange(n)  # every column is touched
    rng = np.random.default_rng(m)
    vv = rng.uniform(0, 1, ii.size).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)).astype(dtype) for r in (m, n, m))
    C = gpu_sddmm(ctx, m, n, ii, jj, vv, A, B)
    check_sddmm(A, B, ii, jj, vv, C)
    check_spmm(B, ii, jj, vv, Y0, gpu_spmm(ctx, m, n, ii, jj, vv, B, Y0))
    S, dC = ctx.plan(m, n, ii, jj, vv), ctx.vals(ii.size, dtype)
    dA, dB, dY = (ctx.panel_from(x) for x in (A, B, Y0))
    ctx.sddmm_spmm(S, dA, dB, dC, dY, chained=True)
    assert np.array_equal(dC.download(), C)
    check_spmm(B, ii, jj, C, Y0, dY.download())
    for h in (S, dA, dB, dY, dC):
        h.close()


# rows of (how many, how long) over `n` columns: workgroups per CU of every launch of SDDMM, SpMM and the
# one-pass call, 0 where nothing limits them; on both sides of every line of the rule
F64_512, F64_1K, F64_2K, F32_ODD, F64_ODD1K, F64_ODD2K = (np.float64, 64), (np.float64, 128), \
    (np.float64, 256), (np.float32, 127), (np.float64, 127), (np.float64, 255)
# rows that leave lanes idle: 24 and 27 of 32 busy, 47, 48 and 50 of 64, 65 and 100 of 128, 130 and 200 of 256
IDLE24, IDLE27, IDLE47, IDLE48, IDLE50, IDLE65, IDLE100, IDLE130, IDLE200 = (
    (np.float64, 2 * n) for n in (24, 27, 47, 48, 50, 65, 100, 130, 200))


@pytest.mark.parametrize("dtype_k,n,rows,want", [
    # the wide launch, by length, panel, wavefronts and lanes
    (F64_512, 133000, [(40000, 12)], (3, 3, 3)), (F64_512, 133000, [(40000, 15)], (3, 3, 3)),
    (F64_512, 133000, [(40000, 16)], (2, 2, 3)), (F64_512, 133000, [(40000, 23)], (2, 2, 3)),
    (F64_512, 133000, [(40000, 31)], (2, 2, 3)), (F64_512, 133000, [(40000, 32)], (2, 2, 2)),
    (F64_512, 49152, [(40000, 32)], (2, 2, 2)), (F64_512, 49151, [(40000, 32)], (3, 3, 3)),
    (F64_512, 32768, [(40000, 32)], (3, 3, 3)), (F64_512, 32767, [(40000, 32)], (0, 0, 0)),
    (F64_512, 133000, [(32768, 32)], (2, 2, 2)), (F64_512, 133000, [(32766, 32)], (0, 0, 0)),
    (F64_1K, 133000, [(40000, 23)], (2, 2, 3)), (F64_1K, 133000, [(40000, 24)], (2, 2, 2)),
    (F64_1K, 327680, [(40000, 16)], (2, 2, 3)),
    (F64_1K, 327681, [(40000, 16)], (0, 3, 0)), (F64_1K, 327681, [(20032, 8), (20032, 24)], (0, 0, 0)),
    (F32_ODD, 133000, [(40000, 16)], (2, 2, 3)), (F32_ODD, 133000, [(40000, 32)], (2, 2, 2)),
    (IDLE27, 133000, [(40000, 31)], (3, 3, 3)), (IDLE27, 133000, [(40000, 32)], (2, 2, 2)),
    (IDLE50, 133000, [(40000, 23)], (3, 3, 3)), (IDLE50, 133000, [(40000, 24)], (2, 2, 3)),
    (IDLE50, 133000, [(40000, 32)], (2, 2, 2)), (IDLE100, 50000, [(20032, 23)], (3, 3, 3)),
    (IDLE100, 50000, [(20032, 24)], (2, 2, 2)), (IDLE47, 133000, [(40000, 15)], (0, 0, 0)),
    (IDLE47, 44621, [(40000, 16)], (0, 3, 0)), (IDLE47, 44620, [(40000, 16)], (0, 0, 0)),
    (IDLE65, 40000, [(20032, 16)], (0, 3, 3)), (IDLE65, 16132, [(20032, 16)], (0, 0, 3)),
    (IDLE65, 16131, [(20032, 16)], (0, 0, 0)),
    (IDLE48, 133000, [(40000, 32)], (2, 2, 2)), ((np.float64, 16), 200000, [(140032, 16)], (2, 2, 0)),
    ((np.float64, 16), 200000, [(140032, 12)], (0, 0, 0)),
    # rows of mixed lengths, all of them in one launch and in two
    (F64_512, 133000, [(20032, 8), (20032, 24)], (3, 3, 3)), (F64_512, 133000, [(36032, 8), (4032, 24)], (0, 3, 0)),
    (F64_512, 133000, [(36032, 7), (4032, 16)], (0, 0, 0)),
    (F64_512, 133000, [(200000, 8), (200000, 24)], ((3, 4), (3, 4), (3, 6))),
    (F64_512, 133000, [(180032, 7), (40000, 20)], ((0, 0), (3, 0), (0, 0))),
    (F64_512, 133000, [(180032, 7), (23040, 20)], ((4, 0), (4, 0), (6, 0))),
    # the short launch, one vector per lane
    (F64_512, 133000, [(40000, 11)], (4, 4, 6)), (F64_512, 133000, [(40000, 6)], (4, 4, 6)),
    (F64_512, 133000, [(40000, 5)], (0, 0, 0)), (F64_512, 131072, [(40000, 6)], (4, 4, 6)),
    (F64_512, 131071, [(40000, 6)], (0, 0, 0)), (F64_1K, 133000, [(40000, 6)], (4, 4, 4)),
    (F64_1K, 327680, [(60000, 6)], (4, 4, 4)), (F64_1K, 327681, [(60000, 6)], (0, 0, 5)),
    (F64_1K, 133000, [(40000, 5)], (0, 0, 5)), (F64_1K, 133000, [(40000, 4)], (0, 0, 0)),
    (F64_1K, 8192, [(40000, 5)], (0, 0, 5)), (F64_1K, 8191, [(40000, 5)], (0, 0, 0)),
    (F64_ODD1K, 16514, [(40000, 5)], (0, 0, 5)), (F64_ODD1K, 16513, [(40000, 5)], (0, 0, 0)),
    (F32_ODD, 133000, [(40000, 6)], (4, 4, 6)), (F32_ODD, 133000, [(40000, 12)], (4, 4, 4)),
    (IDLE27, 156000, [(40000, 6)], (6, 4, 6)), (IDLE24, 180000, [(40000, 6)], (0, 5, 6)),
    (IDLE50, 133000, [(40000, 5)], (0, 6, 0)), (IDLE50, 133000, [(40000, 6)], (6, 6, 6)),
    (IDLE50, 133000, [(40000, 8)], (6, 4, 6)), (IDLE50, 133000, [(40000, 12)], (6, 4, 5)),
    (IDLE50, 41944, [(40000, 6)], (0, 6, 6)), (IDLE50, 41943, [(40000, 6)], (0, 0, 0)),
    (IDLE50, 31458, [(40000, 12)], (0, 0, 5)), (IDLE50, 31457, [(40000, 12)], (0, 0, 0)),
    (IDLE50, 419431, [(80000, 6)], (0, 6, 0)), (IDLE50, 419431, [(80000, 12)], (0, 6, 5)),
    (F64_512, 133000, [(131072, 5)], (0, 7, 0)), (F64_512, 133000, [(131070, 5)], (0, 0, 0)),
    (F64_512, 133000, [(131072, 4)], (0, 7, 0)), (F64_512, 133000, [(131072, 3)], (0, 0, 0)),
    (F64_1K, 327681, [(90000, 5)], (0, 7, 5)), (F32_ODD, 133000, [(140000, 5)], (0, 0, 0)),
    # the short launch, longer rows
    (F64_2K, 4096, [(20000, 3)], (0, 0, 4)), (F64_2K, 4095, [(20000, 3)], (0, 0, 0)),
    (F64_2K, 4096, [(20000, 2)], (0, 0, 0)), (F64_2K, 40000, [(20000, 6)], (4, 4, 4)),
    (F64_ODD2K, 16449, [(20000, 3)], (0, 0, 5)), (F64_ODD2K, 16448, [(20000, 3)], (0, 0, 0)),
    (F64_ODD2K, 40000, [(20000, 6)], (4, 4, 5)), (IDLE100, 20972, [(20000, 7)], (0, 6, 5)),
    (IDLE100, 20971, [(20000, 7)], (0, 0, 0)), (IDLE100, 20972, [(20000, 3)], (0, 0, 5)),
    (IDLE100, 20972, [(20000, 2)], (0, 0, 0)), (IDLE65, 40000, [(20000, 6)], (0, 0, 0)),
    (IDLE100, 50000, [(20000, 7)], (6, 4, 5)), (IDLE65, 40000, [(20000, 7)], (0, 0, 5)),
    (IDLE200, 5243, [(20000, 3)], (0, 0, 4)), (IDLE200, 5242, [(20000, 3)], (0, 0, 0)),
    ((np.float64, 401), 5230, [(20000, 3)], (0, 0, 4)), (IDLE130, 8066, [(20000, 7)], (0, 0, 4)),
    (IDLE130, 8066, [(20000, 6)], (0, 0, 0)), (IDLE130, 8065, [(20000, 7)], (0, 0, 0))])
def test_launches_kept_to_fewer_workgroups_per_cu(ctx, dtype_k, n, rows, want):
    dtype, k = dtype_k
    lengths = np.repeat([length for _, length in rows], [count for count, _ in rows])
    m = lengths.size
    ii, jj = rows_of(lengths, n, m)
    jj[:n] = np.arange(n)  # every column is touched
    S, dC = ctx.plan(m, n, ii, jj, np.ones(jj.size, dtype)), ctx.vals(jj.size, dtype)
    dA, dB, dY = (ctx.panel(r, k, dtype) for r in (m, n, m))
    assert S.info.nqueues == 1 and S.info.cols_touched == n and S.info.nsegments == m
    for call, limits in zip((lambda: ctx.sddmm(S, dA, dB, dC), lambda: ctx.spmm(S, dB, dY),
                             lambda: ctx.sddmm_spmm(S, dA, dB, dC, dY)), want):
        call()
        got = [lds for _, lds in launches(ctx, call)]
        limits = limits if isinstance(limits, tuple) else (limits,)
        assert len(got) == len(limits)
        for lds, limit in zip(sorted(got, reverse=True), limits):
            # a CU's 160 KiB in pieces of 1280 bytes: as many fit as said, and one more does not
            pieces = -(-lds // 1280)
            assert (128 // pieces if pieces else 0) == limit, (got, limits)
    for h in (S, dA, dB, dY, dC):
        h.close()
