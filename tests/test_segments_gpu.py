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


# rows of `length`, `m` of them, over `n` columns: workgroups per CU of SDDMM, SpMM and the one-pass
# call, 0 where nothing limits them; on both sides of every line of the rule
F64_512, F64_1K, F32_ODD, F64_RAG32, F64_RAG64 = (np.float64, 64), (np.float64, 128), (np.float32, 127), \
    (np.float64, 54), (np.float64, 100)


@pytest.mark.parametrize("dtype_k,m,n,length,want", [
    # the wide launch, by length, panel and wavefronts
    (F64_512, 40000, 133000, 16, (3, 3, 0)), (F64_512, 40000, 133000, 15, (0, 0, 0)),
    (F64_512, 40000, 133000, 23, (3, 3, 0)), (F64_512, 40000, 133000, 24, (3, 3, 3)),
    (F64_512, 40000, 49152, 24, (3, 3, 3)), (F64_512, 40000, 49151, 24, (0, 0, 0)),
    (F64_512, 32768, 133000, 24, (3, 3, 3)), (F64_512, 32766, 133000, 24, (0, 0, 0)),
    (F64_1K, 40000, 327680, 16, (3, 3, 0)), (F64_1K, 40000, 327681, 16, (0, 0, 0)),
    # rows that end inside a vector; that leave lanes of 32 and of 64 idle; too many of them
    (F32_ODD, 40000, 133000, 16, (3, 3, 0)), (F32_ODD, 40000, 133000, 24, (3, 3, 3)),
    (F64_RAG32, 40000, 133000, 31, (0, 0, 0)), (F64_RAG32, 40000, 133000, 32, (3, 3, 3)),
    (F64_RAG64, 40000, 133000, 23, (0, 0, 0)), (F64_RAG64, 40000, 133000, 24, (3, 3, 3)),
    ((np.float64, 94), 40000, 133000, 32, (0, 0, 0)), ((np.float64, 96), 40000, 133000, 32, (3, 3, 3)),
    # the short launch
    (F64_512, 40000, 133000, 6, (5, 5, 6)), (F64_512, 40000, 133000, 5, (0, 0, 0)),
    (F64_512, 40000, 131072, 6, (5, 5, 6)), (F64_512, 40000, 131071, 6, (0, 0, 0)),
    (F64_1K, 40000, 133000, 6, (5, 5, 5)), (F64_1K, 55000, 327680, 6, (5, 5, 5)),
    (F64_1K, 55000, 327681, 6, (0, 0, 0)), (F32_ODD, 40000, 133000, 6, (6, 5, 6)),
    (F64_RAG64, 40000, 133000, 6, (6, 5, 6)),
    (F64_512, 131072, 133000, 5, (0, 7, 0)), (F64_512, 131070, 133000, 5, (0, 0, 0)),
    (F64_512, 131072, 133000, 4, (0, 7, 0)), (F64_512, 131072, 133000, 3, (0, 0, 0)),
    (F64_1K, 90000, 327681, 5, (0, 7, 0)), (F32_ODD, 140000, 133000, 5, (0, 0, 0))])
def test_launches_kept_to_fewer_workgroups_per_cu(ctx, dtype_k, m, n, length, want):
    dtype, k = dtype_k
    ii, jj = rows_of([length] * m, n, length)
    touched = min(n, jj.size)
    jj[:touched] = np.arange(touched)
    want_lds = [(160 * 1024 // w) // 1024 * 1024 if w else 0 for w in want]
    S, dC = ctx.plan(m, n, ii, jj, np.ones(jj.size, dtype)), ctx.vals(jj.size, dtype)
    dA, dB, dY = (ctx.panel(r, k, dtype) for r in (m, n, m))
    assert S.info.nqueues == 1 and S.info.cols_touched == n
    for call, lds in zip((lambda: ctx.sddmm(S, dA, dB, dC), lambda: ctx.spmm(S, dB, dY),
                          lambda: ctx.sddmm_spmm(S, dA, dB, dC, dY)), want_lds):
        call()
        assert [b for _, b in launches(ctx, call)] == [lds]
    for h in (S, dA, dB, dY, dC):
        h.close()
