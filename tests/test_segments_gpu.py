"""The default longest segment by rows and width, the fix-up's runs of slots, and rows just
below and at the length from which a pattern of short segments takes the wide launch."""
import numpy as np
import pytest

from spcomm3d_amd import device
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
# workgroups per CU, and with a chunk of segments left over
@pytest.mark.parametrize("dtype,k", [(np.float64, 64), (np.float32, 127)])
@pytest.mark.parametrize("m,length", [(32767, 16), (32768, 16), (32771, 17), (32768, 6), (200001, 16)])
def test_even_rows_over_a_large_panel(ctx, dtype, k, m, length):
    n = 132000
    ii, jj = rows_of([length] * m, n, length)
    jj[:n] = np.arange(n)  # every column is touched
    rng = np.random.default_rng(m)
    vv = rng.uniform(0, 1, ii.size).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)).astype(dtype) for r in (m, n, m))
    check_sddmm(A, B, ii, jj, vv, gpu_sddmm(ctx, m, n, ii, jj, vv, A, B))
    check_spmm(B, ii, jj, vv, Y0, gpu_spmm(ctx, m, n, ii, jj, vv, B, Y0))
