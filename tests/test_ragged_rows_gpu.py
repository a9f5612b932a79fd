"""Dense rows of whole vectors that leave lanes of their group idle: at the edges of every lane count,
over segments of every batch size, and with what the idle lanes load (the row's last vector) infinite."""
import numpy as np
import pytest

from spcomm3d_amd import device
from tests.test_parity_gpu import check_sddmm, check_spmm, gpu_sddmm, gpu_spmm

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    with device.Context(0) as c:
        yield c


# vectors per row: 32, 64, 64 x 2 and 64 x 4 lanes, from the first of each range to the last
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("nvec", [17, 24, 31, 33, 50, 63, 65, 96, 127, 129, 191, 192, 193, 255])
def test_widths_of_every_lane_count(ctx, dtype, nvec):
    k = nvec * 16 // np.dtype(dtype).itemsize
    rng = np.random.default_rng(nvec)
    lengths = [1, 2, 3, 4, 5, 8, 9, 12, 16, 17, 31, 40, 100, 0, 7]  # exact, masked and short batches
    m, n = len(lengths), 60
    ii = np.repeat(np.arange(m, dtype=np.uint32), lengths)
    jj = rng.integers(1, n, ii.size).astype(np.uint32)
    vv = rng.uniform(0.5, 1, ii.size).astype(dtype)
    A, B, Y0 = (rng.uniform(-1, 1, (r, k)).astype(dtype) for r in (m, n, m))
    for seg_max in (20, 4096):
        S = ctx.plan(m, n, ii, jj, vv, seg_max=seg_max)
        dA, dB, dY, dC = ctx.panel_from(A), ctx.panel_from(B), ctx.panel_from(Y0), ctx.vals(ii.size, dtype)
        ctx.sddmm(S, dA, dB, dC)
        check_sddmm(A, B, ii, jj, vv, dC.download())
        ctx.spmm(S, dB, dY)
        check_spmm(B, ii, jj, vv, Y0, dY.download())
        dY.upload(Y0)
        ctx.sddmm_spmm(S, dA, dB, dC, dY, chained=True)
        check_sddmm(A, B, ii, jj, vv, dC.download())
        check_spmm(B, ii, jj, dC.download(), Y0, dY.download())
    # an infinite element in the vector that idle lanes load counts once, and only where it is named
    B[0, -1] = np.inf
    A[3, -1] = np.inf
    A[A == 0], A[:, -1] = 1, np.abs(A[:, -1])
    ii2, jj2 = np.append(ii, 5).astype(np.uint32), np.append(jj, 0).astype(np.uint32)
    o = np.argsort(ii2, kind="stable")
    ii2, jj2 = ii2[o], jj2[o]
    v2 = np.ones(ii2.size, dtype)
    C = gpu_sddmm(ctx, m, n, ii2, jj2, v2, A, B)
    hit = (jj2 == 0) | (ii2 == 3)
    assert np.all(np.isinf(C[hit])) and np.all(np.isfinite(C[~hit]))
    Y = gpu_spmm(ctx, m, n, ii2, jj2, v2, B, Y0)
    want = np.zeros(Y.shape, bool)
    want[5, -1] = True
    assert np.array_equal(np.isposinf(Y), want) and np.all(np.isfinite(Y[~want]))
