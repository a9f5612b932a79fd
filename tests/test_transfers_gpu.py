"""Copies between host memory and a panel, at the sizes where their route changes: the pinned
buffer of an upload, the pieces and buffers of a download, memory that is pinned already."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
MIB = 1 << 20


def host_bytes(n, pinned):
    if not pinned:
        return np.empty(n, dtype=np.uint8), lambda: None
    hip = ctypes.CDLL("libamdhip64.so.7")  # the one the library is linked to
    p = ctypes.c_void_p()
    assert hip.hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(n), 0) == 0
    return (np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_uint8)), (n,)),
            lambda: hip.hipHostFree(p))


@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("nbytes", [4, 4096, MIB // 2 - 4, MIB // 2, MIB // 2 + 4, 2 * MIB + 1020,
                                    4 * MIB, 4 * MIB + 4, 33 * MIB - 4, 41 * MIB + 2044])
@pytest.mark.parametrize("threads", [1, 3])
def test_panel_comes_back_as_it_went(nbytes, pinned, threads):
    from spcomm3d_amd import device
    host, free_host = host_bytes(nbytes, pinned)
    out, free_out = host_bytes(nbytes, pinned)
    host[:] = np.random.default_rng(nbytes).integers(0, 256, nbytes, dtype=np.uint8)
    rows = nbytes // 4
    with device.Context(0, host_threads=threads) as ctx:
        p = ctx.panel(rows, 1, np.float32)
        p.upload(host.view(np.float32))
        device.check(ctx._lib.spc3d_panel_download(p._h, device._vp(out)), "spc3d_panel_download")
        assert np.array_equal(out, host)
        assert np.array_equal(p.download().reshape(-1).view(np.uint8), host)
        p.close()
    free_host()
    free_out()
