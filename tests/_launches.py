"""The kernels that a call launches, read off a recording of it (a HIP graph)."""
import ctypes

from spcomm3d_amd import _capi as capi


class _Dim3(ctypes.Structure):
    _fields_ = [(n, ctypes.c_uint32) for n in "xyz"]


class _KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", _Dim3), ("args", ctypes.c_void_p), ("lds", ctypes.c_uint32)]


def launches(ctx, call):
    """[(workgroups, bytes of dynamic LDS)] of every kernel that `call` queues on the context.  The
    call has run once before: what it allocates is there."""
    lib = ctx._lib
    stream, graph = ctypes.c_void_p(), ctypes.c_void_p()
    capi.check(lib.spc3d_ctx_stream(ctx._h, ctypes.byref(stream)), "spc3d_ctx_stream")
    assert lib.hipStreamBeginCapture(stream, 1) == 0  # thread-local, as the library records
    try:
        call()
    finally:
        assert lib.hipStreamEndCapture(stream, ctypes.byref(graph)) == 0
    n = ctypes.c_size_t()
    assert lib.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert lib.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        kind, p = ctypes.c_int(-1), _KernelNode()
        assert lib.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value == 0:
            assert lib.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
            out.append((p.grid.x, p.lds))
    assert lib.hipGraphDestroy(graph) == 0
    return out
