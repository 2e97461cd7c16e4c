"""The kernel launches of a call: it is recorded into a HIP graph (nothing runs)
and the graph's kernel nodes are read back.  The library's kernels differ by
their workgroups: (64, 4, 1) for one thread per point, one dimension for the
tiled ones."""
import ctypes


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class _KernelNodeParams(ctypes.Structure):      # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("params", ctypes.c_void_p), ("lds", ctypes.c_uint32)]


def launches(capi, call, func=False):
    """call(stream) -> [(workgroups, threads, LDS bytes)] of its kernels (func: and
    their handles); it is run once before, for what a first call sets up"""
    hip = capi.lib()                            # the library's own HIP runtime
    stream, graph, n = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t(0)

    def ok(rc):
        assert rc == 0, f"HIP error {rc}"

    capi.check(hip.hsx_stream_create(ctypes.byref(stream)))
    try:
        call(stream)
        capi.sync(stream)
        ok(hip.hipStreamBeginCapture(stream, 1))            # thread-local
        call(stream)
        ok(hip.hipStreamEndCapture(stream, ctypes.byref(graph)))
        ok(hip.hipGraphGetNodes(graph, None, ctypes.byref(n)))
        nodes = (ctypes.c_void_p * n.value)()
        ok(hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)))
        out = []
        for node in nodes:
            k = _KernelNodeParams()
            ok(hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(k)))
            out.append(((k.grid.x, k.grid.y, k.grid.z), (k.block.x, k.block.y, k.block.z), k.lds)
                       + ((k.func,) if func else ()))
        ok(hip.hipGraphDestroy(graph))
        return out
    finally:
        capi.check(hip.hsx_stream_destroy(stream))
