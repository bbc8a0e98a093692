"""The kernels a call launches, in launch order, by capturing it into a HIP
graph (which is not run): names as the compiler mangled them."""
import ctypes as C

import torch


class _Dim3(C.Structure):
    _fields_ = [("x", C.c_uint32), ("y", C.c_uint32), ("z", C.c_uint32)]


class _KernelParams(C.Structure):   # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", _Dim3),
                ("params", C.c_void_p), ("shared", C.c_uint)]


_KERNEL_NODE = 0     # hipGraphNodeTypeKernel
_THREAD_LOCAL = 1    # hipStreamCaptureModeThreadLocal


def _hip():
    h = C.CDLL(None)   # torch has loaded the HIP runtime
    try:
        h.hipGraphGetNodes
    except AttributeError:
        h = C.CDLL("libamdhip64.so")
    h.hipKernelNameRefByPtr.restype = C.c_char_p
    h.hipKernelNameRefByPtr.argtypes = [C.c_void_p, C.c_void_p]
    return h


def captured_kernels(call):
    """Names; call(stream): launches on the stream it is given, allocating nothing."""
    return [name for name, _ in captured_launches(call)]


def captured_launches(call):
    """As captured_kernels, with each launch's workgroups (x, y, z)."""
    hip = _hip()

    def ok(rc):
        assert rc == 0, f"HIP error {rc}"
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    st, graph = C.c_void_p(stream.cuda_stream), C.c_void_p()
    ok(hip.hipStreamBeginCapture(st, C.c_int(_THREAD_LOCAL)))
    try:
        with torch.cuda.stream(stream):
            call(st)
    finally:
        ok(hip.hipStreamEndCapture(st, C.byref(graph)))
    try:
        n = C.c_size_t()
        ok(hip.hipGraphGetNodes(graph, None, C.byref(n)))
        nodes = (C.c_void_p * n.value)()
        ok(hip.hipGraphGetNodes(graph, nodes, C.byref(n)))
        launches = []
        for node in nodes:
            kind, p = C.c_int(), _KernelParams()
            ok(hip.hipGraphNodeGetType(C.c_void_p(node), C.byref(kind)))
            if kind.value != _KERNEL_NODE:
                continue
            ok(hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(p)))
            launches.append((hip.hipKernelNameRefByPtr(p.func, None).decode(), (p.grid.x, p.grid.y, p.grid.z)))
        return launches
    finally:
        ok(hip.hipGraphDestroy(graph))
