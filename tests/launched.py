"""The kernels that a call launches, read from a capture of it: nothing runs.  For the choices between forms of a kernel that give
the same bits, or go by one name, and so show in time only."""
import ctypes

import torch


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class _KernelNodeParams(ctypes.Structure):   # hipKernelNodeParams
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", _Dim3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint32)]


def _hip():
    """The HIP runtime of this process."""
    with open("/proc/self/maps") as f:
        paths = {line.split()[-1] for line in f if "libamdhip64" in line}
    assert len(paths) == 1, paths
    return ctypes.CDLL(paths.pop())


def launched(call):
    """(threads per workgroup, bytes of dynamic LDS) of every kernel that call(stream) launches on the stream, in order."""
    return [(p.block.x, p.shared) for p in _nodes(call)]


def kernels(call):
    """What tells the kernels of call(stream) apart, in order."""
    return [p.func for p in _nodes(call)]


def _nodes(call):
    hip = _hip()

    def ok(code):
        assert code == 0, "HIP error %d" % code

    stream, graph = torch.cuda.Stream(), ctypes.c_void_p()
    torch.cuda.synchronize()
    ok(hip.hipStreamBeginCapture(ctypes.c_void_p(stream.cuda_stream), 2))   # hipStreamCaptureModeRelaxed: outputs may be allocated
    try:
        call(stream)
    finally:
        ok(hip.hipStreamEndCapture(ctypes.c_void_p(stream.cuda_stream), ctypes.byref(graph)))
    found = []
    try:
        count = ctypes.c_size_t()
        ok(hip.hipGraphGetNodes(graph, None, ctypes.byref(count)))
        nodes = (ctypes.c_void_p * count.value)()
        ok(hip.hipGraphGetNodes(graph, nodes, ctypes.byref(count)))
        for node in nodes:
            kind = ctypes.c_int()
            ok(hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)))
            assert kind.value == 0   # hipGraphNodeTypeKernel
            p = _KernelNodeParams()
            ok(hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)))
            found.append(p)
    finally:
        ok(hip.hipGraphDestroy(graph))
    return found
