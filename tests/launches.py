"""The kernel launches that a call makes, by capturing it: which path a dispatch rule took."""
import ctypes

import torch


class Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]


class KernelNodeParams(ctypes.Structure):
    _fields_ = [("block", Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", Dim3),
                ("params", ctypes.c_void_p), ("shared", ctypes.c_uint)]


def launches(sdamd, call):
    """[((grid x, y, z), block size), ...] of call(stream), in order.  The call runs once first, so that workspaces
    are there."""
    hip = sdamd.lib()  # its symbols include those of the HIP runtime it is linked to
    stream = torch.cuda.Stream()
    s, graph, n = ctypes.c_void_p(stream.cuda_stream), ctypes.c_void_p(), ctypes.c_size_t()
    call(stream.cuda_stream)
    torch.cuda.synchronize()
    assert hip.hipStreamBeginCapture(s, 2) == 0
    try:
        call(stream.cuda_stream)
    finally:
        assert hip.hipStreamEndCapture(s, ctypes.byref(graph)) == 0
    assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
    out = []
    for node in nodes:
        kind, p = ctypes.c_int(), KernelNodeParams()
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        assert kind.value == 0, f"node of type {kind.value}"  # kernels only
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        out.append(((p.grid.x, p.grid.y, p.grid.z), p.block.x))
    assert hip.hipGraphDestroy(graph) == 0
    return out
