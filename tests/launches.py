"""The kernels that a call launches, by name: for tests of the rules that choose between them."""
import ctypes

import torch


class _KernelNode(ctypes.Structure):
    """hipKernelNodeParams"""
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint32 * 3), ("params", ctypes.c_void_p), ("lds", ctypes.c_uint32)]


def _hip():
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    hip.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    return hip


def launched(call):
    """call() captured in a graph that is not run: the mangled names of its kernels, in order."""
    call()  # workspaces are allocated outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    hip, raw = _hip(), ctypes.c_void_p(graph.raw_cuda_graph())
    count = ctypes.c_size_t()
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * count.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(count)) == 0
    names = []
    for node in nodes:
        p = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        names.append(hip.hipKernelNameRefByPtr(p.func, None).decode())
    return names
