"""Which kernels a call launches: the call is captured into a graph, which runs nothing, and the graph's kernel nodes are listed."""
import ctypes

import torch


class _Params(ctypes.Structure):                     # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint * 3), ("args", ctypes.c_void_p),
                ("shared", ctypes.c_uint)]


def _hip():
    """The runtime torch has loaded, which the library's kernels are registered with."""
    with open("/proc/self/maps") as f:
        L = ctypes.CDLL(next(line.split()[-1] for line in f if "libamdhip64" in line))
    L.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    L.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    return L


def kernels(call):
    """Mangled names of the kernels that `call` launches on the current stream, one to a launch."""
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    L, handle, n = _hip(), ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t()
    assert L.hipGraphGetNodes(handle, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert L.hipGraphGetNodes(handle, nodes, ctypes.byref(n)) == 0
    names = []
    for node in nodes:
        kind, p = ctypes.c_int(-1), _Params()
        assert L.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value:                               # a copy
            continue
        assert L.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        names.append(L.hipKernelNameRefByPtr(p.func, None).decode())
    return names
