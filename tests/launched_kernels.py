"""Names of the kernels that a call launches: the call is recorded into a HIP
graph (which launches nothing) and the graph's kernel nodes are read back."""
import ctypes

import torch


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]


class _KernelNodeParams(ctypes.Structure):
    _fields_ = [("block", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", _Dim3), ("params", ctypes.c_void_p), ("lds", ctypes.c_uint)]


def _runtime():
    """The HIP runtime this process already runs on."""
    with open("/proc/self/maps") as f:
        return ctypes.CDLL(next(ln.split()[-1] for ln in f if "libamdhip64" in ln))


def launched_kernels(call):
    """The (mangled) names of the kernels that call() launches on the current
    stream, in order."""
    call()  # first use: one-time set-up of the kernels, outside the capture
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    hip, raw = _runtime(), ctypes.c_void_p(graph.raw_cuda_graph())
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    names = []
    for node in nodes:
        p = _KernelNodeParams()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        names.append(hip.hipKernelNameRefByPtr(ctypes.c_void_p(p.func), None).decode())
    return names
