"""Names of the HIP kernels that a call launches, from a graph capture.

The call is captured on the current stream's side and never replayed; the
kernel nodes' host functions give the (mangled) names, template arguments
included, so a test can say which variant of a kernel a dispatch rule chose.
"""
import ctypes

import torch


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class _KernelNodeParams(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("blockDim", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("gridDim", _Dim3),
                ("kernelParams", ctypes.c_void_p), ("sharedMemBytes", ctypes.c_uint32)]


def _hip():
    """The HIP runtime this process runs on."""
    with open("/proc/self/maps") as f:
        paths = {line.split()[-1] for line in f if "libamdhip64.so" in line}
    assert len(paths) == 1, f"HIP runtimes loaded: {sorted(paths)}"
    lib = ctypes.CDLL(paths.pop())
    vp = ctypes.c_void_p
    lib.hipGraphGetNodes.argtypes = [vp, vp, ctypes.POINTER(ctypes.c_size_t)]
    lib.hipGraphNodeGetType.argtypes = [vp, ctypes.POINTER(ctypes.c_int)]
    lib.hipGraphKernelNodeGetParams.argtypes = [vp, ctypes.POINTER(_KernelNodeParams)]
    lib.hipKernelNameRefByPtr.argtypes = [vp, vp]
    lib.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    return lib


def launched_kernels(call):
    """call() is run once under stream capture; returns its kernels' names."""
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        call()
    hip, raw = _hip(), ctypes.c_void_p(graph.raw_cuda_graph())
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ctypes.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    names = []
    for node in nodes:
        kind = ctypes.c_int(-1)
        assert hip.hipGraphNodeGetType(node, ctypes.byref(kind)) == 0
        if kind.value != 0:  # hipGraphNodeTypeKernel
            continue
        p = _KernelNodeParams()
        assert hip.hipGraphKernelNodeGetParams(node, ctypes.byref(p)) == 0
        name = hip.hipKernelNameRefByPtr(p.func, None)
        assert name, "a captured kernel has no name"
        names.append(name.decode())
    assert names, "no kernel was captured"
    return names
