"""Which kernels of the library a call launches: the call is captured into a HIP
graph and the graph's kernel nodes are matched with the kernel handles that the
library exports."""

import ctypes
import functools
import re
import subprocess

import torch

from sglang_mlx_amd import _lib


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint32), ("y", ctypes.c_uint32), ("z", ctypes.c_uint32)]


class _KernelNodeParams(ctypes.Structure):
    """hipKernelNodeParams (hip/hip_runtime_api.h of ROCm 7.2)."""
    _fields_ = [("blockDim", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("gridDim", _Dim3),
                ("kernelParams", ctypes.c_void_p), ("sharedMemBytes", ctypes.c_uint)]


@functools.lru_cache(None)
def _handles():
    names = subprocess.run(["nm", "-D", "--defined-only", _lib.LIB_PATH], capture_output=True, text=True,
                           check=True).stdout
    lib = _lib.lib()
    return {ctypes.cast(getattr(lib, m.group(1)), ctypes.c_void_p).value: m.group(1)
            for m in re.finditer(r" V (_ZN3pkv\w*kernel\w*)", names)}


def kernels_of(call):
    """[(kernel symbol, workgroups)] of the library's kernels that call() launches on
    the current stream."""
    hip = ctypes.CDLL("libamdhip64.so.7")
    ptr = ctypes.c_void_p
    hip.hipGraphGetNodes.argtypes = [ptr, ctypes.POINTER(ptr), ctypes.POINTER(ctypes.c_size_t)]
    hip.hipGraphNodeGetType.argtypes = [ptr, ctypes.POINTER(ctypes.c_int)]
    hip.hipGraphKernelNodeGetParams.argtypes = [ptr, ctypes.POINTER(_KernelNodeParams)]
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    raw = graph.raw_cuda_graph()
    n = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(n)) == 0
    nodes = (ptr * n.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(n)) == 0
    found = []
    for node in nodes:
        kind = ctypes.c_int(-1)
        assert hip.hipGraphNodeGetType(node, ctypes.byref(kind)) == 0
        if kind.value != 0:  # hipGraphNodeTypeKernel
            continue
        params = _KernelNodeParams()
        assert hip.hipGraphKernelNodeGetParams(node, ctypes.byref(params)) == 0
        name = _handles().get(params.func)
        if name is not None:
            found.append((name, params.gridDim.x * params.gridDim.y * params.gridDim.z))
    assert found
    return found
