"""The kernel launches of a call, from a HIP graph it is captured into (and
which is not run): name, workgroups, threads per workgroup, LDS bytes."""
import ctypes
from typing import NamedTuple


class _Params(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p),
                ("grid", ctypes.c_uint32 * 3), ("args", ctypes.c_void_p), ("lds", ctypes.c_uint32)]


class _Attributes(ctypes.Structure):  # hipFuncAttributes
    _fields_ = [("binary_version", ctypes.c_int), ("cache_mode", ctypes.c_int), ("const_bytes", ctypes.c_size_t),
                ("local_bytes", ctypes.c_size_t), ("max_dynamic", ctypes.c_int), ("max_threads", ctypes.c_int),
                ("registers", ctypes.c_int), ("carveout", ctypes.c_int), ("ptx", ctypes.c_int),
                ("lds", ctypes.c_size_t)]


class Launch(NamedTuple):
    name: str
    groups: int
    threads: int
    lds: int  # static and dynamic


def launches(call):
    import torch

    from iclr_2027_jointoom_amd._abi import load_library

    hip = load_library()  # (its dependencies' symbols too)
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.graph(graph, stream=stream):
        call()
    torch.cuda.current_stream().wait_stream(stream)
    handle = ctypes.c_void_p(int(graph.raw_cuda_graph()))
    count = ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(handle, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * count.value)()
    assert hip.hipGraphGetNodes(handle, nodes, ctypes.byref(count)) == 0
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    out = []
    for node in nodes:
        kind = ctypes.c_int(-1)
        assert hip.hipGraphNodeGetType(ctypes.c_void_p(node), ctypes.byref(kind)) == 0
        if kind.value != 0:  # hipGraphNodeTypeKernel
            continue
        p, a = _Params(), _Attributes()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
        assert hip.hipFuncGetAttributes(ctypes.byref(a), ctypes.c_void_p(p.func)) == 0
        name = (hip.hipKernelNameRefByPtr(ctypes.c_void_p(p.func), None) or b"").decode()
        out.append(Launch(name, p.grid[0] * p.grid[1] * p.grid[2], p.block[0], p.lds + a.lds))
    return out
