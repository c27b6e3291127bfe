"""The kernels that one call enqueues, read from a captured HIP graph, so that
tests and the benchmark can say which kernel and tile a case ran."""
import ctypes
import re
from collections import namedtuple

Launch = namedtuple("Launch", "name template grid")   # template: the integers and booleans, in order
GEMM_KIND = {0: "int8", 1: "int4_k", 2: "int4_n"}
Gemm = namedtuple("Gemm", "kind pieces zp tm tn")


class _Dim3(ctypes.Structure):
    _fields_ = [("x", ctypes.c_uint), ("y", ctypes.c_uint), ("z", ctypes.c_uint)]


class _KernelNodeParams(ctypes.Structure):
    _fields_ = [("blockDim", _Dim3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("gridDim", _Dim3),
                ("kernelParams", ctypes.c_void_p), ("sharedMemBytes", ctypes.c_uint)]


def _hip():
    with open("/proc/self/maps") as f:
        path = next(line.split()[-1] for line in f if "libamdhip64" in line)
    hip = ctypes.CDLL(path)
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    hip.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    return hip


def _parse(mangled, grid):
    # _ZN <len><part> ... [I <template arguments> E] ...
    rest, parts = mangled[len("_ZN"):], []
    while rest and rest[0].isdigit():
        n = re.match(r"\d+", rest).group()
        parts.append(rest[len(n):len(n) + int(n)])
        rest = rest[len(n) + int(n):]
    args = [int(v) for v in re.findall(r"L[ib](\d+)E", rest.split("EEv")[0] + "E")]   # before the result type
    return Launch(parts[-1], tuple(args), grid)


def launches(call, stream):
    """call() enqueues work on `stream` (a torch.cuda.Stream) and allocates
    nothing; returns its kernel launches in order.  Nothing runs."""
    hip, s = _hip(), ctypes.c_void_p(stream.cuda_stream)
    graph = ctypes.c_void_p()
    assert hip.hipStreamBeginCapture(s, 1) == 0
    try:
        call()
    finally:
        rc = hip.hipStreamEndCapture(s, ctypes.byref(graph))
    assert rc == 0
    try:
        n = ctypes.c_size_t()
        assert hip.hipGraphGetNodes(graph, None, ctypes.byref(n)) == 0
        nodes = (ctypes.c_void_p * n.value)()
        assert hip.hipGraphGetNodes(graph, nodes, ctypes.byref(n)) == 0
        out = []
        for node in nodes:
            p = _KernelNodeParams()
            assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(p)) == 0
            name = hip.hipKernelNameRefByPtr(p.func, s).decode()
            out.append(_parse(name, (p.gridDim.x, p.gridDim.y, p.gridDim.z)))
        return out
    finally:
        hip.hipGraphDestroy(graph)


def gemms(ls):
    """The prefill GEMM launches among ls as (kind, pieces per x row, zero points,
    16-row tiles, 128-column tiles)."""
    return [Gemm(GEMM_KIND[t[0]], t[1], bool(t[2]), t[3], t[4]) for n, t, _ in ls if n == "gemm"]
