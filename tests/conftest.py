import ctypes
import os
import re
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu on the GPU box)")


@pytest.fixture(scope="session")
def oracle():
    from oracle.oracle import Oracle
    return Oracle()


@pytest.fixture(scope="session")
def reference():
    """The real vecops CPU matmul, where oracle/_ref was built and the host has AMX."""
    from oracle.oracle import Reference
    ref = Reference.load()
    if ref is None:
        pytest.skip("oracle/_ref/libvecops_ref.so not built or host lacks AMX")
    return ref


@pytest.fixture(scope="session")
def device():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch.device("cuda:0")


def rel_err(got: np.ndarray, want: np.ndarray) -> float:
    """max |got - want| / max(1, |want|, |got|): the scaling of the reference's own
    conversion checks (tests/ops/MatmulConversionTestCommon.h:72-85)."""
    got = np.asarray(got, dtype=np.float64)
    want = np.asarray(want, dtype=np.float64)
    if got.size == 0:
        return 0.0
    scale = np.maximum(1.0, np.maximum(np.abs(got), np.abs(want)))
    return float((np.abs(got - want) / scale).max())


class _KernelNode(ctypes.Structure):  # hipKernelNodeParams
    _fields_ = [("block", ctypes.c_uint32 * 3), ("extra", ctypes.c_void_p), ("func", ctypes.c_void_p), ("grid", ctypes.c_uint32 * 3),
                ("args", ctypes.c_void_p), ("lds", ctypes.c_uint32)]


def launched_kernels(call) -> list[str]:
    """The kernels that ``call`` launches, in order, as "name<template arguments>": read from the nodes of a graph that the call
    is captured into (it is run once before)."""
    import torch
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph(keep_graph=True)
    with torch.cuda.graph(graph):
        call()
    with open("/proc/self/maps") as maps:
        hip = ctypes.CDLL(next(line.split()[-1] for line in maps if "libamdhip64" in line))
    hip.hipKernelNameRefByPtr.restype = ctypes.c_char_p
    hip.hipKernelNameRefByPtr.argtypes = [ctypes.c_void_p, ctypes.c_void_p]
    raw, count = ctypes.c_void_p(graph.raw_cuda_graph()), ctypes.c_size_t(0)
    assert hip.hipGraphGetNodes(raw, None, ctypes.byref(count)) == 0
    nodes = (ctypes.c_void_p * count.value)()
    assert hip.hipGraphGetNodes(raw, nodes, ctypes.byref(count)) == 0
    names = []
    for node in nodes:
        params = _KernelNode()
        assert hip.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), ctypes.byref(params)) == 0, "a node that is no kernel"
        mangled = hip.hipKernelNameRefByPtr(params.func, None).decode().replace("_ZN10vecops_hip", "").replace("12_GLOBAL__N_1", "")
        name, arguments = re.match(r"\d+([a-z]\w*?_kernel)(?:I((?:L[ib]\d+E)+))?", mangled).groups()
        names.append(name + (f"<{','.join(re.findall('[ib]([0-9]+)E', arguments))}>" if arguments else ""))
    return names
