import os
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)


def pytest_configure(config):
    config.addinivalue_line("markers", "gpu: needs a real MI355X (run with -m gpu)")


@pytest.fixture(scope="session")
def oracle():
    from oracle import pyoracle

    pyoracle.lib()
    pyoracle.set_round_mode(pyoracle.ROUND_HALF_AWAY)
    return pyoracle


@pytest.fixture(scope="session")
def golden():
    import json

    with open(os.path.join(ROOT, "tests", "golden", "reference_vectors.json")) as f:
        return json.load(f)


@pytest.fixture(scope="session")
def hipq():
    from torsh_amd import hipq as mod

    mod.load()
    return mod


@pytest.fixture(scope="session")
def ctx(hipq):
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = hipq.Context(0)
    yield c
    torch.cuda.synchronize()
    c.close()


@pytest.fixture(scope="session")
def launched_kernels(hipq):
    """launched_kernels(context with a stream of its own, call) -> names of the kernels that the call launches, in order.  The call
    is captured into a graph that is never launched, so nothing runs on the device."""
    import ctypes as C

    class Dim3(C.Structure):
        _fields_ = [("x", C.c_uint32), ("y", C.c_uint32), ("z", C.c_uint32)]

    class KernelNodeParams(C.Structure):
        _fields_ = [("block", Dim3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", Dim3), ("args", C.c_void_p),
                    ("shared_bytes", C.c_uint)]

    with open("/proc/self/maps") as f:
        hip = C.CDLL(next(line.split()[-1] for line in f if "libamdhip64.so" in line))
    hip.hipKernelNameRefByPtr.restype = C.c_char_p

    def names(ctx, call):
        stream, graph, n = C.c_void_p(ctx.stream_handle), C.c_void_p(), C.c_size_t()
        assert hip.hipStreamBeginCapture(stream, 2) == 0  # relaxed: the call may allocate its outputs
        try:
            call()
        finally:
            assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
        assert hip.hipGraphGetNodes(graph, None, C.byref(n)) == 0
        nodes = (C.c_void_p * n.value)()
        assert hip.hipGraphGetNodes(graph, nodes, C.byref(n)) == 0
        found = []
        for node in nodes:
            params = KernelNodeParams()
            assert hip.hipGraphKernelNodeGetParams(C.c_void_p(node), C.byref(params)) == 0
            found.append(hip.hipKernelNameRefByPtr(C.c_void_p(params.func), stream).decode())
        assert hip.hipGraphDestroy(graph) == 0
        return found

    return names


@pytest.fixture(scope="session")
def stream_ctx(hipq):
    """A context with a stream of its own."""
    import torch

    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    c = hipq.Context(0, own_stream=True)
    yield c
    torch.cuda.synchronize()
    c.close()
