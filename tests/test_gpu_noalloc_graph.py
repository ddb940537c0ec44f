"""hdd_inner_product_noalloc in a captured graph: every replay, with new values and eager calls between
them, gives the sum (integers, so exactly: tests/test_gpu_dot.py)."""
import ctypes as C

import numpy as np
import pytest

from tests.gpu_common import HIP_D2H, HIP_H2D, hip_runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pages", [1, 1003])
def test_replays(pages):
    from hierarchicaldd_amd import hdd
    L, H, P = hdd.lib(), hip_runtime(), C.c_void_p
    H.hipStreamBeginCapture.argtypes = [P, C.c_int]
    H.hipStreamEndCapture.argtypes = [P, C.POINTER(P)]
    H.hipGraphInstantiate.argtypes = [C.POINTER(P), P, P, P, C.c_size_t]
    H.hipGraphLaunch.argtypes = [P, P]
    H.hipGraphExecDestroy.argtypes = [P]
    H.hipGraphDestroy.argtypes = [P]
    n = pages * 256
    rng = np.random.default_rng(pages)
    print(f"[pages {pages}] capture", flush=True)
    ptr, s, graph, run = [P() for _ in range(4)], P(), P(), P()
    try:
        for p, size in zip(ptr, (4 * n, 4 * n, 8, 8)):
            assert H.hipMalloc(C.byref(p), size) == 0
        assert H.hipStreamCreate(C.byref(s)) == 0
        assert L.hdd_inner_product_noalloc(ptr[0], ptr[1], pages, ptr[3], s) == 0  # (finds its scratch array)
        assert H.hipStreamSynchronize(s) == 0
        assert H.hipStreamBeginCapture(s, 2) == 0  # relaxed
        assert L.hdd_inner_product_noalloc(ptr[0], ptr[1], pages, ptr[2], s) == 0
        assert H.hipStreamEndCapture(s, C.byref(graph)) == 0
        assert H.hipGraphInstantiate(C.byref(run), graph, None, None, 0) == 0
        for k in range(5):
            v = [rng.integers(-2048, 2049, n).astype(np.float32) for _ in range(2)]
            for p, h in zip(ptr, v):
                assert H.hipMemcpy(p, h.ctypes.data_as(P), 4 * n, HIP_H2D) == 0
            assert H.hipGraphLaunch(run, s) == 0
            for _ in range(k):
                assert L.hdd_inner_product_noalloc(ptr[0], ptr[1], pages, ptr[3], s) == 0
            assert H.hipGraphLaunch(run, s) == 0
            assert H.hipStreamSynchronize(s) == 0
            out = np.zeros(1)
            assert H.hipMemcpy(out.ctypes.data_as(P), ptr[2], 8, HIP_D2H) == 0
            assert out[0] == float(np.dot(v[0].astype(np.int64), v[1].astype(np.int64))), k
    finally:
        if run:
            H.hipGraphExecDestroy(run)
        if graph:
            H.hipGraphDestroy(graph)
        if s:
            H.hipStreamDestroy(s)
        for p in ptr:
            H.hipFree(p)
