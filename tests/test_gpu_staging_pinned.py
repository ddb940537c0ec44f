"""Whole channels from and to memory that the caller has pinned: the bytes that come back are the bytes
that went in, also mixed with pageable memory."""
import ctypes as C

import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import hip_runtime, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sub,vlevels", [(48, 16, 3), (104, 32, 4)])  # below and above the ring's size
def test_pinned_channels_round_trip(n, sub, vlevels):
    from hierarchicaldd_amd import hdd
    g = hdd.DDSolver(*domain.sphere_case(n, sub, vlevels))
    L, H = hdd.lib(), hip_runtime()
    H.hipHostMalloc.argtypes = [C.POINTER(C.c_void_p), C.c_size_t, C.c_uint]
    H.hipHostFree.argtypes = [C.c_void_p]
    cells = g.n_pages * 256
    print(f"[n {n}] {cells * 4e-6:.1f} MB", flush=True)
    mem = [C.c_void_p(), C.c_void_p()]
    try:
        for p in mem:
            assert H.hipHostMalloc(C.byref(p), 4 * cells, 0) == 0
        pinned_in, pinned_out = (np.ctypeslib.as_array(C.cast(p, C.POINTER(C.c_float)), (cells,)) for p in mem)
        v = np.random.default_rng(n).standard_normal(cells).astype(np.float32)
        out = np.zeros_like(v)
        pinned_in[:] = v
        pinned_out[:] = 0
        ptr = lambda a: a.ctypes.data_as(C.c_void_p)  # noqa: E731
        assert L.hdd_set_channel(g.h, hdd.CH_X, ptr(pinned_in)) == 0
        assert L.hdd_get_channel(g.h, hdd.CH_X, ptr(out)) == 0
        assert same_bits(out, v)
        assert L.hdd_set_channel(g.h, hdd.CH_S, ptr(v)) == 0
        assert L.hdd_get_channel(g.h, hdd.CH_S, ptr(pinned_out)) == 0
        assert same_bits(pinned_out, v)
    finally:
        g.close()
        for p in mem:
            if p:
                H.hipHostFree(p)
