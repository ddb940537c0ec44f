"""Inner product and maximum norm at the edges of their shares: one page, a page more or less than a
workgroup's four, remainders of the four groups in flight, and arrays that start off a 16-byte boundary.

Integer values of up to 2^11: products below 2^24 and their sums below 2^53 are exact, so any order of
summation gives the integer sum itself."""
import ctypes as C

import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import HIP_D2H, HIP_H2D, hip_runtime

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("pages", [1, 3, 4, 5, 1003, 4095, 4097, 16400])
@pytest.mark.parametrize("shift", [(0, 0), (1, 0), (2, 3)])
def test_noalloc_exact_on_integers(pages, shift):
    from hierarchicaldd_amd import hdd
    n = pages * 256
    print(f"[pages {pages}] shift {shift}", flush=True)
    rng = np.random.default_rng(pages)
    v = [rng.integers(-2048, 2049, n).astype(np.float32) for _ in range(2)]
    H, ptr = hip_runtime(), [C.c_void_p() for _ in range(3)]
    out = np.zeros(1)
    try:
        for p, size in zip(ptr, (4 * n + 16, 4 * n + 16, 8)):
            assert H.hipMalloc(C.byref(p), size) == 0
        at = [C.c_void_p(p.value + 4 * k) for p, k in zip(ptr, shift)]
        for p, h in zip(at, v):
            assert H.hipMemcpy(p, h.ctypes.data_as(C.c_void_p), 4 * n, HIP_H2D) == 0
        assert hdd.lib().hdd_inner_product_noalloc(at[0], at[1], pages, ptr[2], None) == 0
        assert H.hipStreamSynchronize(None) == 0
        assert H.hipMemcpy(out.ctypes.data_as(C.c_void_p), ptr[2], 8, HIP_D2H) == 0
    finally:
        for p in ptr:
            H.hipFree(p)
    assert out[0] == float(np.dot(v[0].astype(np.int64), v[1].astype(np.int64)))


def test_context_products_and_norm_of_uneven_problems():
    from hierarchicaldd_amd import hdd
    g = hdd.DDBatch([domain.sphere_case(n, 16, 3) for n in (16, 48, 32)])
    try:
        ends = np.cumsum([g.problem_pages(p) for p in range(3)])
        rng = np.random.default_rng(5)
        a, b = (rng.integers(-2048, 2049, (g.n_pages, 256)).astype(np.float32) for _ in range(2))
        g.set(hdd.CH_Z, a)
        g.set(hdd.CH_R, b)
        dot, norm = (C.c_double * 3)(), (C.c_float * 3)()
        assert hdd.lib().hdd_inner_product(g.h, hdd.CH_Z, hdd.CH_R, dot) == 0
        assert hdd.lib().hdd_convergence_norm(g.h, hdd.CH_Z, norm) == 0
        for p, (first, last) in enumerate(zip(np.r_[0, ends[:-1]], ends)):
            assert dot[p] == float(np.vdot(a[first:last].astype(np.int64), b[first:last].astype(np.int64)))
            assert norm[p] == float(np.abs(a[first:last]).max())
    finally:
        g.close()
