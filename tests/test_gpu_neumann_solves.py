"""The interface solver of a domain without Dirichlet cells on the GPU: its bottom system annihilates the
constant but for 1e-5, and the dense-node plan keeps the triangle of its root there
(tests/test_nodeplan_singular.py). One V-cycle on a right-hand side without a mean, dense nodes against
the per-height form (HDD_DENSE_TOP=0), less their means.

Bar: as between the two float forms of one smooth, two solves, in tests/test_gpu_nodeplan.py (4e-6): the
cycle ends with a smooth, and what came before it is contracted. (With the bottom's inverse rounded to
float the forms differ by 5e-6 at 32^3 and 1e-5 at 48^3.)"""
import os

import numpy as np
import pytest

from hierarchicaldd_amd import domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32, 48])
def test_vcycle_without_dirichlet_cells(n):
    from hierarchicaldd_amd import hdd
    dom, cfg = domain.neumann_box(n, 16, 3, seed=n)
    g = hdd.DDSolver(dom, cfg)
    os.environ["HDD_DENSE_TOP"] = "0"
    try:
        heights = hdd.DDSolver(dom, cfg)
    finally:
        os.environ.pop("HDD_DENSE_TOP", None)
    try:
        b = np.random.default_rng(n).standard_normal(g.interface_dofs(0)).astype(np.float32)
        b -= np.float32(b.mean(dtype=np.float64))
        u, v = (s.sigma_vcycle(b).astype(np.float64) for s in (g, heights))
    finally:
        g.close()
        heights.close()
    u -= u.mean()
    v -= v.mean()
    err = float(np.linalg.norm(u - v) / np.linalg.norm(v))
    print(f"[neumann{n}] dense nodes against the per-height form, less the constant: {err:.1e}")
    assert err < 4e-6
