"""Sweeps of whole clusters in one launch (every V-cycle level whose clusters of coupled cells fit a
workgroup) against one launch per sweep (HDD_BOTTOM_LOCAL=0): the same operations in the same order,
so the bar is equal bits (which also holds the single sweeps that skip what the sweep before left in place
against sweeps that write every cell). The cases have clusters from a few cells (one wavefront, neighbours in
registers) to several per thread, one cluster per workgroup and packed ones, a level 0 whose cluster
edges read interface cells, a single-level V-cycle (200 sweeps of level 0 around nonzero interface
values), and levels on both sides of the size limit."""
import os

import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import random_rhs, same_bits

pytestmark = pytest.mark.gpu


def _blocked(n, sub, vlevels, seed, nV=1):
    rng = np.random.default_rng(seed)
    flags = domain.box_flags(n, domain.random_spheres(rng, n, int(rng.integers(1, 5)), 0.1, 0.3), drop_enclosed=True)
    rhs = rng.standard_normal((n, n, n)).astype(np.float32)
    return domain.domain_from_flags(n, flags, rhs=rhs), domain.DDConfig(sub_size=sub, vlevels=vlevels, nVcycles=nV)


CASES = {
    "box45_sub16": lambda: domain.small_box(45, 16, 3, seed=4),        # level 0 in clusters, odd edge
    "blocked100_sub16": lambda: _blocked(100, 16, 3, 7),               # clusters that lie in up to 13 pages at level 1
    "blocked100_sub32": lambda: _blocked(100, 32, 4, 0),               # level 0 too large, level 1 across page boundaries
    "box136_sub16": lambda: domain.small_box(136, 16, 3, seed=9),      # more clusters than run side by side: packed
    "box33_one_level": lambda: domain.small_box(33, 16, 1, seed=6),    # the bottom is level 0
    "box40_two_cycles": lambda: _blocked(40, 16, 2, 11, nV=2),         # V-cycles that start from a nonzero iterate
}


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("name", list(CASES))
def test_cluster_sweeps_bitwise(name, fp16):
    from hierarchicaldd_amd import hdd
    dom, cfg = CASES[name]()
    print(f"[{name} fp16={fp16}] pages {dom.n_pages}", flush=True)
    tol = 1e-6 * float(np.abs(dom.b).max())
    out = {}
    for mode in ("0", ""):
        os.environ["HDD_BOTTOM_LOCAL"] = mode
        try:
            g = hdd.DDSolver(dom, cfg)
        finally:
            os.environ.pop("HDD_BOTTOM_LOCAL", None)
        try:
            g.set_fp16(fp16)
            b = random_rhs(g.level(0)[1], 31)
            z = g.apply_preconditioner(b)
            z2 = g.apply_preconditioner(b[:, ::-1].copy())
            it, hist, _ = g.solve(tol, 60)
            out[mode] = (g.stats()["bottom_page_local"], z, z2, it, hist, g.get(hdd.CH_X))
        finally:
            g.close()
    a, c = out["0"], out[""]
    assert a[0] == 0 and c[0] == 1
    assert np.isfinite(c[1]).all()
    assert same_bits(a[1], c[1]) and same_bits(a[2], c[2])
    assert a[3] == c[3] and np.array_equal(a[4], c[4]) and same_bits(a[5], c[5])
