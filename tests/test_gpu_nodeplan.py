"""The dense-node form of the interface solver's exact solves on the GPU: against the double factors
and against the per-height form (HDD_DENSE_TOP=0), at odd edges, both subdomain sizes, a single
subdomain, a sparse domain and in a batch.

Bars: a solve runs at most 7 levels, two passes each, and a pass rounds its float sums a few times to
2^-24 of their largest term; the operators are diagonally dominant, so the passes do not amplify:
14 * 6e-8 = 8.4e-7, bar 1e-6 of the largest value against the double factor, and twice that between
the two float forms (a smooth is two solves: 4e-6)."""
import os

import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import rel_err, same_bits

pytestmark = pytest.mark.gpu


def _box(n, sub, vlevels):
    return domain.small_box(n, sub, vlevels, seed=n)


CASES = {
    "box33_sub16": lambda: _box(33, 16, 3),
    "box45_sub16": lambda: _box(45, 16, 3),
    "box67_sub32": lambda: _box(67, 32, 4),
    "one_subdomain_sub32": lambda: _box(32, 32, 4),
    "sphere96_sub16": lambda: domain.sphere_case(96, 16, 3),
    "sparse96_sub16": lambda: domain.sparse_spheres(96, rmin=6, rmax=18, sub=16, vlevels=3),
}


def _smooths(g, seed=3):
    rng = np.random.default_rng(seed)
    out = []
    for l in range(g.sigma_info()[0]):
        n = g.interface_dofs(l)
        if n == 0:
            continue
        b = rng.standard_normal(n).astype(np.float32)
        u = (0.1 * rng.standard_normal(n)).astype(np.float32)
        out.append((l, b, u, g.sigma_smooth(l, b, np.zeros_like(u)), g.sigma_smooth(l, b, u)))
    return out


@pytest.mark.parametrize("name", list(CASES))
def test_solves_against_factors_and_heights(name):
    from hierarchicaldd_amd import hdd
    dom, cfg = CASES[name]()
    print(f"[{name}] pages {dom.n_pages}", flush=True)
    g = hdd.DDSolver(dom, cfg)
    os.environ["HDD_DENSE_TOP"] = "0"
    try:
        heights = hdd.DDSolver(dom, cfg)
    finally:
        os.environ.pop("HDD_DENSE_TOP", None)
    try:
        assert g.stats()["fused_heights"] > 0  # levels of the dense-node plans
        for l, b, u, x, s in _smooths(g):
            ref = g.sigma_factor_solve(l, "Arr", 0, b.astype(np.float64))
            assert rel_err(x, ref) < 1e-6, f"level {l}: {rel_err(x, ref)}"
            assert rel_err(s, heights.sigma_smooth(l, b, u)) < 4e-6, f"level {l}"
    finally:
        g.close()
        heights.close()


def test_batch_shares_blocks_and_keeps_problems_apart():
    """Three problems, two of them equal: each smooth within the bar of its smooth alone, the equal
    ones bit-identical, a second build bit-identical."""
    from hierarchicaldd_amd import hdd
    probs = [_box(45, 16, 3), _box(33, 16, 3), _box(45, 16, 3)]
    alone = [hdd.DDSolver(*p) for p in probs]
    runs = []
    for _ in range(2):
        bt = hdd.DDBatch(probs)
        try:
            res = []
            for l in range(bt.sigma_info()[0]):
                parts = [g.interface_dofs(l) for g in alone]
                rng = np.random.default_rng(l)
                b = [rng.standard_normal(parts[0]).astype(np.float32), rng.standard_normal(parts[1]).astype(np.float32)]
                u = [0.1 * v[::-1].copy() for v in b]
                b, u = b + [b[0]], u + [u[0]]
                s = bt.sigma_smooth(l, np.concatenate(b), np.concatenate(u))
                res.append((np.split(s, np.cumsum(parts)[:-1]), b, u))
        finally:
            bt.close()
        runs.append(res)
    for (s0, b, u), (s1, _, _) in zip(*runs):
        assert all(same_bits(p, q) for p, q in zip(s0, s1))
        assert same_bits(s0[0], s0[2])
    for l, (s, b, u) in enumerate(runs[0]):
        for p, g in enumerate(alone):
            assert rel_err(s[p], g.sigma_smooth(l, b[p], u[p])) < 4e-6, (l, p)
    for g in alone:
        g.close()
