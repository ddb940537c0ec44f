"""Sweeps of whole clusters against one launch per sweep (HDD_BOTTOM_LOCAL=0) where values overflow: the
same cells of z and of the level-0 residual are infinite, of the same sign, or not a number, and every
finite one has equal bits. Right-hand sides of +-3e38, at random and in a checkerboard (whose second
interior sweep overflows), and single infinite ones, beside an obstacle, whose cells lack face neighbours."""
import dataclasses
import os

import numpy as np
import pytest

from hierarchicaldd_amd import domain

pytestmark = pytest.mark.gpu


def _rhs(flags, kind):
    rng = np.random.default_rng(5)
    active = (flags & domain.ACTIVE) != 0
    b = np.zeros(flags.shape, dtype=np.float32)
    if kind == "checkerboard":  # pages start at multiples of 4, 8 and 8 cells
        c = np.arange(256)
        sign = np.where(((c >> 6) + (c >> 3) + c) & 1, np.float32(3e38), np.float32(-3e38))
        b = np.where(active, sign[None, :], np.float32(0)).astype(np.float32)
    elif kind == "huge":
        b[active] = rng.choice(np.array([-3e38, 3e38], dtype=np.float32), int(active.sum()))
    else:
        b[active] = rng.standard_normal(int(active.sum())).astype(np.float32)
        at = rng.choice(np.flatnonzero(active), 20, replace=False)
        b.flat[at] = rng.choice(np.array([np.inf, -np.inf], dtype=np.float32), 20)
    return b


@pytest.mark.parametrize("kind", ["huge", "checkerboard", "infinite"])
@pytest.mark.parametrize("name", ["box45_sub16", "box67_sub32"])
def test_overflow_as_by_single_sweeps(name, kind):
    from hierarchicaldd_amd import hdd
    dom, cfg = domain.small_box(45, 16, 3, seed=4) if name == "box45_sub16" else domain.small_box(67, 32, 4, seed=4)
    cfg = dataclasses.replace(cfg, interior_smoothing=2)
    out = {}
    for mode in ("0", ""):
        os.environ["HDD_BOTTOM_LOCAL"] = mode
        try:
            g = hdd.DDSolver(dom, cfg)
        finally:
            os.environ.pop("HDD_BOTTOM_LOCAL", None)
        try:
            z = g.vcycle(_rhs(g.level(0)[1], kind))
            out[mode] = {"z": z, "residual": g.get(hdd.CH_K)}
        finally:
            g.close()
    for what in ("z", "residual"):
        a, c = out["0"][what], out[""][what]
        print(f"[{name} {kind}] {what}: {np.isnan(a).sum()} / {np.isnan(c).sum()} not a number, {np.isinf(a).sum()} / {np.isinf(c).sum()} infinite "
              f"of {a.size}", flush=True)
        assert np.isnan(a).any() or np.isinf(a).any()
        assert np.array_equal(np.isnan(a), np.isnan(c))
        ok = ~np.isnan(a)
        assert np.array_equal(a[ok].view(np.uint32), c[ok].view(np.uint32))
