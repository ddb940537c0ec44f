"""Clusters of the largest kind the cluster sweeps take: 19^3 cells (a subdomain of 20), seven or eight
cells a thread, more than 64 KiB of LDS; equal bits with one launch per sweep (HDD_BOTTOM_LOCAL=0), in
FP32 and FP16 storage."""
import os

import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import random_rhs, same_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fp16", [False, True])
@pytest.mark.parametrize("vlevels", [1, 3])
def test_wide_clusters_bitwise(vlevels, fp16):
    from hierarchicaldd_amd import hdd
    dom, cfg = domain.small_box(41, 20, vlevels, seed=8)
    print(f"[box41_sub20 vlevels {vlevels} fp16 {fp16}]", flush=True)
    out = {}
    for mode in ("0", ""):
        os.environ["HDD_BOTTOM_LOCAL"] = mode
        try:
            g = hdd.DDSolver(dom, cfg)
        finally:
            os.environ.pop("HDD_BOTTOM_LOCAL", None)
        try:
            g.set_fp16(fp16)
            b = random_rhs(g.level(0)[1], 17)
            out[mode] = (g.stats()["bottom_page_local"], g.apply_preconditioner(b), g.apply_preconditioner(b[:, ::-1].copy()))
        finally:
            g.close()
    a, c = out["0"], out[""]
    assert a[0] == 0 and c[0] == 1
    assert np.isfinite(c[1]).all()
    assert same_bits(a[1], c[1]) and same_bits(a[2], c[2])
