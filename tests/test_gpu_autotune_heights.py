"""The launch-shape autotuner on the plans it works on: the per-height ones, of at least 20,000 rows, which
contexts hold where HDD_DENSE_TOP asks for them and refined solves use (a default context has dense nodes,
which are not tuned). Rows per slice, entries per item, workgroups and the wavefront form of a fused
height are chosen by timing and must not change a bit: histories and solutions with the tuner on and off
(HDD_AUTOTUNE=0)."""
import os

import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import same_bits

pytestmark = pytest.mark.gpu

CASES = {
    "sphere64_sub16": domain.config0,
    "box48_sub16": lambda: domain.small_box(48, 16, 3, seed=2),
    "sphere96_sub32": lambda: domain.sphere_case(96, 32, 4, delta=(32, 32, 32)),  # a fused height (1024 supernodes at one height)
}


@pytest.mark.parametrize("refined", [False, True])
@pytest.mark.parametrize("case", list(CASES))
def test_tuned_plans_bit_identical(case, refined):
    from hierarchicaldd_amd import hdd
    dom, cfg = CASES[case]()
    tol = 1e-6 * float(np.abs(dom.b).max())
    out = {}
    for mode in ("0", "1"):
        env = {"HDD_AUTOTUNE": mode} if refined else {"HDD_AUTOTUNE": mode, "HDD_DENSE_TOP": "0"}
        os.environ.update(env)
        try:
            g = hdd.DDSolver(dom, cfg)
            if refined:
                assert g.stats()["tuned_plans"] == 0
                g.set_sigma_refinement(1)
        finally:
            for k in env:
                os.environ.pop(k, None)
        it, hist, _ = g.solve(tol, 300)
        out[mode] = (it, hist, g.get(hdd.CH_X), g.stats())
        g.close()
    off, on = out["0"], out["1"]
    print(f"[{case}, refined {refined}] iterations {off[0]} / {on[0]}, plans timed {on[3]['tuned_plans']:.0f}, shapes changed "
          f"{on[3]['tuned_launch_shapes']:.0f}, wavefront heights {on[3]['wave_heights']:.0f} of {on[3]['fused_heights']:.0f}")
    assert off[3]["tuned_plans"] == 0 and off[3]["tuned_launch_shapes"] == 0
    assert on[3]["tuned_plans"] >= 1
    assert off[0] == on[0] and np.array_equal(off[1], on[1])
    assert same_bits(off[2], on[2])
