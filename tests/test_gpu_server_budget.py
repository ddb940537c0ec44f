"""A server whose HBM budget lies between a request's two estimates (33^3: 136 MB with the dense-node plans,
24 MB with the per-height ones, tests/test_device_bytes.py) solves it with the per-height plans; tolerances
as for any served request (iterations within +-1 of the solve alone, x within 1e-4)."""
import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import rel_err

pytestmark = pytest.mark.gpu


def test_request_beyond_the_budget_takes_the_per_height_plans():
    from hierarchicaldd_amd import hdd
    dom, cfg = domain.small_box(33, 16, 3, seed=1)
    tol = 1e-6 * float(np.abs(dom.b).max())
    g = hdd.DDSolver(dom, cfg)
    it, _, _ = g.solve(tol, 300)
    x = g.get(hdd.CH_X)
    g.close()
    srv = hdd.Server(setup_threads=1, groups=2, max_batch=2, hbm_budget=60e6)
    try:
        out = [srv.wait(k) for k in [srv.submit(dom, cfg, tol, 300) for _ in range(3)]]
    finally:
        srv.close()
    for st, xs, rep in out:
        print(f"alone {it} served {rep['iterations']}, x rel diff {rel_err(xs, x):.1e}", flush=True)
        assert st == 0 and abs(rep["iterations"] - it) <= 1 and rep["final_norm"] <= tol
        assert rel_err(xs, x) < 1e-4
