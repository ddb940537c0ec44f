"""The interface V-cycle on the device against the same cycle composed in double from the context's own
operators and host factors: edges that leave partial slices of 64 rows, one and several cycles and
smooths, and no smooths at all (where a level starts from u = 0 without a solve).

Bar: each exact solve is within 1e-7 to 2e-7 of its double value, a smooth has two, and the smoother does not
amplify an error (its iteration matrix has eigenvalues in [0, 1)); two cycles of 2 * 2 * 3 + 1 smooths
are 25 * 2 * 1e-7 = 5e-6 of the largest value, 1e-5 with the sparse products' own rounding."""
import numpy as np
import pytest
from scipy.sparse import csr_matrix

from hierarchicaldd_amd import domain

pytestmark = pytest.mark.gpu


class HostCycle:
    def __init__(self, g, cfg):
        self.g, self.cfg = g, cfg
        self.L, self.nsub = g.sigma_info()
        self.n = [g.interface_dofs(l) for l in range(self.L)]

    def mat(self, which, l, sub=0):
        rows, _, ptr, idx, val = self.g.matrix(which, l, sub)
        cols = self.n[l + 1] if which == "Prr" else self.n[l]
        return csr_matrix((val.astype(np.float64), idx, ptr), shape=(rows, cols))

    def coupled(self, l, u):
        out = np.zeros(self.n[l])
        for s in range(self.nsub):
            A = self.mat("Air", l, s)
            if A.shape[0]:
                out += A.T @ self.g.sigma_factor_solve(l, "Aii", s, A @ u)
        return out

    def smooth(self, l, b, u):
        return self.g.sigma_factor_solve(l, "Arr", 0, b + self.coupled(l, u))

    def cycle(self, l, b, u):
        if l == self.L - 1:
            for _ in range(200):
                u = self.smooth(l, b, u)
            return u
        for _ in range(self.cfg.sigma_smoothing):
            u = self.smooth(l, b, u)
        r = b + self.coupled(l, u) - self.mat("Arr", l) @ u
        P = self.mat("Prr", l)
        u = u + P @ self.cycle(l + 1, P.T @ r, np.zeros(self.n[l + 1]))
        for _ in range(self.cfg.sigma_smoothing):
            u = self.smooth(l, b, u)
        return u


@pytest.mark.parametrize("n,sub,smoothing,cycles", [(33, 16, 3, 1), (37, 16, 1, 2), (33, 16, 0, 1), (33, 16, 0, 2), (45, 32, 2, 1)])
def test_vcycle_against_its_operators(n, sub, smoothing, cycles):
    from hierarchicaldd_amd import hdd
    dom, cfg = domain.small_box(n, sub, 3 if sub == 16 else 4, seed=n)
    cfg.sigma_smoothing, cfg.sigma_mg = smoothing, cycles
    g = hdd.DDSolver(dom, cfg)
    try:
        H = HostCycle(g, cfg)
        print(f"[box {n}] interface dofs {H.n}", flush=True)
        b = np.random.default_rng(n).standard_normal(H.n[0]).astype(np.float32)
        ref = np.zeros(H.n[0])
        for _ in range(cycles):
            ref = H.cycle(0, b.astype(np.float64), ref)
        for _ in range(2):  # the second call finds the first one's values in the buffers
            got = g.sigma_vcycle(b)
            assert np.abs(got - ref).max() <= 1e-5 * np.abs(ref).max()
    finally:
        g.close()
