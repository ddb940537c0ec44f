"""Whole channels copied through the pinned ring: the bytes that come back are the bytes that went in, for
a channel of several chunks and a remainder, through two contexts at once, and for one below the ring's size."""
import threading

import numpy as np
import pytest

from hierarchicaldd_amd import domain
from tests.gpu_common import same_bits

pytestmark = pytest.mark.gpu


def _solver(n, sub, vlevels):
    from hierarchicaldd_amd import hdd
    return hdd.DDSolver(*domain.sphere_case(n, sub, vlevels))


@pytest.mark.parametrize("n,sub,vlevels", [(48, 16, 3), (104, 32, 4), (132, 32, 4)])
def test_channels_round_trip(n, sub, vlevels):
    from hierarchicaldd_amd import hdd
    g = _solver(n, sub, vlevels)
    try:
        rng = np.random.default_rng(n)
        print(f"[n {n}] {g.n_pages} pages, {g.n_pages / 4096:.2f} chunks", flush=True)
        sent = {ch: rng.standard_normal((g.n_pages, 256)).astype(np.float32) for ch in (hdd.CH_Z, hdd.CH_R, hdd.CH_X, hdd.CH_S)}
        for ch, v in sent.items():
            g.set(ch, v)
        for ch, v in sent.items():
            assert same_bits(g.get(ch), v)
    finally:
        g.close()


def test_two_contexts_at_once():
    from hierarchicaldd_amd import hdd
    gs = [_solver(104, 32, 4) for _ in range(2)]
    bad = []

    def work(g, seed):
        rng = np.random.default_rng(seed)
        for _ in range(4):
            v = rng.standard_normal((g.n_pages, 256)).astype(np.float32)
            g.set(hdd.CH_X, v)
            if not same_bits(g.get(hdd.CH_X), v):
                bad.append(seed)

    ts = [threading.Thread(target=work, args=(g, k)) for k, g in enumerate(gs)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    for g in gs:
        g.close()
    assert not bad
