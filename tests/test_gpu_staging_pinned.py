"""Whole channels from and to memory that the caller has pinned: the bytes that come back are the bytes
that went in, also mixed with pageable memory."""
import ctypes as C

import pytest
import torch

from hierarchicaldd_amd import domain

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,sub,vlevels", [(48, 16, 3), (104, 32, 4)])  # below and above the ring's size
def test_pinned_channels_round_trip(n, sub, vlevels):
    from hierarchicaldd_amd import hdd
    g = hdd.DDSolver(*domain.sphere_case(n, sub, vlevels))
    L = hdd.lib()
    try:
        cells = g.n_pages * 256
        print(f"[n {n}] {cells * 4e-6:.1f} MB", flush=True)
        gen = torch.Generator().manual_seed(n)
        v = torch.randn(cells, generator=gen)
        pinned_in = torch.empty(cells, pin_memory=True)
        pinned_in.copy_(v)
        pinned_out, out = torch.zeros(cells, pin_memory=True), torch.zeros(cells)
        ptr = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
        assert L.hdd_set_channel(g.h, hdd.CH_X, ptr(pinned_in)) == 0
        assert L.hdd_get_channel(g.h, hdd.CH_X, ptr(out)) == 0
        assert torch.equal(out, v)
        assert L.hdd_set_channel(g.h, hdd.CH_S, ptr(v)) == 0
        assert L.hdd_get_channel(g.h, hdd.CH_S, ptr(pinned_out)) == 0
        assert torch.equal(pinned_out, v)
    finally:
        g.close()
