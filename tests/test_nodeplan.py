"""The dense-node plans of the interface solver's exact solves, on the CPU: every index the kernels
use stays inside its array, and the plan carried out in double gives the solves of its factors
(tests/nodeplan_check.cpp). The bar, 1e-11 relative, is double rounding through a few hundred
terms per row (n eps ~ 5e-14) times the 7-point operators' condition of at most a few hundred."""
import ctypes as C
import os
import subprocess

import pytest

from hierarchicaldd_amd import build, hdd

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("nodeplan") / "nodeplan_check.so")
    cmd = [build.HIPCC, "-O2", "-std=c++17", "-fPIC", "-shared", "-x", "hip", "--offload-arch=gfx950", os.path.join(HERE, "nodeplan_check.cpp"),
           "-o", lib, "-L", build.OUT, "-lhdd", f"-Wl,-rpath,{build.OUT}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    hdd.lib()
    L = C.CDLL(lib)
    L.nodeplan_check.argtypes = [C.c_int] * 7 + [C.POINTER(C.c_double), C.c_char_p, C.c_int]
    return L.nodeplan_check


@pytest.mark.parametrize("box,hole,copies,other,leaf", [
    ((1, 1, 1), 0, 1, 0, 96),      # one row: a block of one tile
    ((2, 4, 2), 0, 1, 1, 96),      # 16 rows: exactly one tile
    ((17, 1, 1), 0, 3, 1, 4),      # 17 rows, a chain of tiny supernodes
    ((5, 5, 7), 0, 15, 1, 96),     # a run of 16 and one more block
    ((5, 5, 7), 0, 17, 1, 96),     # a second run of two
    ((9, 11, 13), 0, 2, 1, 96),    # several heights
    ((24, 9, 9), 17, 1, 1, 48),    # two pieces: a forest
    ((20, 20, 20), 0, 4, 1, 96),
    ((20, 20, 20), 12, 20, 1, 96),
    ((33, 31, 29), 0, 1, 0, 96),   # more than one level
])
def test_plan_solves_its_factors(check, box, hole, copies, other, leaf):
    out = (C.c_double * 5)()
    msg = C.create_string_buffer(256)
    assert check(*box, hole, copies, other, leaf, out, msg, 256) == 0, msg.value.decode()
    print(f"error {out[0]:.1e}, {out[1]:.0f} levels, {out[2]:.0f} blocks for {out[3]:.0f} nodes, largest {out[4]:.0f} rows")
    assert out[0] < 1e-11
    # the copies and the equal factor share their blocks
    nodes = out[3] / (copies + 1 + other)
    assert out[2] <= nodes * (1 + other)
