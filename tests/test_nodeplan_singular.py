"""Dense-node plans where the matrix is nearly singular (no Dirichlet cell: A 1 = 1e-5), on the CPU in
float as the kernels work (tests/nodeplan_singular_check.cpp): a node without boundary rows then keeps
its triangle instead of its inverse, whose rounding would leave an error of 1e-4 to 1e-3 in every row.

Bar, for the error outside the constant: a solve rounds its operands and sums a few times to 2^-24, which
perturbs the system by at most 4 * 2^-24 of its largest eigenvalue (< 12) and so the solution by that over
the smallest eigenvalue outside the constant, 2 - 2 cos(pi / n) of the longest edge n (the rest of the
spectrum of the box without Dirichlet cells; for the other boxes, more)."""
import ctypes as C
import math
import os
import subprocess

import pytest

from hierarchicaldd_amd import build, hdd

HERE = os.path.dirname(os.path.abspath(__file__))
PACKED_OFF = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]  # as the library is built


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    lib = str(tmp_path_factory.mktemp("nodeplan") / "nodeplan_singular_check.so")
    cmd = [build.HIPCC, "-O2", "-std=c++17", "-fPIC", "-shared", "-x", "hip", "--offload-arch=gfx950", *PACKED_OFF,
           os.path.join(HERE, "nodeplan_singular_check.cpp"), "-o", lib, "-L", build.OUT, "-lhdd", f"-Wl,-rpath,{build.OUT}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    hdd.lib()
    L = C.CDLL(lib)
    L.nodeplan_singular_check.argtypes = [C.c_int] * 6 + [C.POINTER(C.c_double), C.c_char_p, C.c_int]
    return L.nodeplan_singular_check


NEUMANN, RING, FACE, CELL = 0, 1, 2, 3


@pytest.mark.parametrize("box,ring,copies,leaf,inverse", [
    ((9, 9, 9), NEUMANN, 1, 96, False),
    ((13, 13, 13), NEUMANN, 1, 96, False),
    ((9, 5, 3), NEUMANN, 3, 4, False),      # a run of three
    ((2, 4, 2), NEUMANN, 1, 96, False),     # 16 rows: exactly one tile
    ((20, 13, 11), NEUMANN, 1, 96, False),  # more than one level
    ((9, 9, 9), RING, 2, 96, True),         # Dirichlet cells all around, on one face: the inverse as before
    ((13, 13, 13), FACE, 1, 96, True),
    ((13, 13, 13), CELL, 1, 96, False),     # one Dirichlet neighbour for 2197 cells
])
def test_nearly_singular(check, box, ring, copies, leaf, inverse):
    out = (C.c_double * 4)()
    msg = C.create_string_buffer(256)
    assert check(*box, ring, copies, leaf, out, msg, 256) == 0, msg.value.decode()
    bar = 4 * 2.0 ** -24 * 12 / (2 - 2 * math.cos(math.pi / max(box)))
    print(f"error outside the constant {out[0]:.1e} (bar {bar:.1e}), {out[2]:.0f} of {out[1]:.0f} closed nodes hold their inverse, "
          f"in double {out[3]:.1e}")
    assert out[1] >= 1 and out[2] == (out[1] if inverse else 0)
    assert out[0] < bar
    # in double: the condition, 12 / 1e-5, times some hundred roundings
    assert out[3] < 1e-16 * 1.2e6 * 300
