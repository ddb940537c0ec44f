"""Copies between the caller's memory and the device: pageable memory through the pinned ring, memory that
is pinned already in one copy of the runtime's (tests/host_stage_check.cpp, on the CPU, the HIP calls
replaced)."""
import os
import subprocess

from hierarchicaldd_amd import build, hdd

HERE = os.path.dirname(os.path.abspath(__file__))
PACKED_OFF = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]  # as the library is built


def test_pinned_memory_skips_the_ring(tmp_path):
    hdd.lib()
    exe = str(tmp_path / "host_stage_check")
    cmd = [build.HIPCC, "-O1", "-std=c++17", "-fopenmp", "-rdynamic", "-x", "hip", "--offload-arch=gfx950", *PACKED_OFF, os.path.join(HERE, "host_stage_check.cpp"),
           "-o", exe, "-L", build.OUT, "-lhdd", f"-Wl,-rpath,{build.OUT}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
