"""hdd_set_sigma_refinement builds the per-height plans of a live context: out of device memory in the
middle of it, the call fails, leaves no plan half there, and can be made again. On the CPU, with the
HIP memory calls replaced (tests/refinement_check.cpp)."""
import os
import subprocess

from hierarchicaldd_amd import build, hdd

HERE = os.path.dirname(os.path.abspath(__file__))
PACKED_OFF = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]  # as the library is built


def test_failed_refinement_can_be_retried(tmp_path):
    hdd.lib()
    exe = str(tmp_path / "refinement_check")
    cmd = [build.HIPCC, "-O1", "-std=c++17", "-fopenmp", "-rdynamic", "-x", "hip", "--offload-arch=gfx950", *PACKED_OFF, os.path.join(HERE, "refinement_check.cpp"),
           "-o", exe, "-L", build.OUT, "-lhdd", f"-Wl,-rpath,{build.OUT}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-2000:]
