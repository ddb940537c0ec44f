"""A V-cycle whose clusters take more than 64 KiB of LDS (19^3 cells of a subdomain of 20) sets no kernel
attributes: its plan did (tests/cluster_launch_check.cpp, on the CPU, the HIP calls replaced)."""
import os
import subprocess

from hierarchicaldd_amd import build, hdd

HERE = os.path.dirname(os.path.abspath(__file__))
PACKED_OFF = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]  # as the library is built


def test_attributes_are_set_with_the_plan(tmp_path):
    hdd.lib()
    exe = str(tmp_path / "cluster_launch_check")
    cmd = [build.HIPCC, "-O1", "-std=c++17", "-fopenmp", "-rdynamic", "-x", "hip", "--offload-arch=gfx950", *PACKED_OFF, os.path.join(HERE, "cluster_launch_check.cpp"),
           "-o", exe, "-L", build.OUT, "-lhdd", f"-Wl,-rpath,{build.OUT}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    env = {k: v for k, v in os.environ.items() if not k.startswith("HDD_")}
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120, env=env)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
