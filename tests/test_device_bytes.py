"""The device bytes a problem is estimated to need, by which the server admits and refuses requests,
against the allocations of the context that is built, on the CPU with the HIP calls replaced
(tests/device_bytes_check.cpp). The estimate carries 10% and 4 MiB of margin; its terms are counts of
the arrays themselves, so it may exceed what is held by that and a few percent more."""
import os
import subprocess

import numpy as np
import pytest

from hierarchicaldd_amd import build, domain, hdd

HERE = os.path.dirname(os.path.abspath(__file__))
PACKED_OFF = ["-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]  # as the library is built


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    hdd.lib()
    d = tmp_path_factory.mktemp("device_bytes")
    exe = str(d / "device_bytes_check")
    cmd = [build.HIPCC, "-O1", "-std=c++17", "-fopenmp", "-rdynamic", "-x", "hip", "--offload-arch=gfx950", *PACKED_OFF, os.path.join(HERE, "device_bytes_check.cpp"),
           "-o", exe, "-L", build.OUT, "-lhdd", f"-Wl,-rpath,{build.OUT}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]

    def run(mode, arg, problems):
        files = []
        for k, (dom, cfg) in enumerate(problems):
            files.append(str(d / f"problem{k}.bin"))
            with open(files[-1], "wb") as f:
                np.array([dom.size[0], cfg.sub_size, cfg.vlevels, dom.n_pages], np.int32).tofile(f)
                np.asarray(dom.page_offsets, np.uint64).tofile(f)
                np.asarray(dom.flags, np.uint32).tofile(f)
                np.asarray(dom.b, np.float32).tofile(f)
        env = {k: v for k, v in os.environ.items() if not k.startswith("HDD_")}
        r = subprocess.run([exe, mode, str(arg)] + files, capture_output=True, text=True, timeout=300, env=env)
        assert r.returncode == 0, r.stdout + r.stderr
        return r.stdout.strip()
    return run


def _blocked(n, sub, vlevels, seed):
    rng = np.random.default_rng(seed)
    flags = domain.box_flags(n, domain.random_spheres(rng, n, 3, 0.1, 0.3), drop_enclosed=True)
    return domain.domain_from_flags(n, flags, rhs=rng.standard_normal((n, n, n))), domain.DDConfig(sub_size=sub, vlevels=vlevels)


CASES = {
    "sphere64_sub16": lambda: [domain.sphere_case(64, 16, 3)],   # many alike subdomains: blocks shared
    "blocked67_sub32": lambda: [_blocked(67, 32, 4, 1)],         # all different
    "box33_sub16": lambda: [domain.small_box(33, 16, 3, seed=1)],
    "sparse96_sub16": lambda: [domain.sparse_spheres(96, rmin=6, rmax=18, sub=16, vlevels=3)],
    "one_subdomain": lambda: [domain.small_box(32, 32, 4, seed=1)],
}


@pytest.mark.parametrize("name", list(CASES))
def test_estimate_covers_what_is_held(name, check):
    est, setup, held, peak = (int(v) for v in check("bytes", 0, CASES[name]()).split())
    print(f"[{name}] estimate {est / 1e6:.1f} MB, held {held / 1e6:.1f}; with set-up {(est + setup) / 1e6:.1f}, peak {peak / 1e6:.1f}")
    assert held <= est <= 1.25 * held + (5 << 20)
    assert peak <= est + setup <= 2.5 * peak + (5 << 20)


def test_estimate_of_the_per_height_plans(check):
    est, setup, held, peak = (int(v) for v in check("bytes", 1, [domain.small_box(33, 16, 3, seed=1)]).split())
    print(f"estimate {est / 1e6:.1f} MB, held {held / 1e6:.1f}, peak {peak / 1e6:.1f}")
    assert held <= est <= 1.25 * held + (5 << 20) and peak <= est + setup


def test_sum_covers_a_batch(check):
    est, setup, held, peak = (int(v) for v in check("bytes", 0, [_blocked(45, 16, 3, 2), domain.small_box(33, 16, 3, seed=1)]).split())
    print(f"estimate {est / 1e6:.1f} MB, held {held / 1e6:.1f}, peak {peak / 1e6:.1f}")
    assert held <= est and peak <= est + setup


def test_tight_budget_takes_the_smaller_plans(check):
    problem = [domain.small_box(33, 16, 3, seed=1)]
    nodes, heights = (int(check("bytes", h, problem).split()[0]) for h in (0, 1))
    assert heights < nodes
    assert check("server", nodes, problem) == "done 0"
    assert check("server", nodes - 1, problem) == "done 1"
    assert check("server", heights, problem) == "done 1"
    assert check("server", heights - 1, problem).startswith("failed: problem needs more device memory")


def test_context_falls_back_when_the_dense_nodes_do_not_fit(check):
    problem = [domain.small_box(33, 16, 3, seed=1)]
    nodes, heights = (int(check("bytes", h, problem).split()[3]) for h in (0, 1))  # peaks of the two forms
    assert check("create", nodes, problem) == f"{nodes} 1"
    peak, dense = (int(v) for v in check("create", nodes - 1, problem).split())
    assert dense == 0 and peak < nodes
    assert check("create", heights, problem) == f"{heights} 0"
    assert check("create", heights // 2, problem).startswith("failed: hipMalloc")
