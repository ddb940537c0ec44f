"""Performance cases of the DD-PCG solver: what its users call, over the range they call it in.

The framework solves the variable-domain Poisson equation on paged SPGrid domains. A program
sets a geometry up once (hdd.DDSolver / hdd.DDBatch: flags, interface operators, factors, device
plans) and then calls it with right-hand sides: whole solves, the preconditioner or the interface
solver inside a loop of its own, the Krylov plugin surface, or the context-free inner product.

Every case is a dict:
  kind      "dot"    hdd_inner_product_noalloc on two device arrays of `pages` pages
            "solve"  DDSolver.solve to max|r| <= tol * max|b|, then x
            "krylov" a PCG loop of the caller's own on the device channels, then x
            "sigma"  DDSolver.sigma_vcycle: one interface multigrid V-cycle
            "apply"  DDSolver.apply_preconditioner: z = M^-1 r
            "batch"  DDBatch.solve_all of `count` uneven problems in one context, then each x
  geometry  "sphere"  n^3 box, Dirichlet ring, one sphere obstacle of radius n/4
            "blocked" the same box with 1-4 random sphere obstacles (geometry_seed)
            "sparse"  union of seeded spheres in a zero-Dirichlet box
  n, sub, vlevels    edge, subdomain edge, V-cycle levels (the reference pairs 16 with 3, 32 with 4)

The geometry is the case's; the seed draws the right-hand side: N(0,1) on the Active cells, as the
served requests carry. Solves run to 1e-6 of max|b|, the framework's stated tolerance, except the
FP64 outer loop, which is there for 1e-8.
"""
from __future__ import annotations

import ctypes
import functools
import math

import numpy as np
import torch

from hierarchicaldd_amd import domain, hdd

MAX_ITERATIONS = 500
ACTIVE, FACE0 = domain.ACTIVE, domain.FACE_MX


def listed():
    return [
        # the inner product a tight loop or a graph capture calls on its own arrays: the page counts
        # of the 64^3 domain (a call is all latency) and of the 256^3 domain (memory bandwidth)
        {"name": "dot_64", "kind": "dot", "pages": 1003},
        {"name": "dot_256", "kind": "dot", "pages": 62075},
        # whole solves of small problems, where every launch counts: the smallest served size, and
        # the 64^3 sphere at both subdomain sizes
        {"name": "solve_32", "kind": "solve", "geometry": "sphere", "n": 32, "sub": 16, "vlevels": 3, "tol": 1e-6},
        {"name": "solve_64_sub16", "kind": "solve", "geometry": "sphere", "n": 64, "sub": 16, "vlevels": 3, "tol": 1e-6},
        {"name": "solve_64_sub32", "kind": "solve", "geometry": "sphere", "n": 64, "sub": 32, "vlevels": 4, "tol": 1e-6},
        # an ordinary request: an edge no page or subdomain divides, several obstacles
        {"name": "solve_100_blocked", "kind": "solve", "geometry": "blocked", "geometry_seed": 0, "n": 100, "sub": 32, "vlevels": 4,
         "tol": 1e-6},
        # the sparse domain at high accuracy: FP64 outer loop to 1e-8
        {"name": "solve_96_sparse_fp64", "kind": "solve", "geometry": "sparse", "geometry_seed": 0, "n": 96, "sub": 16, "vlevels": 3,
         "tol": 1e-8, "fp64": True},
        # a program's own Krylov loop on device channels through the plugin surface
        {"name": "krylov_96", "kind": "krylov", "geometry": "sphere", "n": 96, "sub": 16, "vlevels": 3, "tol": 1e-6},
        # a handful of uneven problems in one context
        {"name": "batch_6", "kind": "batch", "geometry": "blocked", "geometry_seed": 0, "n": 64, "count": 6, "sub": 32, "vlevels": 4,
         "tol": 1e-6},
        # the interface solver alone
        {"name": "sigma_128_blocked", "kind": "sigma", "geometry": "blocked", "geometry_seed": 0, "n": 128, "sub": 32, "vlevels": 4},
        # the preconditioner, which is nearly all of a PCG iteration, at an ordinary large size and on
        # the 256^3 sphere domain of the headline benchmark (the largest case)
        {"name": "apply_160_blocked", "kind": "apply", "geometry": "blocked", "geometry_seed": 0, "n": 160, "sub": 32, "vlevels": 4},
        {"name": "apply_256", "kind": "apply", "geometry": "sphere", "n": 256, "sub": 32, "vlevels": 4},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["dot", "solve", "solve", "solve", "krylov", "sigma", "apply", "batch"])
    if kind == "dot":
        return {"kind": kind, "pages": log_int(64, 62075)}
    top = {"solve": 100, "krylov": 96, "sigma": 160, "apply": 160, "batch": 64}[kind]
    low = 40 if kind == "sigma" else 32  # an edge of 32 is one subdomain of 32: no interface
    case = {"kind": kind, "geometry": rng.choice(["sphere", "blocked", "blocked", "sparse"]), "geometry_seed": rng.randrange(1 << 16),
            "n": log_int(low, top), "tol": 1e-6}
    if kind == "batch":
        case.update(geometry="blocked", count=rng.randint(2, 6))
    if case["geometry"] == "sparse":
        case["n"] = max(case["n"], 64)
    sub16 = case["n"] <= 100 and rng.random() < 0.5
    case.update(sub=16 if sub16 else 32, vlevels=3 if sub16 else 4)
    if kind == "solve" and rng.random() < 0.2:
        case.update(tol=1e-8, fp64=True)
    return case


# ---- inputs -------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=16)
def _geometry(kind, n, geometry_seed):
    """Dense flags of a box geometry (padded to whole pages), or the sparse domain."""
    rng = np.random.default_rng(geometry_seed)
    if kind == "sphere":
        return domain.box_flags(n, [(n // 2, n // 2, n // 2, n // 4)])
    if kind == "blocked":
        return domain.box_flags(n, domain.random_spheres(rng, n, int(rng.integers(1, 5)), 0.1, 0.3), drop_enclosed=True)
    return domain.sparse_spheres(n, rmin=n / 16, rmax=3 * n / 16, seed=geometry_seed)[0]


def _edge(case, index):
    """Edge of problem `index` of a case (a batch's problems are uneven)."""
    return case["n"] if index == 0 else max(32, case["n"] - 8 * index)


def _domain(case, seed, index=0):
    n = _edge(case, index)
    geometry = _geometry(case["geometry"], n, case.get("geometry_seed", 0) + 7919 * index)
    rng = np.random.default_rng([seed, index])
    if case["geometry"] == "sparse":
        flags = geometry.flags
        b = np.where(flags & ACTIVE, rng.standard_normal(flags.shape, dtype=np.float32), np.float32(0))
        return domain.SPGridDomain(geometry.size, geometry.page_offsets, flags, b)
    return domain.domain_from_flags(n, geometry, rhs=rng.standard_normal((n, n, n), dtype=np.float32))


def _domains(case, seed):
    return [_domain(case, seed, i) for i in range(case.get("count", 1))]


def _config(case):
    return domain.DDConfig(sub_size=case["sub"], vlevels=case["vlevels"])


def _tolerance(case, dom):
    return case["tol"] * float(np.abs(dom.b).max())


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _dot_arrays(case, seed):
    gen = torch.Generator().manual_seed(seed)
    return [torch.randn(case["pages"] * 256, generator=gen) for _ in range(2)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "dot":
        a, b = (t.to(_device()) for t in _dot_arrays(case, seed))
        return {"kind": kind, "pages": case["pages"], "a": a, "b": b, "out": torch.zeros(1, dtype=torch.float64, device=a.device)}
    doms = _domains(case, seed)
    cfg = _config(case)
    if kind == "batch":
        return {"kind": kind, "solver": hdd.DDBatch([(d, cfg) for d in doms]), "tol": [_tolerance(case, d) for d in doms]}
    dom = doms[0]
    solver = hdd.DDSolver(dom, cfg)
    state = {"kind": kind, "solver": solver}
    if kind in ("solve", "krylov"):
        state["tol"] = _tolerance(case, dom)
        if case.get("fp64"):
            solver.set_outer_fp64(True)
    elif kind == "sigma":
        state["b"] = np.random.default_rng(seed).standard_normal(solver.interface_dofs(0), dtype=np.float32)
    else:
        state["r"] = dom.b  # the first residual of a solve from x = 0
    return state


# ---- one pass -----------------------------------------------------------------------------------

def _ok(solver, status):
    if status != 0:
        raise hdd.HddError(hdd.lib().hdd_last_error(solver.h).decode())


def _krylov(solver, tol):
    """Preconditioned CG through the plugin surface, x starting at zero."""
    L, h = hdd.lib(), solver.h
    Z, R, K, X, B, Q, S = hdd.CH_Z, hdd.CH_R, hdd.CH_K, hdd.CH_X, hdd.CH_B, hdd.CH_Q, hdd.CH_S
    value, norm = ctypes.c_double(), ctypes.c_float()

    def do(name, *args):
        _ok(solver, getattr(L, name)(h, *args))

    def dot(a, b):
        do("hdd_inner_product", a, b, ctypes.byref(value))
        return np.float32(value.value)

    do("hdd_vector_scale", X, 0.0)
    do("hdd_vector_copy", R, 1.0, B)
    do("hdd_project", R)
    rho_old = None
    for _ in range(MAX_ITERATIONS):
        do("hdd_convergence_norm", R, ctypes.byref(norm))
        if norm.value <= tol:
            break
        do("hdd_apply_preconditioner_channels", Z, R, K)
        rho = dot(Z, R)
        if rho_old is None:
            do("hdd_vector_copy", S, 1.0, Z)
        else:
            do("hdd_vector_copy2", S, float(rho / rho_old), S, Z)
        do("hdd_multiply", S, Q)
        do("hdd_project", Q)
        alpha = rho / dot(S, Q)
        do("hdd_vector_copy2", X, float(alpha), S, X)
        do("hdd_vector_copy2", R, float(-alpha), Q, R)
        rho_old = rho
    return solver.get(X)


def run(state):
    kind = state["kind"]
    if kind == "dot":
        stream = torch.cuda.current_stream().cuda_stream
        st = hdd.lib().hdd_inner_product_noalloc(state["a"].data_ptr(), state["b"].data_ptr(), state["pages"], state["out"].data_ptr(), stream)
        if st != 0:
            raise hdd.HddError(hdd.lib().hdd_last_error(None).decode())
        return state["out"]
    solver = state["solver"]
    if kind == "solve":
        solver.solve(state["tol"], MAX_ITERATIONS)
        return solver.get(hdd.CH_X)
    if kind == "krylov":
        return _krylov(solver, state["tol"])
    if kind == "sigma":
        return solver.sigma_vcycle(state["b"])
    if kind == "apply":
        return solver.apply_preconditioner(state["r"])
    solver.solve_all(state["tol"], MAX_ITERATIONS)
    return [solver.x(p) for p in range(solver.count)]


# ---- what a pass cannot do without --------------------------------------------------------------

_FILL = {"sphere": 0.93, "blocked": 0.87, "sparse": 0.35}  # Active share of the box


def _sigma_work(n, sub):
    """Distinct factor entries that one interface V-cycle applies, twice each (forward, backward):
    3 smooths before and after the coarse level and one residual per level. Entries per row of an
    interface factor grow with the logarithm of its rows (62 at 31k rows, 110 at 1.2M); a
    subdomain's factor holds about 90k entries at sub 16 and 640k at sub 32 (a fifth of that one level
    down), and subdomains of one shape share theirs. The last term is the bottom's combined system."""
    per_axis = max(1, n // sub)
    rows = max(64.0, 3.0 * n * n * (per_axis - 0.5) * 0.9)
    entries = 0.0
    for level, scale in enumerate((1.0, 0.33)):
        m = rows * scale
        arr = m * max(20.0, 9.0 * math.log2(m) - 72.0)
        aii = min(per_axis ** 3, 27) * (90e3 if sub == 16 else 640e3) * (1.0, 0.18)[level]
        entries += 6 * arr + 7 * aii
    entries += 0.078 * rows * max(20.0, 9.0 * math.log2(rows) - 72.0) * 9.0
    return 2 * 4.0 * entries, 4.0 * entries


def _apply_work(case, n):
    """Two V-cycles (14 level-0 sweeps of 16 B and about 10 flops a cell, the coarse levels 1/7 more)
    around one interface V-cycle."""
    cells = n ** 3 * _FILL[case["geometry"]]
    by, fl = _sigma_work(n, case["sub"])
    return by + 14 * 16.0 * cells * 8 / 7, fl + 14 * 20.0 * cells * 8 / 7


def work(case):
    kind = case["kind"]
    if kind == "dot":
        cells = case["pages"] * 256
        return {"bytes": 8.0 * cells + 8, "flops": 2.0 * cells}
    if kind == "sigma":
        by, fl = _sigma_work(case["n"], case["sub"])
        return {"bytes": by, "flops": fl}
    if kind == "apply":
        by, fl = _apply_work(case, case["n"])
        return {"bytes": by, "flops": fl}
    by = fl = 0.0
    for i in range(case.get("count", 1)):
        n = _edge(case, i)
        iterations = 10 + 0.2 * n  # measured 11 at 32, 18 at 64, 27 at 96-100, 50 at 160
        b, f = _apply_work(case, n)
        cells = n ** 3 * _FILL[case["geometry"]]
        by += iterations * (b + 60.0 * cells)
        fl += iterations * (f + 30.0 * cells)
    return {"bytes": by, "flops": fl}


# ---- the same results in 64 bits ----------------------------------------------------------------

def _cells_of_pages(offsets):
    """Cell coordinates [pages, 256, 3] of SPGrid page offsets: the page index interleaves the bits of
    the block coordinates as x, z, y from the lowest; a page is 4 x 8 x 8 cells, z fastest."""
    m = (offsets >> np.uint64(12)).astype(np.int64)
    block = np.zeros((len(m), 3), dtype=np.int64)
    for k in range(21):
        for bit, axis in ((0, 0), (1, 2), (2, 1)):
            block[:, axis] |= ((m >> (3 * k + bit)) & 1) << k
    c = np.arange(256)
    cell = np.stack([c >> 6, (c >> 3) & 7, c & 7], axis=1)
    return block[:, None, :] * np.array([4, 8, 8]) + cell[None]


def _solution(dom):
    """x of A x = b in float64 by conjugate gradients: face f of an Active cell couples it to its
    neighbour (zero where that is Dirichlet), obstacle faces are open (Neumann)."""
    dev = _device()
    cells = _cells_of_pages(dom.page_offsets)
    shape = tuple(int(v) + 2 for v in cells.reshape(-1, 3).max(axis=0) + 1)  # one cell of padding all round
    index = ((cells[..., 0] + 1) * shape[1] + cells[..., 1] + 1) * shape[2] + cells[..., 2] + 1
    index = torch.from_numpy(index.reshape(-1)).to(dev)
    size = shape[0] * shape[1] * shape[2]
    flags = torch.zeros(size, dtype=torch.int64, device=dev)
    flags[index] = torch.from_numpy(dom.flags.reshape(-1).astype(np.int64)).to(dev)
    b = torch.zeros(size, dtype=torch.float64, device=dev)
    b[index] = torch.from_numpy(dom.b.reshape(-1).astype(np.float64)).to(dev)
    active = (flags & ACTIVE) != 0
    b[~active] = 0
    shifts = [-shape[1] * shape[2], shape[1] * shape[2], -shape[2], shape[2], -1, 1]
    faces = [(((flags & (FACE0 << f)) != 0) & active).double() for f in range(6)]
    diag = sum(faces)
    # coupling to Active neighbours only: x is zero elsewhere and stays so
    off = [w * torch.roll(active, -s).double() for w, s in zip(faces, shifts)]

    def apply(v):
        out = diag * v
        for w, s in zip(off, shifts):
            out -= w * torch.roll(v, -s)
        return out

    inv = torch.where(diag > 0, 1.0 / diag.clamp(min=1.0), torch.zeros_like(diag))
    x = torch.zeros_like(b)
    r = b.clone()
    z = inv * r
    p = z.clone()
    rho = torch.dot(r, z)
    stop = 1e-13 * float(r.abs().max())
    for k in range(20000):
        q = apply(p)
        alpha = rho / torch.dot(p, q)
        x += alpha * p
        r -= alpha * q
        if k % 20 == 19 and float(r.abs().max()) <= stop:
            break
        z = inv * r
        rho_new = torch.dot(r, z)
        p = z + (rho_new / rho) * p
        rho = rho_new
    return x[index].reshape(-1, 256).cpu().numpy()


def exact(case, seed):
    kind = case["kind"]
    if kind == "dot":
        a, b = _dot_arrays(case, seed)
        return (a.double() * b.double()).sum().reshape(1)
    if kind in ("sigma", "apply"):
        # the preconditioner is the framework's own operator: nothing outside it gives its values
        return None
    xs = [_solution(d) for d in _domains(case, seed)]
    return xs if kind == "batch" else xs[0]
