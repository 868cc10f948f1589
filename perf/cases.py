"""Performance cases: the work that programs built on this package have it do, over its range.

A case is a dict of plain values.  Its `kind` names one pass through the public API:

  count      update! + neighbour count of a cloud (2D or 3D; FullGrid, a periodic box or spatial
             hashing): what a program does that rebuilds its neighbourhoods every step
  wcsph      one step of weakly compressible SPH: update! + density + equation of state +
             pressure acceleration
  grad       the same step and the gradient of sum |a|^2 with respect to the positions
  interact   update! + TrixiParticles' fluid interact! (the reference's WCSPH benchmark)
  nbody      binning of two different point sets + the n-body closure (the reference's n-body
             benchmark, with probes that are not the bodies)
  periodic   update! + neighbour count + density in a periodic box
  csr        precomputed neighbour lists: build + a density sum over the stored lists
  tlsph      one evaluation of a total-Lagrangian solid over frozen lists: deformation gradient,
             stress, interaction forces
  batch      update! + neighbour count of many uneven independent clouds at once

Clouds are jittered lattices, as in this repository's benchmark and the reference's: `nx`, `ny`,
`nz` points per side (`nz` 0: two dimensions), search radius `factor` lattice spacings.
"""

import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "pointneighbors.jl_amd"))

import pointneighbors as pn  # noqa: E402
from pointneighbors import batch as pn_batch  # noqa: E402
from pointneighbors import sph  # noqa: E402

RHO0, SOUND, GAMMA = 1000.0, 10.0, 7.0
YOUNG, POISSON, PENALTY = 1.4e6, 0.4, 0.1
EOS_B = RHO0 * SOUND**2 / GAMMA


def listed():
    def case(name, kind, nx, ny, nz, factor, dtype="f32", cells="grid", **more):
        return dict(name=name, kind=kind, nx=nx, ny=ny, nz=nz, factor=factor, dtype=dtype, cells=cells, **more)

    return [
        # a small 2D cloud, as in the tutorials: a call is launches and latency
        case("count-2d-2k", "count", 45, 44, 0, 3.0),
        # a small fluid: every step is short and there are many
        case("wcsph-16k", "wcsph", 24, 25, 26, 2.4),
        # the benchmark's fluid
        case("wcsph-1m", "wcsph", 100, 100, 100, 2.4),
        # differentiable simulation: forward and adjoint
        case("grad-2m", "grad", 127, 128, 130, 2.4),
        # the reference's published fluid benchmark, in both its types
        case("interact-f32-1m", "interact", 101, 101, 101, 3.0),
        case("interact-f64-1m", "interact", 101, 101, 101, 3.0, dtype="f64"),
        # accelerations at probe points due to other bodies
        case("nbody-two-sets-500k", "nbody", 81, 80, 79, 3.0, probes=100000),
        # a periodic flow in a box, double precision
        case("periodic-f64-110k", "periodic", 48, 48, 48, 2.4, dtype="f64"),
        # an unbounded domain
        case("hash-1m", "count", 100, 100, 100, 2.4, cells="hash"),
        # lists of an undeformed solid: every row has ties at the search radius
        case("csr-2m", "csr", 128, 128, 128, 3.0, jitter=0.0),
        # the reference's published solid benchmark
        case("tlsph-1m", "tlsph", 101, 101, 101, 3.0, jitter=0.07),
        # many small clouds of uneven size
        case("batch-64", "batch", 10, 0, 0, 2.4, clouds=64, largest=40),
    ]


def draw(rng):
    """Another case of the listed ranges: clouds of about 1000 to 2 million points."""
    kind = rng.choice(["count", "count", "count", "wcsph", "wcsph", "grad", "interact", "interact", "nbody", "periodic",
                       "csr", "tlsph", "batch"])
    dtype = rng.choice(["f32", "f32", "f64"])
    cells = "hash" if kind in ("count", "wcsph") and rng.random() < 0.3 else "grid"
    two_d = rng.random() < 0.25 and kind not in ("batch",)
    most = {"grad": 1.0e6, "csr": 1.0e6, "tlsph": 5.0e5, "periodic": 5.0e5}.get(kind, 1.0e6)
    n = math.exp(rng.uniform(math.log(1000.0), math.log(most)))
    side = n ** (1 / 2 if two_d else 1 / 3)
    sides = [max(10, round(side * rng.uniform(0.8, 1.25))) for _ in range(3)]
    c = dict(kind=kind, nx=sides[0], ny=sides[1], nz=0 if two_d else sides[2], factor=round(rng.uniform(2.0, 3.2), 3),
             dtype=dtype, cells=cells)
    if kind == "nbody":
        c["probes"] = round(math.exp(rng.uniform(math.log(500.0), math.log(2.0e5))))
    if kind in ("csr", "tlsph"):
        c["jitter"] = round(rng.uniform(0.0, 0.1), 3)
    if kind == "batch":
        c.update(nx=8, ny=0, nz=0, clouds=rng.randint(5, 64), largest=rng.randint(12, 40))
    return c


# --------------------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------------------
class State:
    pass


def _types(case):
    return (np.float64, torch.float64) if case["dtype"] == "f64" else (np.float32, torch.float32)


def _sides(case):
    return [s for s in (case["nx"], case["ny"], case["nz"]) if s > 0]


def _lattice(sides, jitter, gen, normal=False):
    """(N, D) Float64 jittered lattice on the GPU, lattice units, x fastest, first point at 1."""
    axes = [torch.arange(s, dtype=torch.float64, device="cuda") for s in reversed(sides)]
    pts = torch.stack([g.reshape(-1) for g in reversed(torch.meshgrid(*axes, indexing="ij"))], dim=1) + 1.0
    if jitter:
        if normal:
            pts += jitter * torch.randn(pts.shape, generator=gen, dtype=torch.float64, device="cuda").clamp(-4, 4)
        else:
            pts += jitter * (2.0 * torch.rand(pts.shape, generator=gen, dtype=torch.float64, device="cuda") - 1.0)
    return pts


def _cell_sorted(pts, factor):
    """The order of the reference's benchmark clouds: by cells, first dimension slowest."""
    key = torch.zeros(len(pts), dtype=torch.int64, device=pts.device)
    for d in range(pts.shape[1]):
        key = key * 4096 + (pts[:, d] / factor).floor().to(torch.int64)
    return pts[torch.argsort(key, stable=True)]


def _grid(case, lo, hi, r, n, periodic_box=None):
    nd = len(lo)
    if case["cells"] == "hash":
        cl = pn.SpatialHashingCellList[nd](list_size=2 * n)
    else:
        cl = pn.FullGridCellList(min_corner=lo, max_corner=hi, search_radius=r)
    return pn.GridNeighborhoodSearch[nd](search_radius=r, n_points=n, cell_list=cl, periodic_box=periodic_box)


def _batch_sides(case, seed):
    """Sides of the cubic clouds of a batch: sizes log-uniform, the largest among them."""
    rng = np.random.default_rng([seed, 5])
    lo, hi = 3 * math.log(case["nx"]), 3 * math.log(case["largest"])
    return [case["largest"]] + [max(2, int(round(math.exp(v / 3)))) for v in rng.uniform(lo, hi, case["clouds"] - 1)]


def prepare(case, seed):
    dt, tdt = _types(case)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    s = State()
    s.case, s.kind = case, case["kind"]
    if s.kind == "batch":
        r = dt(case["factor"])
        pts, cls, sizes = [], [], []
        for c in _batch_sides(case, 1):
            p = _lattice([c] * 3, 0.25, gen).to(tdt)
            corner = np.full(3, 0.5, dtype=dt), np.full(3, c + 0.5, dtype=dt)
            cls.append(pn.FullGridCellList(min_corner=corner[0], max_corner=corner[1], search_radius=r))
            pts.append(p)
            sizes.append(len(p))
        s.x = torch.cat(pts).contiguous().t()
        s.nhs = pn_batch.BatchedGridNeighborhoodSearch(3, search_radius=r, cell_lists=cls, n_points=sizes)
        s.counts = torch.zeros(s.x.shape[1], dtype=torch.int32, device="cuda")
        s.nhs.update(s.x)
        return s

    sides, factor = _sides(case), case["factor"]
    nd = len(sides)
    spacing = 0.01 if s.kind in ("count", "wcsph", "periodic") else 1.0
    if s.kind in ("interact", "nbody"):
        spacing = 1.0 / (max(sides) + 1)
    normal = s.kind in ("interact", "nbody", "tlsph")
    jitter = case.get("jitter", 0.07 if normal else 0.1)
    pts = _lattice(sides, jitter, gen, normal)
    if normal:
        pts = _cell_sorted(pts, factor)
    if s.kind == "periodic":
        pts = pts - 0.5  # the lattice tiles the box
    x = (pts * spacing).to(tdt).contiguous()
    n = len(x)
    r = dt(factor * spacing)
    s.h = float(r) / 2
    s.r, s.spacing, s.n = r, spacing, n
    s.x = x.t()
    lo = np.full(nd, 0.5 * spacing, dtype=dt)
    hi = (np.array(sides, dtype=dt) + dt(0.5)) * dt(spacing)

    def rand(*shape):
        return torch.rand(shape, generator=gen, dtype=tdt, device="cuda")

    def vectors(rows):
        return torch.zeros((n, rows), dtype=tdt, device="cuda").t()

    if s.kind == "periodic":
        box = pn.PeriodicBox(min_corner=np.zeros(nd, dtype=dt), max_corner=np.array(sides, dtype=dt) * dt(spacing))
        s.nhs = _grid(case, box.min_corner, box.max_corner, r, n, box)
        s.box = [float(v) for v in box.size]
        s.counts = torch.zeros(n, dtype=torch.int32, device="cuda")
        s.rho = torch.zeros(n, dtype=tdt, device="cuda")
        s.mass = (0.95 + 0.1 * rand(n)) * (RHO0 * spacing**nd)
        s.f_count = pn.CountNeighbors(s.counts, accumulate=False)
        s.f_rho = sph.SPHDensity(s.rho, s.mass, s.h, accumulate=False)
    elif s.kind == "csr":
        inner = _grid(dict(case, cells="grid"), lo - dt(1), hi + dt(1), r, n)
        s.nhs = pn.PrecomputedNeighborhoodSearch[nd](search_radius=r, n_points=n, update_neighborhood_search=inner)
        s.rho = torch.zeros(n, dtype=tdt, device="cuda")
        s.mass = 0.95 + 0.1 * rand(n)
        s.f_rho = sph.SPHDensity(s.rho, s.mass, s.h, "wendland_c2", accumulate=False)
        return s
    elif s.kind == "tlsph":
        pre = pn.PrecomputedNeighborhoodSearch[nd](search_radius=r, n_points=n)
        pn.initialize(pre, s.x, s.x)
        s.nhs = pn.freeze_neighborhood_search(pre)
        s.mass = torch.full((n,), 0.1, dtype=tdt, device="cuda")
        s.rho = torch.full((n,), RHO0, dtype=tdt, device="cuda")
        s.volume = s.mass / s.rho
        s.L = sph.tlsph_correction_matrix(s.nhs, s.x, s.volume, s.h)
        # a smooth deformation, another one for each seed
        phase = 6.0 * torch.rand(nd, generator=gen, dtype=torch.float64, device="cuda")
        x64 = s.x.t().double()
        s.now = (1.01 * x64 + 0.02 * torch.sin(0.3 * x64 + phase)).to(tdt).contiguous().t()
        return s
    elif s.kind == "nbody":
        s.nhs = _grid(case, np.zeros(nd, dtype=dt), hi + dt(spacing), r, n)
        m = case["probes"]
        u = torch.rand((m, nd), generator=gen, dtype=torch.float64, device="cuda")
        span = torch.tensor([float(v) for v in sides], dtype=torch.float64, device="cuda") * spacing
        s.probes = _cell_sorted(u * span + 0.5 * spacing, float(r)).to(tdt).contiguous().t()
        s.mass = 1e10 * (1 + rand(n))
        s.dv = torch.zeros((m, nd), dtype=tdt, device="cuda").t()
        s.f = pn.NBodyAcceleration(s.dv, s.mass, accumulate=False)
    else:
        s.nhs = _grid(case, lo - 2 * r, hi + 2 * r, r, n)
        if s.kind == "count":
            s.counts = torch.zeros(n, dtype=torch.int32, device="cuda")
            s.f = pn.CountNeighbors(s.counts, accumulate=False)
        elif s.kind in ("wcsph", "grad"):
            s.mass = (0.95 + 0.1 * rand(n)) * (RHO0 * spacing**nd)
            s.rho = torch.zeros(n, dtype=tdt, device="cuda")
            s.P = torch.zeros(n, dtype=tdt, device="cuda")
            s.dv = vectors(nd)
            s.f_rho = sph.SPHDensity(s.rho, s.mass, s.h, accumulate=False)
            s.f_dv = sph.SPHPressureAcceleration(s.dv, s.mass, s.P, s.h, accumulate=False)
        else:
            s.density = 1000 + rand(n)
            s.mass = torch.full((n,), float(dt(0.1) * dt(spacing)), dtype=tdt, device="cuda")
            v = torch.empty((n, nd + 1), dtype=tdt, device="cuda")
            v[:, :nd] = 0.2 * (rand(n, nd) - 0.5)
            v[:, nd] = s.density
            s.v = v.t()
            s.p = pn.state_equation_cole(s.density, 1000.0, SOUND, 1.0)
            s.dv = vectors(nd + 1)
            s.f = pn.WCSPHInteraction(s.dv, s.v, s.p, s.mass, s.h, SOUND, accumulate=False)
    pn.initialize(s.nhs, s.x, s.x)
    return s


# --------------------------------------------------------------------------------------
# One pass
# --------------------------------------------------------------------------------------
def run(s):
    x, nhs, kind = s.x, s.nhs, s.kind
    if kind == "batch":
        nhs.update(x)
        nhs.count_neighbors(s.counts)
        return {"counts": s.counts}
    if kind == "csr":
        pn.initialize(nhs, x, x)
        pn.foreach_point_neighbor(s.f_rho, x, x, nhs)
        return {"row_ptr": nhs.neighbor_lists.row_ptr, "col_idx": nhs.neighbor_lists.col_idx, "rho": s.rho}
    if kind == "tlsph":
        F = sph.tlsph_deformation_gradient(nhs, x, s.now, s.volume, s.h, correction=s.L)
        P = sph.tlsph_pk1_corrected(F, s.rho, YOUNG, POISSON, correction=s.L)
        dv = sph.tlsph_interaction(nhs, x, s.now, s.mass, s.rho, P, s.h, F=F, young_modulus=YOUNG,
                                   penalty_alpha=PENALTY)
        return {"F": F, "P": P, "dv": dv}
    pn.update(nhs, x, x)
    if kind == "count":
        pn.foreach_point_neighbor(s.f, x, x, nhs)
        return {"counts": s.counts}
    if kind == "periodic":
        pn.foreach_point_neighbor(s.f_count, x, x, nhs)
        pn.foreach_point_neighbor(s.f_rho, x, x, nhs)
        return {"counts": s.counts, "rho": s.rho}
    if kind == "nbody":
        pn.foreach_point_neighbor(s.f, s.probes, x, nhs)
        return {"dv": s.dv}
    if kind == "interact":
        pn.foreach_point_neighbor(s.f, x, x, nhs)
        return {"dv": s.dv}
    if kind == "wcsph":
        pn.foreach_point_neighbor(s.f_rho, x, x, nhs)
        sph.tait_pressure_term(s.rho, RHO0, SOUND, GAMMA, out=s.P)
        pn.foreach_point_neighbor(s.f_dv, x, x, nhs)
        return {"rho": s.rho, "dv": s.dv}
    xg = x.detach().requires_grad_(True)
    rho = sph.sph_density(xg, s.mass, nhs, s.h)
    p = EOS_B * ((rho / RHO0) ** GAMMA - 1.0)
    a = sph.sph_pressure_acceleration(xg, s.mass, p / (rho * rho), nhs, s.h)
    (g,) = torch.autograd.grad((a * a).sum(), xg)
    return {"rho": rho.detach(), "a": a.detach(), "grad": g}


# --------------------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------------------
def work(case):
    size = 8 if case["dtype"] == "f64" else 4
    kind = case["kind"]
    if kind == "batch":
        n, nd = sum(c**3 for c in _batch_sides(case, 1)), 3
    else:
        n, nd = int(np.prod(_sides(case))), len(_sides(case))
    per = math.pi * case["factor"] ** 2 if nd == 2 else 4 / 3 * math.pi * case["factor"] ** 3
    pairs = n * per
    test = 3 * nd  # operations of a pair's squared distance and its comparison
    # values read and written per point, operations per pair
    if kind in ("count", "batch"):
        return {"bytes": n * (nd * size + 4), "flops": pairs * test}
    if kind == "periodic":
        return {"bytes": n * (nd * size + 4 + 2 * size), "flops": pairs * (2 * test + 12)}
    if kind == "wcsph":
        return {"bytes": n * size * (nd + 1 + 1 + nd), "flops": pairs * (2 * test + 12 + 14 + 2 * nd)}
    if kind == "grad":
        return {"bytes": n * size * (3 * nd + 2), "flops": pairs * (4 * test + 2 * (12 + 14 + 2 * nd) + 60)}
    if kind == "interact":
        return {"bytes": n * size * (3 * nd + 4), "flops": pairs * (test + 40)}
    if kind == "nbody":
        m = case["probes"]
        return {"bytes": size * (n * (nd + 1) + 2 * m * nd), "flops": m * per * (test + 8 + 2 * nd)}
    if kind == "csr":
        return {"bytes": 4 * (n + pairs) + n * size * (nd + 2), "flops": pairs * (test + 12)}
    mats = nd * nd
    return {"bytes": 4 * (n + pairs) + n * size * (2 * nd + 2 + 3 * mats + nd),
            "flops": pairs * (2 * test + 10 + 3 * mats + 10 + 6 * mats + 20)}


# --------------------------------------------------------------------------------------
# 64-bit results (neighbour sets by the stated predicate in the case's type, sums in Float64)
# --------------------------------------------------------------------------------------
def _for_pairs(x, y, r, fn, most=4_000_000):
    """fn(slice of x, j, pos_diff in Float64, d^2 in Float64, neighbour mask), one stencil row of
    cells at a time; pos_diff and d^2 of the predicate are evaluated in the type of x and y."""
    nd, dev = x.shape[1], x.device
    size = float(r) * 1.001
    lo = torch.minimum(x.amin(0), y.amin(0)).double() - size
    cx, cy = (((p.double() - lo) / size).floor().to(torch.int64) for p in (x, y))
    dims = torch.maximum(cx.amax(0), cy.amax(0)) + 2
    strides = [1]
    for d in range(1, nd):
        strides.append(strides[-1] * int(dims[d - 1]))
    st = torch.tensor(strides, device=dev)
    kx, ky = (cx * st).sum(1), (cy * st).sum(1)
    order = torch.argsort(ky)
    sky = ky[order]
    r2 = torch.tensor(r * r, dtype=x.dtype, device=dev)
    rows = [dy * strides[1] + (dz * strides[2] if nd == 3 else 0) for dz in ((-1, 0, 1) if nd == 3 else (0,))
            for dy in (-1, 0, 1)]
    ends = [(torch.searchsorted(sky, kx + o - 1), torch.searchsorted(sky, kx + o + 1, right=True)) for o in rows]
    width = max(1, max(int((e - b).max()) for b, e in ends))
    chunk = max(1, most // width)
    for q0 in range(0, len(x), chunk):
        q = slice(q0, min(len(x), q0 + chunk))
        for b, e in ends:
            k = b[q, None] + torch.arange(width, device=dev)
            inside = k < e[q, None]
            j = order[k.clamp(max=len(y) - 1)]
            pd = x[q, None, :] - y[j]
            d2 = pd[..., 0] * pd[..., 0]
            for d in range(1, nd):
                d2 = d2 + pd[..., d] * pd[..., d]
            near = inside & (d2 <= r2)
            pd64 = x[q, None, :].double() - y[j].double()
            fn(q, j, pd64, (pd64 * pd64).sum(-1), near)


def _cubic(nd, h):
    s = 1 / (math.pi * h**3) if nd == 3 else 10 / (7 * math.pi * h * h)
    w = lambda r: 0.25 * s * ((2 - r / h).clamp(min=0) ** 3 - 4 * (1 - r / h).clamp(min=0) ** 3)  # noqa: E731
    dw = lambda r: s / h * (3 * (1 - r / h).clamp(min=0) ** 2 - 0.75 * (2 - r / h).clamp(min=0) ** 2)  # noqa: E731
    d2w = lambda r: s / h**2 * (1.5 * (2 - r / h).clamp(min=0) - 6 * (1 - r / h).clamp(min=0))  # noqa: E731
    return w, dw, d2w


def _wendland(nd, h):
    s = 21 / (16 * math.pi * h**3) if nd == 3 else 7 / (4 * math.pi * h * h)
    w = lambda r: s * (1 - 0.5 * r / h).clamp(min=0) ** 4 * (2 * r / h + 1)  # noqa: E731
    dw = lambda r: s / h * -5 * (r / h) * (1 - 0.5 * r / h).clamp(min=0) ** 3  # noqa: E731
    return w, dw


def _density64(x, y, r, mass, w):
    rho = torch.zeros(len(x), dtype=torch.float64, device=x.device)

    def add(q, j, pd, d2, near):
        rho[q] += torch.where(near, mass[j] * w(d2.sqrt()), 0.0).sum(1)

    _for_pairs(x, y, r, add)
    return rho


def exact(case, seed):
    kind = case["kind"]
    if kind in ("count", "batch"):
        return None  # whole numbers only
    s = prepare(case, seed)
    x = s.x.t()
    nd = x.shape[1]
    zeros = lambda *shape: torch.zeros(shape, dtype=torch.float64, device="cuda")  # noqa: E731
    if kind == "nbody":
        p, m, dv = s.probes.t(), s.mass.double(), zeros(case["probes"], nd)
        tiny = math.sqrt(torch.finfo(x.dtype).eps)

        def add(q, j, pd, d2, near):
            c = torch.where(near & (d2 >= tiny * tiny), -6.6743e-11 * m[j] * d2.clamp(min=1e-300) ** -1.5, 0.0)
            dv[q] += (c[..., None] * pd).sum(1)

        _for_pairs(p, x, s.r, add)
        return {"dv": dv.t()}
    mass = s.mass.double()
    if kind == "periodic":
        w, _, _ = _cubic(nd, s.h)
        # the images that touch the box; the kernel vanishes at the search radius, so a pair that
        # rounding moves across it changes nothing
        y, m = x.double(), mass
        for d in range(nd):
            lo, hi = y[:, d] < 1.01 * float(s.r), y[:, d] > s.box[d] - 1.01 * float(s.r)
            shift = torch.zeros(nd, dtype=torch.float64, device="cuda")
            shift[d] = s.box[d]
            y, m = torch.cat([y, y[lo] + shift, y[hi] - shift]), torch.cat([m, m[lo], m[hi]])
        return {"counts": None, "rho": _density64(x.double(), y, float(s.r), m, w)}
    if kind == "csr":
        return {"row_ptr": None, "col_idx": None, "rho": _density64(x, x, s.r, mass, _wendland(nd, s.h)[0])}
    if kind in ("wcsph", "grad"):
        w, dw, d2w = _cubic(nd, s.h)
        rho = _density64(x, x, s.r, mass, w)
        P = EOS_B * ((rho / RHO0) ** GAMMA - 1) / rho**2
        a = zeros(len(x), nd)

        def press(q, j, pd, d2, near):
            d = d2.sqrt()
            c = torch.where(near & (d2 > 0), -mass[j] * (P[q, None] + P[j]) * dw(d) / d.clamp(min=1e-300), 0.0)
            a[q] += (c[..., None] * pd).sum(1)

        _for_pairs(x, x, s.r, press)
        if kind == "wcsph":
            return {"rho": rho, "dv": a.t()}
        ab, g, Pb = 2 * a, zeros(len(x), nd), zeros(len(x))

        def press_adj(q, j, pd, d2, near):
            d = d2.sqrt().clamp(min=1e-300)
            v = pd / d[..., None]
            u = mass[j][..., None] * ab[q, None] - mass[q, None, None] * ab[j]
            on = near & (d2 > 0)
            w1, w2 = torch.where(on, dw(d), 0.0), torch.where(on, d2w(d), 0.0)
            vu = (v * u).sum(-1)
            Pb[q] -= (w1 * vu).sum(1)
            c = P[q, None] + P[j]
            t = (w2 * vu)[..., None] * v + (w1 / d)[..., None] * (u - vu[..., None] * v)
            g[q] -= torch.where(on[..., None], c[..., None] * t, 0.0).sum(1)

        _for_pairs(x, x, s.r, press_adj, 2_000_000)
        q7 = (rho / RHO0) ** GAMMA
        rb = Pb * EOS_B * (GAMMA * q7 / rho**3 - 2 * (q7 - 1) / rho**3)

        def dens_adj(q, j, pd, d2, near):
            d = d2.sqrt().clamp(min=1e-300)
            c = torch.where(near & (d2 > 0), (rb[q, None] * mass[j] + rb[j] * mass[q, None]) * dw(d) / d, 0.0)
            g[q] += (c[..., None] * pd).sum(1)

        _for_pairs(x, x, s.r, dens_adj)
        return {"rho": rho, "a": a.t(), "grad": g.t()}
    if kind == "interact":
        _, dw = _wendland(nd, s.h)
        v, rho, p = s.v.t()[:, :nd].double(), s.v.t()[:, nd].double(), s.p.double()
        dv, tiny, h = zeros(len(x), nd + 1), math.sqrt(torch.finfo(x.dtype).eps), s.h

        def add(q, j, pd, d2, near):
            d = d2.sqrt()
            on = near & (d >= tiny)
            gw = torch.where(on, dw(d) / d.clamp(min=1e-300), 0.0)
            ra, rb, mb = rho[q, None], rho[j], mass[j]
            vr = ((v[q, None] - v[j]) * pd).sum(-1)
            c = -mb * (p[q, None] + p[j]) / (ra * rb)
            mu = h * vr / (d2 + 0.01 * h * h)
            c = c - torch.where(vr < 0, mb * (-0.02 * SOUND * mu) / ((ra + rb) / 2), 0.0)
            dv[q, :nd] += ((c * gw)[..., None] * pd).sum(1)
            dv[q, nd] += ((ra / rb * mb * vr + 0.1 * h * SOUND * mb / rb * 2 * (ra - rb)) * gw).sum(1)

        _for_pairs(x, x, s.r, add)
        return {"dv": dv.t()}
    # total-Lagrangian solid
    w, dw = _wendland(nd, s.h)
    X, now, L, vol, rho = x.double(), s.now.t().double(), s.L.double(), s.volume.double(), s.rho.double()
    G, dv = zeros(len(x), nd, nd), zeros(len(x), nd)

    def grad(q, j, pd, d2, near):
        d = d2.sqrt()
        c = torch.where(near & (d2 > 0), vol[j] * dw(d) / d.clamp(min=1e-300), 0.0)
        dx = now[j] - now[q, None]
        for a in range(nd):
            G[q, a] += ((c * dx[..., a])[..., None] * pd).sum(1)

    _for_pairs(x, x, s.r, grad)
    F = torch.bmm(G, L.contiguous())
    lam, mu = YOUNG * POISSON / ((1 + POISSON) * (1 - 2 * POISSON)), YOUNG / (2 * (1 + POISSON))
    eye = torch.eye(nd, dtype=torch.float64, device="cuda")
    E = 0.5 * (torch.bmm(F.transpose(1, 2).contiguous(), F) - eye)
    S = lam * E.diagonal(dim1=1, dim2=2).sum(1)[:, None, None] * eye + 2 * mu * E
    P = torch.bmm(torch.bmm(F, S), L.contiguous()) / (rho * rho)[:, None, None]

    def force(q, j, pd, d2, near):
        d = d2.sqrt()
        on = near & (d2 > 0)
        c = torch.where(on, mass[j] * dw(d) / d.clamp(min=1e-300), 0.0)
        xab = now[q, None] - now[j]
        n2 = (xab * xab).sum(-1).clamp(min=1e-300)
        delta = torch.zeros_like(d)
        for a in range(nd):
            dv[q, a] += (c * ((P[q, None, a] + P[j][..., a, :]) * pd).sum(-1)).sum(1)
            delta += (((F[q, None, a] + F[j][..., a, :]) * pd).sum(-1) - 2 * xab[..., a]) * xab[..., a]
        f = 0.5 * PENALTY * YOUNG / rho[q, None] * vol[j] * w(d) / d2.clamp(min=1e-300) * delta / n2
        dv[q] += (torch.where(on, f, 0.0)[..., None] * xab).sum(1)

    _for_pairs(x, x, s.r, force, 1_500_000)
    return {"F": F, "P": P, "dv": dv.t()}
