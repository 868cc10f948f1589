"""The run kernels (csrc/pn_runs.h): the matrix-core prefilter's error bound, and traversals at
the sizes where runs, tiles, parts and gaps begin and end, against the oracle."""

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors import sph, synthetic

EPS = 2.0**-18  # PREFILTER_EPS


def split(v):
    v = np.asarray(v, dtype=np.float32)
    h = v.astype(np.float16)
    return h.astype(np.float64), (v - h.astype(np.float32)).astype(np.float16).astype(np.float64)


@pytest.mark.parametrize("extent", [1.6, 4.0, 34.0])
def test_prefilter_error_bound(extent):
    """The 16 products of the estimate, summed exactly, are within PREFILTER_EPS / 2 of the squared
    distance minus r^2 (the other half is left to the additions' rounding: 16 of at most 2^-23 of
    the terms' sum, which (2 |q| + r)^2 + r^2 bounds near the search radius)."""
    rng = np.random.default_rng(int(extent * 10))
    n = 200000
    r = rng.uniform(1.0, 2.0, n).astype(np.float32)
    q = (rng.uniform(-1, 1, (n, 3)) * [extent, 1.1, 1.1]).astype(np.float32)
    u = rng.standard_normal((n, 3))
    u /= np.linalg.norm(u, axis=1)[:, None]
    c = (q + u * (r * rng.uniform(0.9, 1.1, n))[:, None]).astype(np.float32)
    want = ((q.astype(np.float64) - c) ** 2).sum(1) - r.astype(np.float64) ** 2
    nc = (c * c).sum(1, dtype=np.float32)
    m = (q * q).sum(1, dtype=np.float32) - r * r
    got = np.zeros(n)
    for d in range(3):
        ch, cl = split(np.float32(16) * c[:, d])
        qh, ql = split(np.float32(-32) * q[:, d])
        got += ch * qh + cl * qh + ch * ql + (cl * ql if d == 2 else 0)
    (nh, nl), (mh, ml) = split(nc), split(m)
    got += 256 * (nh + nl) + 256 * (mh + ml)
    bound = EPS * ((2 * np.linalg.norm(q.astype(np.float64), axis=1) + r) ** 2 + r.astype(np.float64) ** 2)
    assert (np.abs(got / 256 - want) <= 0.5 * bound).all()


torch = pytest.importorskip("torch")


def clouds(D):
    rng = np.random.default_rng(D)
    side = {1: 700, 2: 40, 3: 13}[D]
    lattice = synthetic.jittered_lattice((side,) * D, 1.0, 0.0, dtype=np.float64)
    yield "ties", lattice, 2.0
    yield "ties-shifted", lattice * 0.1 + 0.37, 0.3
    for n in (1, 7, 8, 9, 31, 32, 33, 63, 65, 1500):
        yield f"uniform-{n}", rng.uniform(0, 12, (n, D)), 1.7
    dense = rng.normal(3.0, 0.2, (700, D))  # more candidates than a part, more queries than a run
    yield "dense-and-sparse", np.concatenate([dense, rng.uniform(-40, 40, (300, D))]), 1.0
    yield "far-from-origin", rng.uniform(0, 5, (900, D)) * 2.0**-6 + 1000.0, 1.1 * 2.0**-6
    yield "huge-radius", rng.uniform(0, 9, (600, D)) * 2.0**60, 1.3 * 2.0**60  # the general path


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("D", [1, 2, 3])
def test_runs_equal_oracle(orc, D, dtype):
    from test_gpu_parity import dev, gpu_counts, gpu_sums, make_nhs, oracle_like
    for name, pts, r in clouds(D):
        print(D, dtype.__name__, name, flush=True)
        pts, r = pts.astype(dtype), dtype(r)
        nhs = make_nhs(pts, r, pts.min(axis=0) - 3 * r, pts.max(axis=0) + 3 * r, cap=1000)
        x = dev(pts)
        pn.initialize(nhs, x, x)
        og = oracle_like(orc, nhs, dtype)
        assert og.build(pts)[0] == orc.OK
        _, _, cnt, total, _ = og.traverse(pts, pts)
        assert np.array_equal(gpu_counts(nhs, x, x), cnt), name
        assert np.array_equal(gpu_sums(nhs, x, x), total), name
        # queries of their own, some cells of the grid without any
        sub = np.arange(0, len(pts), 3)
        got = gpu_counts(nhs, x, x, points=sub)
        assert np.array_equal(got[sub], cnt[sub]), name
        # moved in place: the cells of the binning decide which candidates are looked at
        moved = (pts + dtype(0.4) * r * np.sin(7 * np.arange(pts.size)).reshape(pts.shape)).astype(dtype)
        x.copy_(torch.as_tensor(moved.T.copy(), device="cuda"))
        _, _, cnt, total, _ = og.traverse(moved, moved)
        assert np.array_equal(gpu_counts(nhs, x, x), cnt), name
        assert np.array_equal(gpu_sums(nhs, x, x), total), name


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("D", [2, 3])
def test_run_sums_equal_slices(D, dtype):
    """Density and pressure acceleration against the per-query-slice kernel (algorithm 1): sums of
    n terms in another order differ by at most n u times the sum of the terms' magnitudes, and a
    term by a few u."""
    from test_gpu_parity import dev, make_nhs
    u = np.finfo(dtype).eps
    for name, pts, r in clouds(D):
        if name == "huge-radius":
            continue
        pts, r = pts.astype(dtype), dtype(r)
        nhs = make_nhs(pts, r, pts.min(axis=0) - 3 * r, pts.max(axis=0) + 3 * r, cap=1000)
        x = dev(pts)
        n, h = len(pts), float(r) / 2
        pn.initialize(nhs, x, x)
        tdt = x.dtype
        mass = 0.5 + torch.rand(n, dtype=tdt, device="cuda")
        cnt = torch.zeros(n, dtype=torch.int32, device="cuda")
        pn.foreach_point_neighbor(pn.CountNeighbors(cnt), x, x, nhs)
        out = []
        for algorithm in (0, 1):
            nhs.set_tuning("algorithm", algorithm)
            rho = torch.zeros(n, dtype=tdt, device="cuda")
            dv = torch.zeros((n, D), dtype=tdt, device="cuda").t()
            pn.foreach_point_neighbor(sph.SPHDensity(rho, mass, h), x, x, nhs)
            pn.foreach_point_neighbor(sph.SPHPressureAcceleration(dv, mass, mass, h), x, x, nhs)
            out.append((rho, dv))
        terms = cnt.double() + 16
        assert ((out[0][0] - out[1][0]).abs().double() <= terms * u * out[1][0].double()).all(), name
        # |m_j (P_i + P_j) W'| <= 1.5 * 3 * W(0) / h: the cubic spline's steepest slope is -W(0) / h
        scale = 4.5 * sph_peak(D, h) / h * cnt.double()
        assert ((out[0][1] - out[1][1]).abs().double().amax(dim=0) <= terms * u * scale).all(), name


def sph_peak(D, h):
    """W(0) of the cubic spline."""
    return 1 / (np.pi * h**3) if D == 3 else 10 / (7 * np.pi * h * h)
