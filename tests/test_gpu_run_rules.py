"""Traversals at the sizes where the choice of the kernel or of its split changes: the cell kernel
for sparse queries and for small 2D clouds, two wavefronts a window up to 576 windows, rows of few
points far apart.  Counts equal those of the cell kernel ("algorithm" 1); density sums agree within
the reordering bound: n non-negative terms in another order differ by at most n u times their sum,
and a term by a few u."""

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors import sph

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def compare(pts, r, queries=None):
    from test_gpu_parity import dev, make_nhs
    dtype = pts.dtype.type
    r = dtype(r)
    nhs = make_nhs(pts, r, pts.min(axis=0) - 3 * r, pts.max(axis=0) + 3 * r, cap=1000)
    y = dev(pts)
    x = y if queries is None else dev(queries)
    pn.initialize(nhs, x, y)
    mass = 0.5 + torch.rand(len(pts), dtype=y.dtype, device="cuda")
    out = []
    for algorithm in (0, 1):
        nhs.set_tuning("algorithm", algorithm)
        cnt = torch.zeros(x.shape[1], dtype=torch.int32, device="cuda")
        rho = torch.zeros(x.shape[1], dtype=y.dtype, device="cuda")
        pn.foreach_point_neighbor(pn.CountNeighbors(cnt), x, y, nhs)
        pn.foreach_point_neighbor(sph.SPHDensity(rho, mass, float(r) / 2), x, y, nhs)
        out.append((cnt, rho))
    assert torch.equal(out[0][0], out[1][0])
    bound = (out[1][0].double() + 16) * np.finfo(dtype).eps * out[1][1].double()
    assert ((out[0][1] - out[1][1]).abs().double() <= bound).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("D,n", [(2, 32767), (2, 32768), (3, 4608), (3, 4609), (3, 9217), (2, 3), (3, 1)])
def test_clouds(D, n, dtype):
    pts = np.random.default_rng(n).uniform(0.0, n ** (1 / D), (n, D)).astype(dtype)
    compare(pts, 2.1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("n_x", [1, 499, 500, 501, 4000])
def test_sparse_queries(D, n_x, dtype):
    rng = np.random.default_rng(n_x)
    side = 4000 ** (1 / D)
    pts = rng.uniform(0.0, side, (4000, D)).astype(dtype)
    compare(pts, 2.3, rng.uniform(0.0, side, (n_x, D)).astype(dtype))


@pytest.mark.parametrize("D", [2, 3])
@pytest.mark.parametrize("gap", [3.0, 11.0, 12.0, 13.0, 40.0])
def test_thin_rows(D, gap):
    """Points `gap` cells apart in x, two to a place: every row is thin."""
    x = np.repeat(np.arange(120) * gap, 2) + np.tile([0.2, 0.7], 120)
    rows = np.stack([np.concatenate([x, x + 0.4])] + [np.repeat([0.5, 1.3], 240)] * (D - 1), axis=1)
    pts = np.concatenate([rows, rows + np.eye(D)[1] * 0.9]).astype(np.float32)
    if D == 2:  # enough points for the run kernel
        pts = np.concatenate([pts + np.float32([0.0, 5.0 * k]) for k in range(69)])
    compare(pts, 1.0)
