"""Runs that cover 32 cells: there the split coordinates of the estimate are largest and its error
bound widest.  Points one to a cell along x, each with partners placed around it at r times
1 + k u for a few small k, so that almost every pair near a query lies within the margin of the
search radius or next to it; sets equal the oracle's."""

import numpy as np
import pytest

import pointneighbors as pn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("radius", [1.0, 1.999, 0.0137])  # at both ends of the scaled range and between
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("D", [1, 2, 3])
def test_pairs_at_the_radius(orc, D, dtype, radius):
    from test_gpu_parity import dev, gpu_counts, gpu_sums, make_nhs, oracle_like
    rng = np.random.default_rng(D)
    rows, per = 1 if D == 1 else 11, 4  # 2D and 3D: enough points for the run kernels of pair sums
    n = 640 * rows
    x = np.zeros((n, D))
    x[:, 0] = np.tile(np.arange(640), rows) + rng.uniform(0.0, 0.5, n)
    x[:, 1:] = rng.uniform(0.0, 0.9, (n, D - 1))
    if D > 1:
        x[:, 1] += 8.0 * np.repeat(np.arange(rows), 640)
    u = rng.standard_normal((n, per, D))
    u /= np.linalg.norm(u, axis=2)[..., None]
    # from the type's own rounding to beyond the margin (2^-18 of up to 70^2, relative to r^2)
    off = rng.choice([0.0, 1e-7, -1e-7, 1e-6, -1e-6, 1e-5, -1e-5, 1e-4, -1e-4, 1e-3, -1e-3, 1e-2, -1e-2], (n, per, 1))
    partners = x[:, None, :] + u * (1.0 + off)
    pts = (radius * np.concatenate([x, partners.reshape(-1, D)])).astype(dtype)
    pts = pts[rng.permutation(len(pts))]
    r = dtype(radius)
    nhs = make_nhs(pts, r, pts.min(axis=0) - 3 * r, pts.max(axis=0) + 3 * r, cap=1000)
    y = dev(pts)
    pn.initialize(nhs, y, y)
    og = oracle_like(orc, nhs, dtype)
    assert og.build(pts)[0] == orc.OK
    _, _, cnt, total, _ = og.traverse(pts, pts)
    assert np.array_equal(gpu_counts(nhs, y, y), cnt) and nhs.last_traversal() == "runs"
    assert np.array_equal(gpu_sums(nhs, y, y), total) and nhs.last_traversal() == "runs"
    # the centres alone as queries of the same rows: runs of one point a cell
    q = dev((radius * x).astype(dtype))
    _, _, cnt, total, _ = og.traverse((radius * x).astype(dtype), pts)
    assert np.array_equal(gpu_counts(nhs, q, y), cnt) and nhs.last_traversal() == "runs"
    assert np.array_equal(gpu_sums(nhs, q, y), total)
