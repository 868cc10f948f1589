"""Traversals of a periodic grid's own points after their coordinates moved without a new binning
(pn_grid_refresh, then PN_QUERIES_GRID).  With three cells a dimension every pair of cells is
adjacent, so the neighbours are all pairs whose distance to the nearest image, in the arithmetic of
compute_periodic_distance (src/neighborhood_search.jl:428-436), is at most r."""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors._lib import PN_QUERIES_GRID, check, load

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def neighbors(pts, size, r):
    """(counts, sums of neighbour indices), every operation rounded to the points' type."""
    pd = pts[:, None, :] - pts[None, :, :]

    def squared(p):
        s = p[..., 0] * p[..., 0]
        for d in range(1, p.shape[-1]):
            s = s + p[..., d] * p[..., d]
        return s

    d2 = squared(pd)
    image = pd - size * np.rint(pd / size)
    near = np.where(d2 > r * r, squared(image), d2) <= r * r
    return near.sum(1), (near * np.arange(len(pts))).sum(1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("D,n", [(1, 60), (2, 200), (3, 700)])
@pytest.mark.parametrize("move", [0.0, 0.0099, 0.2, 1.4])
def test_moved_points_in_three_cells(D, n, dtype, move):
    from test_gpu_parity import dev
    rng = np.random.default_rng(n)
    r, size = dtype(1.0), np.full(D, 3.0, dtype=dtype)
    pts = rng.uniform(0.0, 3.0, (n, D))
    # pairs whose images are just within r on the far side of the box once the first has moved
    pts[0::7, 0] = 0.998
    pts[1::7, 0] = 2.005
    pts[1::7, 1:] = pts[0::7, 1:][: len(pts[1::7])]
    moved = pts + move * rng.uniform(-1.0, 1.0, pts.shape)
    moved[0::7, 0] = pts[0::7, 0] + 0.9 * move
    moved[0::7, 1:], moved[1::7] = pts[0::7, 1:], pts[1::7]
    pts, moved = pts.astype(dtype), moved.astype(dtype)
    box = pn.PeriodicBox(min_corner=np.zeros(D, dtype=dtype), max_corner=size)
    cl = pn.FullGridCellList(min_corner=box.min_corner, max_corner=box.max_corner, search_radius=r)
    nhs = pn.GridNeighborhoodSearch[D](search_radius=r, n_points=n, periodic_box=box, cell_list=cl)
    assert list(nhs.n_cells) == [3] * D
    x, y = dev(pts), dev(moved)
    pn.initialize(nhs, x, x)
    check(load().pn_grid_refresh(nhs._handle, ctypes.c_void_p(y.data_ptr()), n))
    counts = torch.zeros(n, dtype=torch.int32, device="cuda")
    sums = torch.zeros(n, dtype=torch.int64, device="cuda")
    check(load().pn_count_neighbors(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(counts.data_ptr()), 0))
    check(load().pn_sum_neighbor_indices(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(sums.data_ptr()), 0, 0))
    want_counts, want_sums = neighbors(moved, size, r)
    assert np.array_equal(counts.cpu().numpy(), want_counts)
    assert np.array_equal(sums.cpu().numpy(), want_sums)
