"""A captured traversal replayed over coordinates that moved without a new binning (pn_grid_refresh)
after the capture: cell membership stays that of the last update! (src/nhs_grid.jl:543-545), so a
pair within r is found only where the cells of its points as binned are adjacent."""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors._lib import PN_QUERIES_GRID, check, load

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def neighbors(pts, cells, r):
    """(counts, sums of neighbour indices) of the pairs in adjacent cells, every operation rounded."""
    pd = pts[:, None, :] - pts[None, :, :]
    d2 = pd[..., 0] * pd[..., 0]
    for d in range(1, pts.shape[1]):
        d2 = d2 + pd[..., d] * pd[..., d]
    near = (d2 <= r * r) & (np.abs(cells[:, None, :] - cells[None, :, :]).max(axis=-1) <= 1)
    return near.sum(1), (near * np.arange(len(pts))).sum(1)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("D,n", [(1, 40), (2, 400), (3, 1500)])
def test_moved_between_replays(D, n, dtype):
    from test_gpu_parity import dev, make_nhs
    rng = np.random.default_rng(n)
    side = (n / 4.0) ** (1 / D)
    pts = rng.uniform(0.0, side, (n, D)).astype(dtype)
    lo, hi, r = np.full(D, -2.0, dtype=dtype), np.full(D, side + 2, dtype=dtype), dtype(1.0)
    nhs = make_nhs(pts, r, lo, hi, cap=1000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    counts = torch.zeros(n, dtype=torch.int32, device="cuda")
    sums = torch.zeros(n, dtype=torch.int64, device="cuda")

    def traverse():
        check(load().pn_count_neighbors(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(counts.data_ptr()), 0))
        check(load().pn_sum_neighbor_indices(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(sums.data_ptr()), 0, 0))

    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        nhs._set_stream(x)
        traverse()
    nhs._set_stream(x)
    for move in (0.0, 0.7, 2.0, 0.0):
        now = (pts + move * rng.uniform(-1.0, 1.0, pts.shape)).astype(dtype)
        y = dev(now)
        check(load().pn_grid_refresh(nhs._handle, ctypes.c_void_p(y.data_ptr()), n))
        cells = np.floor((pts - nhs.cell_list.min_corner.astype(dtype)) / np.asarray(nhs.cell_size, dtype)).astype(int)
        want_counts, want_sums = neighbors(now, cells, r)
        for again in range(2):
            graph.replay() if again == 0 else traverse()
            assert np.array_equal(counts.cpu().numpy(), want_counts)
            assert np.array_equal(sums.cpu().numpy(), want_sums)
            counts.fill_(-1)
            sums.fill_(-1)
    # binned again: the cells are those of the points where they are
    pn.update(nhs, y, y)
    graph.replay()
    brute = neighbors(now, np.zeros_like(now), r)
    assert np.array_equal(counts.cpu().numpy(), brute[0])
    assert np.array_equal(sums.cpu().numpy(), brute[1])
