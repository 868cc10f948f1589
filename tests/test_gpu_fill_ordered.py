"""Neighbour lists of clouds that the sorted fill takes, 3D with 100,000 points and more in the order of
their cells and 14 and more a cell, against the fill by cells and the separate sort ("algorithm" 1): the
same integers."""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors._lib import PN_QUERIES_GRID, check, load

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def ordered(n, a_cell, seed, dtype):
    """n uniform points in the order of their cells of edge 1, which hold a_cell on average."""
    from test_gpu_fill_sorted import cloud
    pts = cloud(n, a_cell, seed, dtype)
    cell = np.floor(pts - pts.min(axis=0) + 0.001).astype(np.int64)
    return pts[np.lexsort(cell.T)]


def same_lists(nhs, x, y, base=0):
    from test_gpu_fill_sorted import lists
    (rp, col), (rp1, col1) = lists(nhs, x, y, base)
    return torch.equal(rp, rp1) and torch.equal(col, col1)


@pytest.mark.parametrize("dtype,radius", [(np.float32, np.float32), (np.float64, np.float64), (np.float32, np.float64),
                                          (np.float64, np.float32)])
@pytest.mark.parametrize("n,a_cell", [(100_000, 15.5), (100_000, 25.0), (120_000, 42.0)])
def test_fill(n, a_cell, dtype, radius):
    from test_gpu_parity import dev, make_nhs
    pts = ordered(n, a_cell, 5, dtype)
    nhs = make_nhs(pts, radius(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000)
    y = dev(pts)
    pn.initialize(nhs, y, y)
    assert same_lists(nhs, y, y, base=1)
    x = dev(pts[np.random.default_rng(6).permutation(n)] + dtype(0.4))  # another cloud's lists in this one
    pn.initialize(nhs, x, y)
    assert same_lists(nhs, x, y)


def fill(nhs, n, moved=None):
    """(row_ptr, col with a margin, number of entries); `moved` are the coordinates at the fill."""
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    rp = torch.empty(n + 1, dtype=torch.int32, device="cuda")
    nnz, most = ctypes.c_int64(), ctypes.c_int64()
    check(load().pn_csr_count(nhs._handle, PN_QUERIES_GRID, n, vp(rp), 0, ctypes.byref(nnz), ctypes.byref(most)))
    if moved is not None:
        check(load().pn_grid_refresh(nhs._handle, vp(moved), n))
    col = torch.full((nnz.value + 64,), -77, dtype=torch.int32, device="cuda")
    check(load().pn_csr_fill(nhs._handle, PN_QUERIES_GRID, n, vp(rp), vp(col), 0))
    assert nhs.last_traversal() == "sorted fill"
    assert (col[nnz.value:] == -77).all()
    return rp, col, nnz.value


def test_selected_points_and_moved_coordinates():
    from test_gpu_parity import dev, make_nhs
    pts = ordered(300_000, 42.0, 7, np.float32)
    nhs = make_nhs(pts, np.float32(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000)
    y, n = dev(pts), len(pts)
    selected = np.flatnonzero(np.arange(n) % 3 > 0)
    pn.initialize(nhs, y, y, eachindex_y=selected)
    assert nhs.stats()[0] == len(selected)
    assert same_lists(nhs, y, y)
    nhs.set_tuning("algorithm", 0)
    pn.initialize(nhs, y, y)
    center = y.mean(dim=1, keepdim=True)
    rp, col, nnz = fill(nhs, n, ((y - center) * 0.9 + center).t().contiguous().t())
    # more neighbours than were counted: rows keep to their places, ascending up to what was not written
    rows, col = rp.long().cpu().numpy(), col.cpu().numpy()[:nnz]
    assert (col < n).all()
    inside = np.ones(nnz, dtype=bool)
    inside[rows[1:-1][rows[1:-1] < nnz]] = False
    step = np.diff(col.astype(np.int64))
    assert (step[inside[1:]] > 0)[(col[1:] != -77)[inside[1:]]].all()


@pytest.mark.parametrize("status_read", ["stats", "check"])
def test_after_replayed_binnings(status_read):
    """The fill is sized by the device's counters, not by those that the host has read."""
    from test_gpu_parity import dev, make_nhs
    n = 120_000
    pts = ordered(n, 16.0, 3, np.float32)
    side = float(pts.max())
    closer = (0.3 * side + 0.72 * pts).astype(np.float32)  # fuller cells by a factor of 2 to 3
    nhs = make_nhs(pts, np.float32(1.0), np.full(3, -3.0, np.float32), np.full(3, side + 3, np.float32), cap=1000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pn.update(nhs, x, x, check_errors=False)
    nhs._set_stream(x)
    for cloud in (pts, closer, pts, closer):
        x.copy_(torch.as_tensor(cloud.T.copy(), device="cuda"))
        graph.replay()
        if cloud is pts:
            nhs.stats() if status_read == "stats" else nhs.check()
        rp, col, nnz = fill(nhs, n)
        other = pn.GridNeighborhoodSearch[3](search_radius=np.float32(1.0), n_points=n, cell_list=nhs.cell_list)
        other.set_tuning("algorithm", 1)
        pn.initialize(other, x, x)
        rp1 = torch.empty_like(rp)
        total, most = ctypes.c_int64(), ctypes.c_int64()
        vp = lambda t: ctypes.c_void_p(t.data_ptr())
        check(load().pn_csr_count(other._handle, PN_QUERIES_GRID, n, vp(rp1), 0, ctypes.byref(total),
                                  ctypes.byref(most)))
        col1 = torch.empty(total.value, dtype=torch.int32, device="cuda")
        check(load().pn_csr_fill(other._handle, PN_QUERIES_GRID, n, vp(rp1), vp(col1), 0))
        assert torch.equal(rp, rp1) and torch.equal(col[:nnz], col1)
