"""Neighbour lists of clouds that the sorted fill takes (3D, 100,000 points and more, 12 and more a
cell), against the fill by cells and the separate sort ("algorithm" 1): the same integers."""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors._lib import PN_QUERIES_GRID, load

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SENTINEL = -77


def cloud(n, a_cell, seed, dtype):
    """n uniform points whose cells of edge 1 hold a_cell on average."""
    rng = np.random.default_rng(seed)
    return rng.uniform(0.0, (n / a_cell) ** (1 / 3), (n, 3)).astype(dtype)


def lists(nhs, x, y, base=0):
    """(row_ptr, col) by each algorithm; col has a margin that nothing may write to."""
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    out = []
    for algorithm in (0, 1):
        nhs.set_tuning("algorithm", algorithm)
        mode, xx = nhs._prepare(x, y, None)
        n = xx.shape[1]
        rp = torch.empty(n + 1, dtype=torch.int32, device="cuda")
        nnz, mx = ctypes.c_int64(), ctypes.c_int64()
        assert load().pn_csr_count(nhs._handle, mode, n, vp(rp), 0, ctypes.byref(nnz), ctypes.byref(mx)) == 0
        col = torch.full((nnz.value + 64,), SENTINEL, dtype=torch.int32, device="cuda")
        assert load().pn_csr_fill(nhs._handle, mode, n, vp(rp), vp(col), base) == 0
        assert (col[nnz.value:] == SENTINEL).all()
        out.append((rp, col))
    return out


@pytest.mark.parametrize("dtype,radius", [(np.float32, np.float32), (np.float64, np.float64), (np.float32, np.float64),
                                          (np.float64, np.float32)])
@pytest.mark.parametrize("n,a_cell", [(100_000, 12.5), (100_000, 25.0), (120_000, 42.0)])
def test_fill(n, a_cell, dtype, radius):
    from test_gpu_parity import dev, make_nhs
    pts = cloud(n, a_cell, 5, dtype)
    nhs = make_nhs(pts, radius(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000)
    y = dev(pts)
    pn.initialize(nhs, y, y)
    (rp, col), (rp1, col1) = lists(nhs, y, y, base=1)
    assert torch.equal(rp, rp1) and torch.equal(col, col1)
    x = dev(cloud(n + 3, a_cell, 6, dtype))  # another cloud's lists in this one
    pn.initialize(nhs, x, y)
    (rp, col), (rp1, col1) = lists(nhs, x, y)
    assert torch.equal(rp, rp1) and torch.equal(col, col1)


def test_selected_points_and_moved_coordinates():
    from test_gpu_parity import dev, make_nhs
    pts = cloud(200_000, 28.0, 7, np.float32)
    nhs = make_nhs(pts, np.float32(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000)
    y = dev(pts)
    pn.initialize(nhs, y, y, eachindex_y=range(1, 200_000, 2))
    (rp, col), (rp1, col1) = lists(nhs, y, y)
    assert torch.equal(rp, rp1) and torch.equal(col, col1)
    # more neighbours than were counted: rows keep to their places
    pn.initialize(nhs, y, y)
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    n = len(pts)
    rp = torch.empty(n + 1, dtype=torch.int32, device="cuda")
    nnz, mx = ctypes.c_int64(), ctypes.c_int64()
    assert load().pn_csr_count(nhs._handle, PN_QUERIES_GRID, n, vp(rp), 0, ctypes.byref(nnz), ctypes.byref(mx)) == 0
    col = torch.full((nnz.value + 64,), SENTINEL, dtype=torch.int32, device="cuda")
    center = y.mean(dim=1, keepdim=True)
    closer = ((y - center) * 0.9 + center).t().contiguous().t()
    assert load().pn_grid_refresh(nhs._handle, vp(closer), n) == 0
    assert load().pn_csr_fill(nhs._handle, PN_QUERIES_GRID, n, vp(rp), vp(col), 0) == 0
    rows, col = rp.long().cpu().numpy(), col.cpu().numpy()
    assert (col[nnz.value:] == SENTINEL).all() and (col[:nnz.value] < n).all()
    inside = np.ones(nnz.value, dtype=bool)  # ascending within each row up to what was not written
    inside[rows[1:-1][rows[1:-1] < nnz.value]] = False
    step = np.diff(col[:nnz.value].astype(np.int64))
    assert (step[inside[1:]] > 0)[(col[1:nnz.value] != SENTINEL)[inside[1:]]].all()
