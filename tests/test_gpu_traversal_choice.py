"""Which kernel a traversal is launched with, on both sides of the lines where the choice changes.
(That the kernels agree there is tested in test_gpu_run_rules.py and test_gpu_fill_sorted.py.)"""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors import sph
from pointneighbors._lib import PN_QUERIES_GRID, check, load

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def search(D, n, a_cell, dtype=np.float32, seed=1):
    """A grid of n uniform points, a_cell per cell of edge 1."""
    from test_gpu_parity import dev, make_nhs
    pts = np.random.default_rng(seed).uniform(0.0, (n / a_cell) ** (1 / D), (n, D)).astype(dtype)
    nhs = make_nhs(pts, dtype(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    return nhs, x


def count(nhs, x, y):
    pn.foreach_point_neighbor(pn.CountNeighbors(torch.zeros(x.shape[1], dtype=torch.int32, device="cuda")), x, y, nhs)
    return nhs.last_traversal()


def density(nhs, x, y):
    m = torch.ones(y.shape[1], dtype=y.dtype, device="cuda")
    rho = torch.zeros(x.shape[1], dtype=y.dtype, device="cuda")
    pn.foreach_point_neighbor(sph.SPHDensity(rho, m, 0.5), x, y, nhs)
    return nhs.last_traversal()


@pytest.mark.parametrize("chunk", [-1, 0, 1])
def test_knobs(chunk):
    nhs, x = search(3, 5000, 10.0)
    assert nhs.last_traversal() == "none"
    nhs.set_tuning("chunk", chunk)
    assert count(nhs, x, x) == "runs" and density(nhs, x, x) == "runs"
    nhs.set_tuning("algorithm", 1)
    assert count(nhs, x, x) == ("slices" if chunk == 0 else "slices (large chunks)")
    assert density(nhs, x, x) == ("slices (large chunks)" if chunk == 1 else "slices")


@pytest.mark.parametrize("n,a_cell,want", [(32767, 5.0, "cells"), (32768, 5.0, "runs"), (65535, 8.0, "cells"),
                                           (65536, 8.0, "runs"), (262143, 11.0, "cells"), (262144, 11.0, "runs")])
def test_2d(n, a_cell, want):
    nhs, x = search(2, n, a_cell)
    assert density(nhs, x, x) == want and count(nhs, x, x) == "runs"


@pytest.mark.parametrize("side,r,want", [(90, 3.2, "runs"), (91, 3.2, "cells"), (91, 2.0, "runs"), (181, 2.6, "cells"),
                                         (182, 2.6, "runs"), (255, 3.2, "cells"), (256, 3.2, "runs")])
def test_2d_periodic(side, r, want):
    from test_gpu_parity import dev
    pts = (np.stack(np.meshgrid(*[np.arange(side)] * 2, indexing="ij"), -1).reshape(-1, 2) + 0.5).astype(np.float32)
    size = np.full(2, side, np.float32)
    box = pn.PeriodicBox(min_corner=np.zeros(2, np.float32), max_corner=size)
    cl = pn.FullGridCellList(min_corner=box.min_corner, max_corner=box.max_corner, search_radius=np.float32(r))
    nhs = pn.GridNeighborhoodSearch[2](search_radius=np.float32(r), n_points=len(pts), periodic_box=box, cell_list=cl)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    assert density(nhs, x, x) == want and count(nhs, x, x) == "runs"


@pytest.mark.parametrize("D,n,a_cell,kinds", [(3, 100_000, 0.02, "cells cells"), (3, 100_000, 0.2, "runs runs"),
                                              (2, 100_000, 0.05, "cells cells"), (2, 100_000, 0.2, "runs runs"),
                                              (3, 20_000, 0.05, "runs cells"), (3, 20_000, 0.3, "runs runs"),
                                              (3, 8000, 0.02, "runs runs")])
def test_sparse_clouds(D, n, a_cell, kinds):
    nhs, x = search(D, n, a_cell)
    assert [count(nhs, x, x), density(nhs, x, x)] == kinds.split()


@pytest.mark.parametrize("n_x,want", [(13333, "cells"), (13334, "runs")])
def test_sparse_queries(n_x, want):
    nhs, y = search(3, 80_000, 10.0)
    x = y[:, :n_x].t().contiguous().t()
    assert count(nhs, x, y) == want


@pytest.mark.parametrize("D,n,a_cell,order,want", [(3, 100_000, 16.0, "cells", "sorted fill"),
                                                   (3, 99_999, 16.0, "cells", "cells"),
                                                   (3, 100_000, 12.5, "cells", "cells"),
                                                   (2, 100_000, 16.0, "cells", "cells"),
                                                   (3, 100_000, 16.0, "none", "cells")])
def test_list_fill(D, n, a_cell, order, want):
    nhs, x = search(D, n, a_cell)
    if order == "cells":
        sorted_idx = torch.empty(n, dtype=torch.int32, device="cuda")
        check(load().pn_grid_copy_cells(nhs._handle, None, ctypes.c_void_p(sorted_idx.data_ptr())))
        x = x[:, sorted_idx.long()].t().contiguous().t()
        pn.initialize(nhs, x, x)
    vp = lambda t: ctypes.c_void_p(t.data_ptr())
    rp = torch.empty(n + 1, dtype=torch.int32, device="cuda")
    nnz, longest = ctypes.c_int64(), ctypes.c_int64()
    check(load().pn_csr_count(nhs._handle, PN_QUERIES_GRID, n, vp(rp), 0, ctypes.byref(nnz), ctypes.byref(longest)))
    assert nhs.last_traversal() == "cells"
    col = torch.empty(nnz.value, dtype=torch.int32, device="cuda")
    check(load().pn_csr_fill(nhs._handle, PN_QUERIES_GRID, n, vp(rp), vp(col), 0))
    assert nhs.last_traversal() == want


def test_full_rows_in_an_empty_domain():
    """Points one to a cell on a plane of a wide domain: rows of cells are full, runs are long."""
    from test_gpu_parity import dev, make_nhs
    rng = np.random.default_rng(2)
    pts = np.zeros((320 * 320, 3), np.float32)
    pts[:, :2] = np.stack(np.meshgrid(*[np.arange(320)] * 2), -1).reshape(-1, 2) + rng.uniform(0.1, 0.9, (320 * 320, 2))
    nhs = make_nhs(pts, np.float32(1.0), np.full(3, -50.0, np.float32), np.full(3, 370.0, np.float32), cap=1000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    assert count(nhs, x, x) == "runs" and density(nhs, x, x) == "runs"
