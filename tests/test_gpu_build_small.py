"""Cell lists at the sizes where the binning changes its kernels: one workgroup up to 4096 points in
up to 11,264 cells, one workgroup's scan up to 16,384 cells.  Cell offsets, the order inside the cells
and the neighbour counts against numpy and all pairs; errors are reported and do not outlive their
binning."""

import numpy as np
import pytest

import pointneighbors as pn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def cells_of(nhs, C):
    import ctypes
    from pointneighbors._lib import load
    n, nonempty, most = nhs.stats()
    start = np.empty(C + 1, dtype=np.int32)
    idx = np.empty(max(n, 1), dtype=np.int32)
    ptr = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    s, i = (torch.empty(a.size, dtype=torch.int32, device="cuda") for a in (start, idx))
    assert load().pn_grid_copy_cells(nhs._handle, ctypes.c_void_p(s.data_ptr()), ctypes.c_void_p(i.data_ptr())) == 0
    return s.cpu().numpy(), i.cpu().numpy()[:n], nonempty, most


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n,side,D", [(1, 4, 2), (3, 4, 3), (1025, 10, 3), (4096, 18, 3), (4097, 18, 3), (4096, 100, 2),
                                      (4096, 110, 2), (5000, 123, 2), (5000, 126, 2), (2000, 2, 3)])
def test_cells(n, side, D, dtype):
    from test_gpu_parity import dev, make_nhs
    rng = np.random.default_rng(n + side)
    pts = rng.uniform(0.0, side, (n, D)).astype(dtype)
    nhs = make_nhs(pts, dtype(1.0), np.zeros(D), np.full(D, float(side)), cap=5000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    dims = np.asarray(nhs.cell_list.n_cells)[:D]
    lo = np.asarray(nhs.cell_list.min_corner, dtype=np.float64)[:D]
    cell = np.floor(pts.astype(np.float64) - lo).astype(np.int64)
    cell_low = np.floor((pts - lo.astype(dtype)) / dtype(1.0)).astype(np.int64)
    cell = np.where(cell == cell_low, cell, cell_low)  # the reference divides in the coordinate type
    key = np.zeros(n, dtype=np.int64)
    for d in reversed(range(D)):
        key = key * dims[d] + cell[:, d]
    C = int(np.prod(dims))
    start, idx, nonempty, most = cells_of(nhs, C)
    counts = np.bincount(key, minlength=C)
    assert np.array_equal(np.diff(start), counts) and start[0] == 0
    assert nonempty == (counts > 0).sum() and most == counts.max()
    if most <= 1024:
        assert np.array_equal(idx, np.argsort(key, kind="stable"))
    cnt = torch.zeros(n, dtype=torch.int32, device="cuda")
    pn.foreach_point_neighbor(pn.CountNeighbors(cnt), x, x, nhs)
    want = np.zeros(n, dtype=np.int64)
    for b in range(0, n, 512):
        d2 = np.zeros((len(pts[b:b + 512]), n), dtype=dtype)
        for d in range(D):
            diff = pts[b:b + 512, None, d] - pts[None, :, d]
            d2 = d2 + diff * diff
        want[b:b + 512] = (d2 <= dtype(1.0)).sum(axis=1)
    assert np.array_equal(cnt.cpu().numpy(), want)


@pytest.mark.parametrize("n", [100, 4096, 4097, 40000])
def test_error_is_of_its_binning(n):
    from test_gpu_parity import dev, make_nhs
    rng = np.random.default_rng(3)
    pts = rng.uniform(0.0, 20.0, (n, 3)).astype(np.float32)
    nhs = make_nhs(pts, np.float32(1.0), np.zeros(3), np.full(3, 20.0), cap=5000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    bad = pts.copy()
    bad[n // 2] = 500.0
    with pytest.raises(pn.PointNeighborsError):
        pn.initialize(nhs, dev(bad), dev(bad))
    pn.initialize(nhs, x, x)
    assert nhs.stats()[0] == n
