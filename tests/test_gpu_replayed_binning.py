"""Traversals of a grid whose binning is replayed from a captured graph and drops points outside the
domain: the points that are left are found and counted as by a binning of them alone, whatever
number of points the host has read before."""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors._lib import PN_QUERIES_GRID, check, load

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

UNTOUCHED = -7


@pytest.mark.parametrize("n", [700, 40_000])
@pytest.mark.parametrize("D", [2, 3])
def test_dropped_points(n, D):
    from test_gpu_parity import dev, gpu_counts, make_nhs
    rng = np.random.default_rng(n)
    side = (n / 8.0) ** (1 / D)
    pts = rng.uniform(0.0, side, (n, D)).astype(np.float32)
    lo, hi = np.full(D, -1.0, np.float32), np.full(D, side + 1, np.float32)
    r = np.float32(1.0)
    nhs = make_nhs(pts, r, lo, hi, cap=1000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pn.update(nhs, x, x, check_errors=False)
    nhs._set_stream(x)
    graph.replay()
    assert nhs.stats()[0] == n
    for dropped in (range(0), range(0, n, 3), range(n // 2, n), range(0)):
        keep = np.ones(n, bool)
        keep[list(dropped)] = False
        cloud = pts.copy()
        cloud[~keep] = np.nan
        x.copy_(torch.as_tensor(cloud.T.copy(), device="cuda"))
        graph.replay()
        counts = torch.full((n,), UNTOUCHED, dtype=torch.int32, device="cuda")
        sums = torch.full((n,), UNTOUCHED, dtype=torch.int64, device="cuda")
        check(load().pn_count_neighbors(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(counts.data_ptr()), 0))
        check(load().pn_sum_neighbor_indices(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(sums.data_ptr()), 0, 0))
        alone = make_nhs(pts[keep], r, lo, hi, cap=1000)
        z = dev(pts[keep])
        pn.initialize(alone, z, z)
        want = np.full(n, UNTOUCHED)
        want[keep] = gpu_counts(alone, z, z)
        assert np.array_equal(counts.cpu().numpy(), want)
        # sums of original indices: of a binning of the kept points by a selection list
        listed = make_nhs(pts, r, lo, hi, cap=1000)
        w = dev(pts)
        pn.initialize(listed, w, w, eachindex_y=np.flatnonzero(keep))
        full = torch.full((n,), UNTOUCHED, dtype=torch.int64, device="cuda")
        check(load().pn_sum_neighbor_indices(listed._handle, PN_QUERIES_GRID, ctypes.c_void_p(full.data_ptr()), 0, 0))
        assert torch.equal(sums, full)


@pytest.mark.parametrize("n,fewer", [(700, 40), (700, 699), (40_000, 300), (40_000, 39_000)])
def test_more_points_than_the_host_knows(n, fewer):
    """A replay bins more points than the program's own last update did."""
    from test_gpu_parity import dev, gpu_counts, gpu_sums, make_nhs
    side = (n / 8.0) ** (1 / 3)
    pts = np.random.default_rng(n).uniform(0.0, side, (n, 3)).astype(np.float32)
    nhs, plain = (make_nhs(pts, np.float32(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000) for _ in range(2))
    x = dev(pts)
    pn.initialize(nhs, x, x)
    pn.initialize(plain, x, x)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pn.update(nhs, x, x, check_errors=False)
    nhs._set_stream(x)
    check(load().pn_grid_update(nhs._handle, ctypes.c_void_p(x.data_ptr()), n, 0, fewer, None))
    graph.replay()
    counts = torch.zeros(n, dtype=torch.int32, device="cuda")
    sums = torch.zeros(n, dtype=torch.int64, device="cuda")
    check(load().pn_count_neighbors(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(counts.data_ptr()), 0))
    check(load().pn_sum_neighbor_indices(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(sums.data_ptr()), 0, 0))
    assert np.array_equal(counts.cpu().numpy(), gpu_counts(plain, x, x))
    assert np.array_equal(sums.cpu().numpy(), gpu_sums(plain, x, x))


@pytest.mark.parametrize("algorithm", [0, 1])
@pytest.mark.parametrize("D", [1, 3])
def test_host_knows_of_an_empty_binning(D, algorithm):
    """The host has read the status of a replay that dropped every point; the next one bins them all."""
    from test_gpu_parity import dev, gpu_counts, make_nhs
    n = 700
    pts = np.random.default_rng(n).uniform(0.0, 5.0, (n, D)).astype(np.float32)
    nhs, plain = (make_nhs(pts, np.float32(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000) for _ in range(2))
    x, y = dev(pts), dev(pts)
    pn.initialize(nhs, x, x)
    pn.initialize(plain, y, y)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        pn.update(nhs, x, x, check_errors=False)
    nhs._set_stream(x)
    x.fill_(float("nan"))
    graph.replay()
    assert nhs.stats()[0] == 0
    x.copy_(y)
    graph.replay()
    nhs.set_tuning("algorithm", algorithm)
    counts = torch.full((n,), UNTOUCHED, dtype=torch.int32, device="cuda")
    check(load().pn_count_neighbors(nhs._handle, PN_QUERIES_GRID, ctypes.c_void_p(counts.data_ptr()), 0))
    assert np.array_equal(counts.cpu().numpy(), gpu_counts(plain, y, y))
