"""Neighbour lists of a grid whose binning is replayed from a captured graph: the host's copy of the
grid's counters is then that of an earlier binning, and a fill sized by it would cut lists short."""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors._lib import PN_QUERIES_GRID, check, load

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

N = 120_000
SENTINEL = -77


def vp(t):
    return ctypes.c_void_p(t.data_ptr())


def lists(nhs):
    """(row_ptr, col) of the sorted fill and of the fill by cells."""
    out = []
    for algorithm in (0, 1):
        nhs.set_tuning("algorithm", algorithm)
        rp = torch.empty(N + 1, dtype=torch.int32, device="cuda")
        nnz, longest = ctypes.c_int64(), ctypes.c_int64()
        check(load().pn_csr_count(nhs._handle, PN_QUERIES_GRID, N, vp(rp), 0, ctypes.byref(nnz), ctypes.byref(longest)))
        col = torch.full((nnz.value,), SENTINEL, dtype=torch.int32, device="cuda")
        check(load().pn_csr_fill(nhs._handle, PN_QUERIES_GRID, N, vp(rp), vp(col), 0))
        out.append((rp, col))
    nhs.set_tuning("algorithm", 0)
    return out


@pytest.mark.parametrize("status_read", ["stats", "check"])
def test_lists_after_replayed_binnings(status_read):
    from test_gpu_parity import dev, make_nhs
    side = (N / 14.0) ** (1 / 3)
    rng = np.random.default_rng(3)
    pts = rng.uniform(0.0, side, (N, 3)).astype(np.float32)
    # drawn together: fuller cells than the status that the host has read, by a factor of 2 to 3
    closer = (0.3 * side + 0.72 * pts).astype(np.float32)
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
        (rp, col), (rp1, col1) = lists(nhs)
        assert torch.equal(rp, rp1) and torch.equal(col, col1)


@pytest.mark.parametrize("shift", [0.0, 0.37])
def test_captured_fill(shift):
    """A captured fill is replayed over the binning of a cloud that moved as a whole, exactly: the
    lists are the same, the cells are not."""
    from test_gpu_parity import dev, make_nhs
    side = (N / 14.0) ** (1 / 3)
    rng = np.random.default_rng(4)
    # multiples of 2^-12: differences stay exact under the shift
    pts = (np.round(rng.uniform(0.0, side, (N, 3)) * 4096) / 4096).astype(np.float32)
    moved = (pts + np.float32(np.round(shift * 4096) / 4096)).astype(np.float32)
    nhs = make_nhs(pts, np.float32(1.0), np.full(3, -3.0, np.float32), np.full(3, side + 3, np.float32), cap=1000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    torch.cuda.synchronize()
    binning, fill = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(binning):
        pn.update(nhs, x, x, check_errors=False)
    nhs._set_stream(x)
    binning.replay()
    (rp, col), _ = lists(nhs)
    got = torch.full_like(col, SENTINEL)
    torch.cuda.synchronize()
    with torch.cuda.graph(fill):
        nhs._set_stream(x)
        check(load().pn_csr_fill(nhs._handle, PN_QUERIES_GRID, N, vp(rp), vp(got), 0))
    nhs._set_stream(x)
    for cloud in (pts, moved, pts):
        x.copy_(torch.as_tensor(cloud.T.copy(), device="cuda"))
        got.fill_(SENTINEL)
        binning.replay()
        fill.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, col)
