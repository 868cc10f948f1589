"""Crowded cells in a one-workgroup binning: the order inside the cells is that of the original indices
on both sides of the line where the placement changes (fullest cell of 64 points), for whole clouds
and for lists of points in order, out of order and with repetitions."""

import numpy as np
import pytest

import pointneighbors as pn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def check_order(nhs, keys, selection):
    from test_gpu_build_small import cells_of
    C = int(np.prod(nhs.cell_list.n_cells))
    start, idx, nonempty, most = cells_of(nhs, C)
    key = keys[selection]
    counts = np.bincount(key, minlength=C)
    assert np.array_equal(np.diff(start), counts)
    assert nonempty == (counts > 0).sum() and most == counts.max()
    assert np.array_equal(idx, selection[np.lexsort((selection, key))])


@pytest.mark.parametrize("n,crowd", [(63, 63), (64, 64), (65, 64), (700, 65), (1024, 1024), (2000, 63), (2000, 64),
                                     (3333, 500), (4095, 1000), (4096, 64)])
@pytest.mark.parametrize("D", [2, 3])
def test_order(n, crowd, D):
    from test_gpu_parity import dev, make_nhs
    rng = np.random.default_rng(n + crowd)
    side = 19 if D == 3 else 90
    pts = np.empty((n, D), np.float32)
    # `crowd` points in the fullest cell, the others 1 to 8 a cell
    cell = rng.permutation(side**D)[np.arange(n) // 8 + 1]
    at = rng.permutation(n)
    cell[at[:crowd]] = cell[at[0]] = side**D // 2
    for d in range(D):
        pts[:, d] = (cell // side**d) % side + rng.uniform(0.01, 0.99, n)
    nhs = make_nhs(pts, np.float32(1.0), np.zeros(D, np.float32), np.full(D, float(side), np.float32), cap=5000)
    lo = np.asarray(nhs.cell_list.min_corner, dtype=np.float32)[:D]
    dims = np.asarray(nhs.cell_list.n_cells)[:D]
    c = np.floor((pts - lo) / np.float32(1.0)).astype(np.int64)
    keys = sum(c[:, d] * int(np.prod(dims[:d])) for d in range(D))
    x = dev(pts)
    everything = np.arange(n)
    selections = [everything, everything[: n // 2 + 1], everything[::-1].copy(), np.sort(rng.integers(0, n, n)),
                  rng.permutation(n), np.repeat(everything[n // 2:], 2)[:n]]
    for k, sel in enumerate(selections):
        pn.initialize(nhs, x, x, **({} if k == 0 else {"eachindex_y": sel}))
        check_order(nhs, keys, sel)
