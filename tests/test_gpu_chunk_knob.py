"""The knob "chunk" on a FullGridCellList: it selects the cell kernel's variant where a traversal takes
that kernel, with the same neighbour sets."""

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors import sph

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,dtype,periodic", [(2, np.float32, False), (2, np.float64, False), (3, np.float32, False),
                                              (3, np.float32, True), (3, np.float64, True)])
def test_variants_of_the_cell_kernel(D, dtype, periodic):
    from test_gpu_parity import dev
    rng = np.random.default_rng(D)
    side = 24 if D == 3 else 80
    pts = rng.uniform(0.0, side, (9000, D)).astype(dtype)
    r = dtype(1.9)
    kw = {}
    lo, hi = np.zeros(D, dtype=dtype), np.full(D, side, dtype=dtype)
    if periodic:
        kw["periodic_box"] = pn.PeriodicBox(min_corner=lo, max_corner=hi)
    cl = pn.FullGridCellList(min_corner=lo, max_corner=hi, search_radius=r, max_points_per_cell=1000)
    nhs = pn.GridNeighborhoodSearch[D](search_radius=r, n_points=len(pts), cell_list=cl, **kw)
    y = dev(pts)
    x = y[:, ::20].t().contiguous().t()  # sparse queries: cells
    pn.initialize(nhs, x, y)
    mass = 0.5 + torch.rand(len(pts), dtype=y.dtype, device="cuda")
    out = []
    for chunk in (0, 1, -1):
        nhs.set_tuning("chunk", chunk)
        counts = torch.zeros(x.shape[1], dtype=torch.int32, device="cuda")
        rho = torch.zeros(x.shape[1], dtype=y.dtype, device="cuda")
        pn.foreach_point_neighbor(pn.CountNeighbors(counts), x, y, nhs)
        pn.foreach_point_neighbor(sph.SPHDensity(rho, mass, float(r) / 2), x, y, nhs)
        assert nhs.last_traversal() == ("cells" if chunk == 0 else "cells (large chunks)")
        out.append((counts, rho))
    for counts, rho in out[1:]:
        assert torch.equal(counts, out[0][0])
        # n non-negative terms in another order, a term by a few u
        bound = (counts.double() + 16) * np.finfo(dtype).eps * out[0][1].double()
        assert ((rho - out[0][1]).abs().double() <= bound).all()
