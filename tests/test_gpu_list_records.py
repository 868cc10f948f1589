"""The list kernels over packed records against the same kernels over the separate fields: the
lanes add the same terms in the same order, so the results are equal bit for bit.  (The field
kernels are compared with the oracle in test_gpu_tlsph.py and test_gpu_periodic.py.)"""

import ctypes

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors import sph, synthetic
from pointneighbors._lib import PN_ERR_ARGUMENT, PN_ERR_UNSUPPORTED, load
from test_gpu_parity import dev

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def both(monkeypatch, f):
    """f() with the records forced and with the fields forced."""
    def records(nl, ndims, code, n, rows, records=1):
        return torch.full((load().pn_list_pack_bytes(code, records * n),), 255, dtype=torch.uint8, device="cuda")
    out = []
    for choose in (records, lambda *a, **k: None):
        monkeypatch.setattr(sph, "_list_records", choose)
        out.append(f())
    return out


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("shape,radius", [((1, 1), 1.0), ((3, 11), 0.2), ((40, 33), 3.0), ((9, 8, 7), 1.6),
                                          ((17, 16, 15), 3.1)])
def test_density(monkeypatch, shape, radius, dt, periodic):
    nd = len(shape)
    Y = synthetic.jittered_lattice(shape, 1.0, 0.2, dtype=dt, seed=2)
    box = None
    if periodic:
        box = pn.PeriodicBox(min_corner=[dt(0)] * nd, max_corner=[dt(max(s, 4 * radius)) for s in shape])
    p = pn.PrecomputedNeighborhoodSearch(nd, search_radius=dt(radius), n_points=len(Y), max_neighbors=4096,
                                         periodic_box=box)
    n_x = max(1, len(Y) - 3)
    x, y = dev(Y[::-1][:n_x].copy()), dev(Y)  # lists of one cloud in another, of fewer points
    pn.initialize(p, x, y)
    m = torch.as_tensor((1.0 + 0.1 * synthetic.uniform(5, len(Y))).astype(dt), device="cuda")

    def run(points=None):
        rho = torch.full((n_x,), 0.5, dtype=m.dtype, device="cuda")
        f = sph.SPHDensity(rho, m, radius / 2)
        pn.foreach_point_neighbor(f, x, y, p, **({} if points is None else dict(points=points)))
        return rho

    a, b = both(monkeypatch, run)
    assert torch.equal(a, b) and torch.isfinite(a).all()
    some = list(range(n_x - 1, -1, -3))
    a, b = both(monkeypatch, lambda: run(some))
    assert torch.equal(a, b)


@pytest.mark.parametrize("shape", [(1, 2), (30, 27), (3, 3, 2), (16, 15, 14)])
def test_deformation_gradient(monkeypatch, shape):
    X = synthetic.jittered_lattice(shape, 1.0, 0.15, dtype=np.float32, seed=9)
    n, nd = X.shape
    Xd = dev(X)
    p = pn.PrecomputedNeighborhoodSearch(nd, search_radius=np.float32(2.6), n_points=n, max_neighbors=4096)
    pn.initialize(p, Xd, Xd)
    rng = np.random.default_rng(1)
    x = dev((X + 0.1 * rng.standard_normal(X.shape)).astype(np.float32))
    V = torch.as_tensor((1.0 + 0.1 * synthetic.uniform(5, n)).astype(np.float32), device="cuda")
    L = torch.as_tensor(rng.standard_normal((n, nd, nd)).astype(np.float32), device="cuda")
    for kw in ({}, {"correction": L}, {"_invert": True}):
        a, b = both(monkeypatch, lambda: sph.tlsph_deformation_gradient(p, Xd, x, V, 1.3, **kw))
        assert torch.equal(torch.nan_to_num(a), torch.nan_to_num(b))
    some = list(range(n - 1, -1, -2))
    a, b = both(monkeypatch, lambda: sph.tlsph_deformation_gradient(p, Xd, x, V, 1.3, points=some)[some])
    assert torch.equal(a, b)


def test_rule_and_refusals():
    n, entries = 200_000, 20_000_000
    nl = pn.nhs_precomputed.NeighborLists(None, torch.empty(entries, dtype=torch.int32, device="cuda"), n, 4096)
    assert sph._list_records(nl, 3, 0, n, n).numel() == 16 * n
    assert sph._list_records(nl, 3, 1, n, n).numel() == 32 * n
    assert sph._list_records(nl, 2, 0, n, n, records=2).numel() == 32 * n
    assert sph._list_records(nl, 2, 1, n, n) is None            # half of each record is padding
    assert sph._list_records(nl, 3, 0, n, n // 2) is None       # too few selected rows
    assert sph._list_records(nl, 3, 0, 5 * n, n) is None        # too many points to pack
    ws = torch.zeros(64, dtype=torch.uint8, device="cuda")
    i = torch.zeros(2, dtype=torch.int32, device="cuda")
    v = torch.zeros(4, dtype=torch.float64, device="cuda")
    ptr = lambda t, off=0: ctypes.c_void_p(t.data_ptr() + off)
    dens = lambda dtype, n_y, w: load().pn_list_sph_density_packed(
        ptr(i), ptr(i), 1, 0, 3, dtype, 0, 1.0, ptr(v), ptr(v), n_y, ptr(v), 0, 1, None, ptr(v), 0, 1.0, None, w, None)
    grad = lambda dtype, w: load().pn_list_tlsph_deformation_grad_packed(
        ptr(i), ptr(i), 1, 0, 3, dtype, 0, 1.0, ptr(v), ptr(v), ptr(v), None, 0, 0, 1, None, ptr(v), w, None)
    assert dens(0, 1, ptr(ws, 8)) == PN_ERR_ARGUMENT and dens(0, 1, None) == PN_ERR_ARGUMENT
    assert dens(0, 0, ptr(ws)) == PN_ERR_ARGUMENT
    assert grad(0, ptr(ws, 8)) == PN_ERR_ARGUMENT and grad(0, None) == PN_ERR_ARGUMENT
    assert grad(1, ptr(ws)) == PN_ERR_UNSUPPORTED
    assert load().pn_list_pack_bytes(2, 1) == -1 and load().pn_list_pack_bytes(0, -1) == -1
