"""The default traversal reads the coordinates as they are now: after an update and after an in-place
move its sums are those of the per-query slices ("algorithm" 1), an independent kernel, within the
bound of another order of the same terms, and those of a search built anew.  The keys "pair_cache"
and "pair_cache_per_point" are accepted and change nothing."""

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors import sph, synthetic

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def setup(dtype):
    from test_gpu_parity import dev, make_nhs
    pts = synthetic.jittered_lattice((36, 37, 38), 0.01, 0.001, dtype=dtype, seed=3)
    r = dtype(2) * (dtype(1.2) * dtype(0.01))
    make = lambda: make_nhs(pts, r, pts.min(axis=0) - 3 * r, pts.max(axis=0) + 3 * r)
    x = dev(pts)
    nhs = make()
    pn.initialize(nhs, x, x)
    return nhs, x, make


def sums(nhs, x, algorithm=0):
    nhs.set_tuning("algorithm", algorithm)
    n, dt = x.shape[1], x.dtype
    mass = torch.full((n,), 1e-3, dtype=dt, device="cuda")
    rho, e = torch.zeros(n, dtype=dt, device="cuda"), torch.zeros(n, dtype=dt, device="cuda")
    counts = torch.zeros(n, dtype=torch.int32, device="cuda")
    pn.foreach_point_neighbor(sph.SPHDensity(rho, mass, float(nhs.search_radius) / 2), x, x, nhs)
    pn.foreach_point_neighbor(sph.WendlandPairEnergy(e, 1.0, float(nhs.search_radius)), x, x, nhs)
    pn.foreach_point_neighbor(pn.CountNeighbors(counts), x, x, nhs)
    nhs.set_tuning("algorithm", 0)
    return counts, rho, e


def assert_same(got, want):
    assert torch.equal(got[0], want[0])
    u = torch.finfo(got[1].dtype).eps
    for a, b in zip(got[1:], want[1:]):  # non-negative terms in another order, a term by a few u
        assert ((a - b).abs().double() <= (want[0].double() + 16) * u * b.double()).all()


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_update(dtype):
    nhs, x, make = setup(dtype)
    before = sums(nhs, x)
    x.add_(torch.empty_like(x).uniform_(-5e-4, 5e-4))
    pn.update(nhs, x, x)
    got = sums(nhs, x)
    assert not torch.equal(got[0], before[0])
    assert_same(got, sums(nhs, x, 1))
    new = make()
    pn.initialize(new, x, x)
    for a, b in zip(got, sums(new, x)):
        assert torch.equal(a, b)


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_in_place(dtype):
    nhs, x, _ = setup(dtype)
    before = sums(nhs, x)
    x.add_(torch.empty_like(x).uniform_(-3e-3, 3e-3))
    got = sums(nhs, x)
    assert not torch.equal(got[0], before[0])
    assert_same(got, sums(nhs, x, 1))


def test_keys_without_effect():
    nhs, x, _ = setup(np.float32)
    before = sums(nhs, x)
    for key, value in (("pair_cache", 1), ("pair_cache_per_point", 12)):
        nhs.set_tuning(key, value)
        for a, b in zip(before, sums(nhs, x)):
            assert torch.equal(a, b)
    for key, value in (("pair_cache", 2), ("pair_cache_per_point", -1)):
        with pytest.raises(pn.ArgumentError):
            nhs.set_tuning(key, value)
