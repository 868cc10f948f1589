"""How the run kernels share their windows of sorted positions among workgroups: every window is taken
once, whatever the number of windows on an XCD and of workgroups, and wavefronts that share a window
take each of its runs once."""

import numpy as np
import pytest

import pointneighbors as pn

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 8, 9, 63, 64, 65, 71, 520, 8191, 8192, 8193, 12_287, 12_289, 16_385, 24_575, 24_577,
                               32_767, 49_153, 65_535, 65_537, 300_001])
def test_every_point_once(n):
    from test_gpu_parity import dev, gpu_sums, make_nhs
    rng = np.random.default_rng(n)
    # a slab of short rows and a thin last layer: windows of one and of many runs
    pts = rng.uniform(0.0, 1.0, (n, 3)) * [5.0, max(1.0, (n / 40) ** 0.5), max(1.0, (n / 40) ** 0.5)]
    pts[: n // 9, 2] = pts[:, 2].max() + 1.0
    pts = pts.astype(np.float32)
    nhs = make_nhs(pts, np.float32(1.0), pts.min(axis=0) - 3, pts.max(axis=0) + 3, cap=1000)
    x = dev(pts)
    pn.initialize(nhs, x, x)
    nhs.set_tuning("algorithm", 1)
    counts = torch.zeros(n, dtype=torch.int32, device="cuda")
    pn.foreach_point_neighbor(pn.CountNeighbors(counts), x, x, nhs)
    sums = gpu_sums(nhs, x, x)
    nhs.set_tuning("algorithm", 0)
    for blocks in (8, 24, 1 << 20):
        nhs.set_tuning("persist_blocks", blocks)
        # accumulating: a window taken twice, or by two wavefronts, would add twice
        got = torch.full((n,), 100, dtype=torch.int32, device="cuda")
        pn.foreach_point_neighbor(pn.CountNeighbors(got, accumulate=True), x, x, nhs)
        assert torch.equal(got, counts + 100), blocks
        assert nhs.last_traversal() == "runs"
        assert np.array_equal(gpu_sums(nhs, x, x), sums), blocks
