"""The autotuner's default space: a candidate chunk is timed only where the step's traversal has one."""

import numpy as np
import pytest

import pointneighbors as pn
from pointneighbors import autotune

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_x,timed", [(9000, 12), (400, 16)])
def test_default_space(n_x, timed):
    from test_gpu_parity import dev, make_nhs
    pts = np.random.default_rng(1).uniform(0.0, 12.0, (9000, 3)).astype(np.float32)
    nhs = make_nhs(pts, np.float32(1.5), pts.min(axis=0) - 5, pts.max(axis=0) + 5, cap=1000)
    y = dev(pts)
    x = y if n_x == 9000 else y[:, :n_x].t().contiguous().t()
    counts = torch.zeros(n_x, dtype=torch.int32, device="cuda")
    f = pn.CountNeighbors(counts, accumulate=False)

    def step():
        pn.update(nhs, x, y)
        pn.foreach_point_neighbor(f, x, y, nhs)

    best, table = autotune.autotune(nhs, step, reps=1, warmup=1)
    assert len(table) == timed and best in [e["params"] for e in table]
    assert len({tuple(sorted(e["params"].items())) for e in table}) == timed
