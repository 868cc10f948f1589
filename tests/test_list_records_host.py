"""When the list kernels take a workspace of packed records: by the number of entries, and not where
the memory has no room for it."""

from types import SimpleNamespace

import pytest

from pointneighbors import sph
from pointneighbors._lib import PN_FLOAT32, PN_FLOAT64

torch = pytest.importorskip("torch")


def lists(n, entries):
    col = SimpleNamespace(numel=lambda: entries, device=torch.device("cpu"))
    return SimpleNamespace(n=n, col_idx=col)


def test_rule():
    assert sph._list_records(lists(100_000, 12_000_000), 3, PN_FLOAT32, 100_000, 100_000).numel() == 1_600_000
    assert sph._list_records(lists(100_000, 12_000_000), 3, PN_FLOAT32, 100_000, 100_000, 2).numel() == 3_200_000
    assert sph._list_records(lists(100_000, 12_000_000), 3, PN_FLOAT64, 100_000, 100_000).numel() == 3_200_000
    assert sph._list_records(lists(100_000, 11_999_999), 3, PN_FLOAT32, 100_000, 100_000) is None
    assert sph._list_records(lists(100_000, 12_000_000), 3, PN_FLOAT32, 100_000, 99_000) is None
    assert sph._list_records(lists(600_000, 12_000_000), 3, PN_FLOAT32, 600_000, 600_000) is None
    assert sph._list_records(lists(100_000, 12_000_000), 2, PN_FLOAT64, 100_000, 100_000) is None


def test_without_room(monkeypatch):
    def full(*args, **kwargs):
        raise torch.OutOfMemoryError("no room")

    monkeypatch.setattr(torch, "empty", full)
    assert sph._list_records(lists(100_000, 12_000_000), 3, PN_FLOAT32, 100_000, 100_000) is None
