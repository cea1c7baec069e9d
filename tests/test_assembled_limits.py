"""Limits of the assembly by rows that need no GPU: meshes beyond them are left
to the hash table."""
from types import SimpleNamespace

import torch

from afsi_gpu_amd.mac.assembled import AssembledTransfer
from afsi_gpu_amd.mac.grid import MACGrid


def routed_to_the_table(nodes, points=4):
    weights = torch.ones((2, points), dtype=torch.float64)
    geometry = SimpleNamespace(cells=torch.ones((2, 4), dtype=torch.int64), weights=weights, node_count=nodes)
    transfer = SimpleNamespace(geometry=geometry, grid=MACGrid((8, 8, 8), (1., 1., 1.)), max_entries=10)
    try:
        return AssembledTransfer._rows(transfer, None, None) is None
    except AttributeError:  # went on to allocate and launch
        return False


def test_a_wave_per_row_has_to_fit_one_launch(monkeypatch):
    monkeypatch.setattr(torch, 'empty', lambda *a, **k: None)
    monkeypatch.setattr(torch, 'zeros', lambda *a, **k: None)
    limit = (2 ** 32 // 64 - 7) // 3  # 64 threads for each of the 3 N rows, rounded up to 8 rows
    assert routed_to_the_table(limit + 1) and routed_to_the_table(2 ** 28 - 1)
    assert not routed_to_the_table(limit - 1)
    assert routed_to_the_table(100, points=65) and not routed_to_the_table(100, points=64)
