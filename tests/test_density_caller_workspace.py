"""A workspace that the caller sized for the algorithm it asks for is used, with
that algorithm, also where the op by itself would take another."""
import pytest
import torch

from dreamplace_amd import _native as N
from dreamplace_amd import electric_overflow as eo


@pytest.mark.parametrize("room,runs", [("global", N.DP_SCATTER_GLOBAL), ("tiled", N.DP_SCATTER_TILED),
                                       (None, N.DP_SCATTER_TILED)])
def test_workspace(monkeypatch, room, runs):
    monkeypatch.setattr(eo, "TILED_MIN_CELLS", 1)
    monkeypatch.setattr(N, "require_gpu", lambda *a, **k: None)
    monkeypatch.setattr(N, "stream_ptr", lambda device=None: 0)
    calls = []
    monkeypatch.setattr(N, "call", lambda name, *a: calls.append(a))
    n, nb = 100, 64
    ones = torch.ones(n)
    ws = None
    if room:
        ws = torch.empty(N.query("dp_density_map_workspace_bytes", nb, nb, n, 64,
                                 eo.algorithm_code(room), N.DP_FLOAT32), dtype=torch.uint8)
    eo.ElectricDensityMapFunction.forward(
        torch.zeros(2 * n), ones, ones, ones, ones, ones, None, None, None, 0.9, 0.0, 0.0, 64.0,
        64.0, 1.0, 1.0, n, 0, 0, None, nb, nb, 3, 3, 3, 3, True, None, algorithm="global",
        large_capacity=64, workspace=ws)
    args = calls[0]
    assert args[20] == runs
    assert ws is None or args[23] == ws.data_ptr()
