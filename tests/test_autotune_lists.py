"""The tuner keeps the lists of a launch shape only where that shape is taken, or where they were there before."""
import pytest
import torch

from inching_amd import autotune, hessian, ops


class _Tiles:
    TILE, LANES = 16, 32

    def __init__(self, *args):
        pass


@pytest.mark.parametrize("there", [False, True])
@pytest.mark.parametrize("wins", [False, True])
def test_rejected_row_tiles_are_given_back(monkeypatch, wins, there):
    z = torch.zeros(4, 3, dtype=torch.float64)
    A = hessian.BlockHessian(z, torch.arange(5), torch.arange(4, dtype=torch.int32), None, torch.zeros(36), None, 1.0, 8.0)
    A._col16 = None
    monkeypatch.setattr(ops, "BsrTiles", _Tiles)
    if there:
        A.bsr_tiles()
    monkeypatch.setattr(autotune, "_load", lambda: None)
    monkeypatch.setattr(autotune, "_save", lambda: None)
    monkeypatch.setattr(autotune, "_cache", {})
    ms = iter([1.0] * len(autotune.BSR_LANES) + [0.5 if wins else 2.0])
    monkeypatch.setattr(autotune, "_time", lambda fn, reps: next(ms))
    best = autotune.best_config(A, "f32")
    assert (best == autotune.BSR_TILE) == wins
    assert ("_bsr_tiles" in A.__dict__) == (wins or there)
