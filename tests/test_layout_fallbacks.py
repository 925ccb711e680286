"""Which failures of a layout's construction let a matrix take its next form, and which reach the caller."""
import threading

import pytest
import torch

from inching_amd import hessian, ops
from inching_amd._lib import InchingError


def _matrix():
    z = torch.zeros(4, 3, dtype=torch.float64)
    return hessian.BlockHessian(z, torch.arange(5), torch.arange(4, dtype=torch.int32), None, None, None, 1.0, 8.0)


LAYOUTS = [("tiles", "Tiles"), ("bsr_tiles", "BsrTiles")]


@pytest.mark.parametrize("method,layout", LAYOUTS)
@pytest.mark.parametrize("error", [InchingError("x", -3, "full"), torch.OutOfMemoryError("full")])
def test_layouts_without_room_are_none(monkeypatch, method, layout, error):
    def refuse(*args, **kw):
        raise error

    A = _matrix()
    monkeypatch.setattr(ops, layout, refuse)
    if layout == "BsrTiles":
        monkeypatch.setattr(refuse, "TILE", 16, raising=False)
    assert getattr(A, method)() is None
    monkeypatch.setattr(ops, layout, None)     # not asked again
    assert getattr(A, method)() is None


@pytest.mark.parametrize("method,layout", LAYOUTS)
@pytest.mark.parametrize("status", [-1, -2, -5])
def test_other_errors_reach_the_caller_each_time(monkeypatch, method, layout, status):
    def fail(*args, **kw):
        raise InchingError("x", status, "broken")

    A = _matrix()
    monkeypatch.setattr(ops, layout, fail)
    if layout == "BsrTiles":
        monkeypatch.setattr(fail, "TILE", 16, raising=False)
    for _ in range(2):
        with pytest.raises(InchingError) as e:
            getattr(A, method)()
        assert e.value.status == status


@pytest.mark.parametrize("method,layout", LAYOUTS)
def test_a_second_thread_does_not_see_a_layout_half_made(monkeypatch, method, layout):
    entered, go = threading.Event(), threading.Event()
    first = threading.get_ident()

    def slow(*args, **kw):
        if threading.get_ident() != first:
            entered.set()
            assert go.wait(30)
        return "layout"

    A = _matrix()
    monkeypatch.setattr(ops, layout, slow)
    if layout == "BsrTiles":
        monkeypatch.setattr(slow, "TILE", 16, raising=False)
    t = threading.Thread(target=getattr(A, method))
    t.start()
    assert entered.wait(30)
    assert getattr(A, method)() == "layout"
    go.set()
    t.join()
    assert getattr(A, method)() == "layout"
