"""BlockHessian.matfree's choice between the tile form and the cluster layout."""
import pytest
import torch

from inching_amd.synth import globule

pytestmark = pytest.mark.gpu


def _matrix(n=1500, seed=3):
    from inching_amd.hessian import build_hessian
    return build_hessian(globule(n, seed=seed), 8.0, precision=())


@pytest.mark.parametrize("columns", [1, 7])
def test_block_product_does_not_depend_on_earlier_calls(cuda, columns):
    from inching_amd import chebyshev as CH
    from inching_amd.operator import Operator
    print("case: matfree before and after an operator, %d columns" % columns, flush=True)
    A = _matrix()
    X = torch.randn(4500, columns, dtype=torch.float64, device="cuda")
    first = A.matfree(X)
    Operator(A, "mf64", pol=CH.design_filter(1.0, 3.0, (1.0, 80.0), 5120, 5, 0.7))
    assert A.tiles() is not None
    assert torch.equal(A.matfree(X), first)


@pytest.mark.parametrize("shape", [(1500, 3), (4500,), (1500, 3, 2), (4500, 2, 2), (1500, 6)])
def test_block_product_takes_every_shape_on_both_forms(cuda, shape, monkeypatch):
    """Shapes of 3 n x r values: the tile form takes what the cluster layout takes. Row sums of at most 200 terms."""
    from inching_amd import hessian
    print("case: matfree %s" % (shape,), flush=True)
    A = _matrix()
    X = torch.randn(shape, dtype=torch.float64, device="cuda")
    want = A.matfree(X)
    assert "_tiles" not in A.__dict__
    monkeypatch.setattr(hessian, "TILE_APPLY_TERMS", 0)
    got = A.matfree(X)
    assert A.tiles() is not None and got.shape == want.shape
    assert float((got - want).abs().max()) <= 1e-12 * float(want.abs().max())


def test_block_product_refuses_wrong_sizes_on_both_forms(cuda, monkeypatch):
    from inching_amd import hessian
    print("case: matfree of wrong sizes", flush=True)
    A = _matrix()
    bad = torch.randn(4501, dtype=torch.float64, device="cuda")
    for line in (float("inf"), 0):
        monkeypatch.setattr(hessian, "TILE_APPLY_TERMS", line)
        with pytest.raises((ValueError, RuntimeError)):
            A.matfree(bad)
        with pytest.raises((ValueError, RuntimeError)):
            A.matfree(torch.randn(4500, 2, device="cuda"))
        with pytest.raises((ValueError, RuntimeError)):
            A.matfree(torch.empty(4500, 0, dtype=torch.float64, device="cuda"))


def test_block_product_workspace_is_bounded(cuda):
    """The tile form packs 64 columns at a time: its workspace does not grow past them, and columns around the passes
    are those of the narrower products."""
    from inching_amd._lib import call
    print("case: workspace of a wide block", flush=True)
    A = _matrix()
    T = A.tiles()
    size = [int(call("inch_anm_tile_apply_work_size", T.ntile, T.shape[0], r)) for r in (1, 4, 5, 64, 65, 1000)]
    assert size == [12 * T.slots * g for g in (1, 1, 2, 16, 16, 16)]
    X = torch.randn(4500, 197, dtype=torch.float64, device="cuda")
    Y = torch.full_like(X, float("nan"))
    T.apply(X, Y, 1.0)
    for c0, c1 in ((0, 64), (64, 128), (128, 192), (192, 197), (60, 70)):
        part = torch.empty(4500, c1 - c0, dtype=torch.float64, device="cuda")
        T.apply(X[:, c0:c1].contiguous(), part, 1.0)
        assert torch.equal(Y[:, c0:c1], part)


def test_block_product_without_room_for_its_workspace(cuda, monkeypatch):
    from inching_amd import hessian, ops
    print("case: no room for the packed columns", flush=True)
    A = _matrix()
    X = torch.randn(4500, 5, dtype=torch.float64, device="cuda")
    want = A.matfree(X)
    monkeypatch.setattr(hessian, "TILE_APPLY_TERMS", 0)

    def full(*args):
        raise torch.OutOfMemoryError("no room")

    assert A.tiles() is not None
    monkeypatch.setattr(ops, "_scratch", full)
    assert torch.equal(A.matfree(X), want)


def test_solver_keeps_to_one_layout(cuda):
    """A filtered matrix-free solve counts, filters and checks on the tiles, without a second layout for its blocks."""
    from inching_amd.hessian import rigid_body_basis
    from inching_amd.pipeline import lowest_modes
    print("case: layouts of a solve", flush=True)
    A = _matrix(900)
    r = lowest_modes(A, 8, Q=rigid_body_basis(A.xyz), precision="mf64")
    assert r.converged and A.tiles() is not None and "_clusters" not in A.__dict__
