"""Products recorded into a graph on a matrix whose layouts no earlier product has made: every replay equals the eager
result, with eager work between the replays."""
import numpy as np
import pytest
import torch

from inching_amd.synth import globule

pytestmark = pytest.mark.gpu


def _matrix():
    from inching_amd.hessian import build_hessian
    return build_hessian(globule(1500, seed=7), 8.0, precision=())


def _replays(graph, x, y, reference):
    """Three replays on new inputs, each against ``reference(x)``; row sums of at most 200 terms in another order."""
    for k in range(3):
        x.copy_(torch.as_tensor(np.random.default_rng(k).standard_normal(tuple(x.shape)), device="cuda"))
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        want = reference(x)
        assert float((y - want).abs().max()) <= 1e-12 * float(want.abs().max())


@pytest.mark.parametrize("lanes", [None, 6001])
def test_capture_of_a_plain_product(cuda, lanes):
    from inching_amd import chebyshev as CH
    from inching_amd.operator import Operator
    print("case: capture of a filtered operator's plain product, lanes %s" % lanes, flush=True)
    A, B = _matrix(), _matrix()
    op = Operator(A, "mf64", pol=CH.design_filter(1.0, 3.0, (1.0, 80.0), 5120, 5, 0.7), lanes=lanes)
    assert ("_clusters" in A.__dict__) == (lanes is not None)
    x = torch.zeros(4500, dtype=torch.float64, device="cuda")
    y = torch.empty_like(x)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        op.spmv(x, y)
    _replays(g, x, y, B.matfree)
    op.spmv(x, y)                 # outside: the layout
    assert op.lanes == 6001 and float((y - B.matfree(x)).abs().max()) <= 1e-12 * float(y.abs().max())


@pytest.mark.parametrize("line", [0.0, float("inf")])
def test_capture_of_a_block_product(cuda, line, monkeypatch):
    from inching_amd import hessian
    print("case: capture of a block product, line %g" % line, flush=True)
    A, B = _matrix(), _matrix()
    monkeypatch.setattr(hessian, "TILE_APPLY_TERMS", line)
    X = torch.zeros(4500, 5, dtype=torch.float64, device="cuda")
    out = torch.empty_like(X)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out.copy_(A.matfree(X))
    assert "_tiles" not in A.__dict__ and "_clusters" not in A.__dict__
    _replays(g, X, out, B.matfree)
    h = torch.cuda.CUDAGraph()
    A.matfree(X)
    with torch.cuda.graph(h):
        out.copy_(A.matfree(X))
    _replays(h, X, out, B.matfree)
