"""BlockHessian.matfree's choice between the tile form and the cluster layout."""
import pytest
import torch

from helpers import small_globule

pytestmark = pytest.mark.gpu


def _matrix(n=1500, seed=3):
    from inching_amd.hessian import build_hessian
    return build_hessian(small_globule(n, seed=seed), 8.0, precision=())


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
