"""Launch codes that a caller names: the cluster layout's are refused, or ignored, where there is no such layout."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _pol():
    from types import SimpleNamespace
    return SimpleNamespace(AdjustedCoefficients=np.array([0.3, -0.7, 0.2]), AdjustedDegree=2, cc=40.0, dd=39.0)


def test_cluster_code_without_the_layout_is_refused(cuda):
    """More neighbours than a cluster's list holds, where the tiles would still fit."""
    from inching_amd.hessian import build_hessian
    from inching_amd.operator import Operator
    print("case: code 6001 on 1,340 atoms within one cutoff", flush=True)
    A = build_hessian(np.random.default_rng(3).uniform(0.0, 4.0, (1340, 3)), 8.0, precision=())
    assert A.clusters() is None and A.tiles() is not None
    v = torch.randn(A.shape[0], dtype=torch.float64, device="cuda")
    with pytest.raises(ValueError):
        Operator(A, "mf64", pol=_pol(), lanes=6001).apply(v, torch.empty_like(v))
    Operator(A, "mf64", pol=_pol()).apply(v, torch.empty_like(v))


def test_cluster_code_with_periodic_images_keeps_their_kernel(cuda):
    from inching_amd.hessian import build_hessian
    from inching_amd.operator import Operator
    from test_gpu_pbc import _slab
    print("case: code 6001 with periodic images", flush=True)
    A = build_hessian(_slab(700, (40.0, 36.0), 12.0, seed=3), 8.0, precision=(), box=(40.0, 36.0))
    v = torch.randn(A.shape[0], dtype=torch.float64, device="cuda")
    a, b = torch.empty_like(v), torch.empty_like(v)
    op = Operator(A, "mf64", pol=_pol(), lanes=6001)
    assert op.rec is None
    op.apply(v, a)
    Operator(A, "mf64", pol=_pol()).apply(v, b)
    assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
