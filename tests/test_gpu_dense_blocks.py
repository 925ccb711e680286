"""Dense row-block kernels at the edges of their column tiles: the Gram product with 16, 32 and 64
columns per workgroup (one block of rows staged once against itself), and the projection out -= W^T V
with its few-row form (at most 8 rows) and the matrix-core form. Both against numpy in extended
precision; a sum of n products in any order is off by at most n eps times the sum of magnitudes."""
import numpy as np
import pytest
import torch

from inching_amd import ops

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


def _rows(rng, k, n, pad=0):
    base = rng.standard_normal((k, n + pad))
    dev = torch.as_tensor(base, device="cuda")
    return base[:, :n], dev[:, :n]


@pytest.mark.parametrize("n", [1, 31, 33, 2500])
@pytest.mark.parametrize("k1,k2", [(1, 1), (3, 16), (64, 17), (65, 32), (20, 33), (64, 64), (5, 65), (33, 130)])
def test_gram_tiles(n, k1, k2):
    rng = np.random.default_rng(1000 * k1 + k2 + n)
    X, dX = _rows(rng, k1, n, 3)
    Y, dY = _rows(rng, k2, n)
    G = ops.gram(dX, dY).cpu().numpy()
    ref = X.astype(np.longdouble) @ Y.T.astype(np.longdouble)
    assert np.all(np.abs(G - ref) <= n * EPS * (np.abs(X) @ np.abs(Y).T) + 1e-300)


@pytest.mark.parametrize("k", [1, 16, 17, 32, 33, 64, 65])
def test_gram_with_itself(k):
    rng = np.random.default_rng(k)
    n = 1500
    X, dX = _rows(rng, k, n, 5)
    bound = n * EPS * (np.abs(X) @ np.abs(X).T)
    ref = X.astype(np.longdouble) @ X.T.astype(np.longdouble)
    assert np.all(np.abs(ops.gram(dX, dX).cpu().numpy() - ref) <= bound)
    # fewer rows of the same block on one side: two operands at one address
    assert np.all(np.abs(ops.gram(dX, dX[:(k + 1) // 2]).cpu().numpy() - ref[:, :(k + 1) // 2])
                  <= bound[:, :(k + 1) // 2])


@pytest.mark.parametrize("n", [1, 255, 257, 1100])
@pytest.mark.parametrize("m", [1, 6, 8, 9, 64, 65, 130])
@pytest.mark.parametrize("k", [1, 16, 17, 33, 65])
def test_rr_project(n, m, k):
    rng = np.random.default_rng(100 * m + k + n)
    V, dV = _rows(rng, m, n, 7)
    W = rng.standard_normal((m, k))
    out = rng.standard_normal((k, n))
    dout = torch.as_tensor(out, device="cuda")
    ops.rr_project(dV, m, torch.as_tensor(W, device="cuda"), dout)
    ref = out.astype(np.longdouble) - W.T.astype(np.longdouble) @ V.astype(np.longdouble)
    assert np.all(np.abs(dout.cpu().numpy() - ref) <= (m + 1) * EPS * (np.abs(out) + np.abs(W).T @ np.abs(V)))
