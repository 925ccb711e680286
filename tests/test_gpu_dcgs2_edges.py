"""The delayed CGS2 step over one vector and the multi-dot at the edges of their work splits: chunks of the dot
products, the narrow and the wide update (131,072, 262,144 and 786,432 dofs), row tiles of 1, 2, 4 and 8, the
largest basis whose coefficients one workgroup forms (256 rows) and one beyond it. Reference: the definition in
extended precision. Rows have norm about 1: a dot product of n terms is off by at most n eps times its sum of
magnitudes, a coefficient by (J + 2) of these, a corrected vector by J coefficients more."""
import numpy as np
import pytest
import torch

from inching_amd import ops

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps
CASES = ([(n, J) for n in (300, 1023, 1025, 4099) for J in (1, 2, 3, 5, 8, 9, 33)]
         + [(n, J) for n in (131072, 131073, 262145, 786433, 1100001) for J in (1, 6)]
         + [(2000, 256), (2000, 257)])


@pytest.mark.parametrize("n,J", CASES)
@pytest.mark.parametrize("last", [False, True])
def test_dcgs2_edges(n, J, last):
    rng = np.random.default_rng(n + J)
    i = J - 1
    V = rng.standard_normal((J + 1, n + 1)) / np.sqrt(n)
    u = rng.standard_normal(n) / np.sqrt(n)
    beta = rng.uniform(0.5, 1.5, J)
    Vd, ud, bd = (torch.as_tensor(x, device="cuda") for x in (V, u, beta))
    al = torch.zeros(J, dtype=torch.float64, device="cuda")
    bo = torch.zeros(1, dtype=torch.float64, device="cuda")
    Vv = Vd[:, :n]
    ops.dcgs2_step(Vv, J, ud, al, bd, bo, vnext=None if last else Vv[J])
    Vg, ug, a, bo = Vd.cpu().numpy(), ud.cpu().numpy(), al.cpu().numpy()[i], bo.item()
    assert np.array_equal(Vg[:i], V[:i]) and np.array_equal(Vg[:, n:], V[:, n:])
    Vs, us = V[:J, :n].astype(np.longdouble), u.astype(np.longdouble)
    sv, g = Vs @ us, (Vs @ Vs[i])[:i]
    ci = sv[i] - g @ sv[:i]
    cf = np.concatenate([sv[:i] - ci * g, [ci]])
    un, vn = us - cf @ Vs, Vs[i] - g @ Vs[:i]
    tol = 8 * J * (J + 2) * (n + J) * EPS * 1.5 ** 4      # norms and coefficients stay under 1.5 here
    assert np.abs(ug - un).max() <= tol and np.abs(Vg[i, :n] - vn).max() <= tol
    assert abs(a - (ci - (beta[i - 1] * g[i - 1] if i else 0.0))) <= tol
    nrm = np.sqrt((un * un).sum())
    assert abs(bo - nrm) <= tol * np.sqrt(n)
    if last:
        assert np.array_equal(Vg[J], V[J])
    else:
        assert np.abs(Vg[J, :n] - ug / bo).max() <= 4 * EPS * np.abs(ug / bo).max()


@pytest.mark.parametrize("n", [1, 255, 257, 5003])
@pytest.mark.parametrize("J", [1, 2, 4, 5, 8, 9, 12])
def test_multidot_tiles(n, J):
    rng = np.random.default_rng(n + J)
    V, u = rng.standard_normal((J, n + 2)), rng.standard_normal(n)
    h = torch.empty(J, dtype=torch.float64, device="cuda")
    ops.multidot(torch.as_tensor(V, device="cuda")[:, :n], J, torch.as_tensor(u, device="cuda"), h,
                 ops.Workspace(J, "cuda"))
    ref = V[:, :n].astype(np.longdouble) @ u
    assert np.all(np.abs(h.cpu().numpy() - ref) <= n * EPS * (np.abs(V[:, :n]) @ np.abs(u)))
