"""The segmented delayed CGS2 step at the edges of its work split: row tiles of 8, 1,024-dof blocks of a
quarter chunk, odd segment starts (pairs that are 8-byte aligned only), an odd row stride, chunk counts around
the 8 XCDs, and the widths of the coefficient sums. Reference: the definition in extended precision. Rows of V
and u have norm about 1, so a dot product of n terms is off by at most n eps, a coefficient by (J + 2) of
these, and a corrected vector by J coefficients more."""
import numpy as np
import pytest
import torch

from inching_amd.batch import SegOps, Segments

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("sizes,chunk", [([1], 4096), ([3, 1, 2], 4096), ([4095, 4096, 4097], 4096),
                                         ([5001, 9000, 12289], 4096), ([700, 333], 64), ([8192], 1024),
                                         ([20003], 8192)])
@pytest.mark.parametrize("J", [1, 2, 8, 9, 32, 33, 128])
def test_seg_dcgs2_edges(sizes, chunk, J):
    rng = np.random.default_rng(sum(sizes) + J)
    ptr = np.concatenate([[0], np.cumsum(sizes)])
    n, S, i = int(ptr[-1]), len(sizes), J - 1
    V = rng.standard_normal((J, n + 3))
    u = rng.standard_normal(n)
    for s in range(S):
        sl = slice(ptr[s], ptr[s + 1])
        V[:, sl] /= np.sqrt(sizes[s])
        u[sl] /= np.sqrt(sizes[s])
    beta = rng.uniform(0.5, 1.5, S)
    Vd = torch.as_tensor(V, device="cuda")
    ud = torch.as_tensor(u, device="cuda")
    al = torch.zeros(S, dtype=torch.float64, device="cuda")
    bo = torch.zeros_like(al)
    so = SegOps(Segments(ptr, "cuda", chunk=chunk), max(J, 2), "cuda")
    so.dcgs2(Vd[:, :n], J, ud, al, torch.as_tensor(beta, device="cuda") if J > 1 else None, bo)
    Vg, ug, al, bo = Vd.cpu().numpy(), ud.cpu().numpy(), al.cpu().numpy(), bo.cpu().numpy()
    assert np.array_equal(Vg[:i], V[:i]) and np.array_equal(Vg[:, n:], V[:, n:])
    for s in range(S):
        sl = slice(ptr[s], ptr[s + 1])
        Vs, us = V[:, sl].astype(np.longdouble), u[sl].astype(np.longdouble)
        sv, g = Vs @ us, (Vs @ Vs[i])[:i]
        ci = sv[i] - g @ sv[:i]
        cf = np.concatenate([sv[:i] - ci * g, [ci]])
        un, vn = us - cf @ Vs, Vs[i] - g @ Vs[:i]
        scale = max(1.0, float(np.abs(Vs).max()), float(np.abs(cf).max()), float((Vs * Vs).sum(1).max())) ** 4
        tol = 8 * J * (J + 2) * (sizes[s] + J) * EPS * scale
        assert tol < 1e-2 or sizes[s] < 64      # many rows over a few dofs: coefficients are large, the bound loose
        assert np.abs(ug[sl] - un).max() <= tol and np.abs(Vg[i, sl] - vn).max() <= tol
        assert abs(al[s] - (ci - (beta[s] * g[i - 1] if i else 0.0))) <= tol
        assert abs(bo[s] - np.sqrt((un * un).sum())) <= tol * np.sqrt(sizes[s])
