"""The Hotelling term in two launches (row counts around its tiles, plain and with the unpacking of slot order) and
the three-term Lanczos step (vectors shorter and longer than one grid of blocks, records), against extended
precision. A dot product of n terms is off by at most n eps times the sum of magnitudes."""
import numpy as np
import pytest
import torch

from inching_amd import ops

pytestmark = pytest.mark.gpu

EPS = np.finfo(np.float64).eps


@pytest.mark.parametrize("n", [3, 255, 768, 30003, 600000])
@pytest.mark.parametrize("m", [1, 4, 5, 8, 9, 16])
@pytest.mark.parametrize("slots", [False, True])
def test_shift_apply(n, m, slots):
    rng = np.random.default_rng(n + m)
    Q, v, u0 = rng.standard_normal((m, n)) / np.sqrt(n), rng.standard_normal(n), rng.standard_normal(n)
    Qd, vd, u = (torch.as_tensor(x, device="cuda") for x in (Q, v, u0))
    ws = ops.Workspace(m, "cuda")
    if slots:
        atoms = np.full(n // 3 + 5, -1, dtype=np.int32)
        atoms[rng.permutation(atoms.size)[:n // 3]] = rng.permutation(n // 3)
        acc = rng.standard_normal((atoms.size, 3))
        for at, row in zip(atoms, acc):
            if at >= 0:
                u0[3 * at:3 * at + 3] = row
        u.fill_(float("nan"))
        ops.shift_apply(Qd, vd, -40.0, u, ws, atoms=torch.as_tensor(atoms, device="cuda"),
                        acc=torch.as_tensor(acc, device="cuda"))
    else:
        ops.shift_apply(Qd, vd, -40.0, u, ws)
    L = np.longdouble
    h = Q.astype(L) @ v
    ref = u0 + 40.0 * (Q.T.astype(L) @ h)
    herr = n * EPS * (np.abs(Q) @ np.abs(v))
    tol = (m + 4) * EPS * (np.abs(u0) + 40.0 * np.abs(Q).T @ np.abs(h).astype(float)) + 40.0 * np.abs(Q).T @ herr
    assert np.all(np.abs(u.cpu().numpy() - ref) <= tol)


def test_shift_apply_refusals():
    Q = torch.zeros((17, 9), dtype=torch.float64, device="cuda")
    v = torch.zeros(9, dtype=torch.float64, device="cuda")
    with pytest.raises(ValueError):
        ops.shift_apply(Q, v, 1.0, torch.zeros_like(v), ops.Workspace(17, "cuda"))
    with pytest.raises(ops.InchingError):
        ops.shift_apply(Q[:2], v, 1.0, v, ops.Workspace(2, "cuda"))


@pytest.mark.parametrize("n", [3, 254 * 3, 1025 * 3, 150000])
@pytest.mark.parametrize("records", [False, True])
def test_lanczos3_step(n, records):
    rng = np.random.default_rng(n)
    v, vp, f0 = (rng.standard_normal(n) / np.sqrt(n) for _ in range(3))
    beta = 0.7
    vd, vpd, fd = (torch.as_tensor(x, device="cuda") for x in (v, vp, f0))
    out = torch.tensor([0.0, beta, 0.0], dtype=torch.float64, device="cuda")
    step = ops.Lanczos3("cuda")
    step.update(vd, fd, out[0:1], v_prev=vpd, beta=out[1:2])
    w = torch.empty_like(vd)
    rec = torch.full((2 * n,), 5.0, dtype=torch.float64, device="cuda") if records else None
    step.scale(fd, out[2:3], w, rec=rec)
    L = np.longdouble
    f = f0.astype(L) - beta * vp.astype(L)
    alpha = v.astype(L) @ f
    f = f - alpha * v
    nrm = np.sqrt((f * f).sum())
    tol = 16 * n * EPS                      # norms are near 1
    assert abs(out[0].item() - alpha) <= tol and abs(out[2].item() - nrm) <= tol
    assert np.abs(fd.cpu().numpy() - f).max() <= tol and np.abs(w.cpu().numpy() - f / nrm).max() <= tol / nrm ** 2
    if records:
        r = rec.view(-1, 6)
        assert torch.equal(r[:, 3:].reshape(-1), w) and bool((r[:, :3] == 5.0).all())
    fd.copy_(torch.as_tensor(f0))
    step.update(vd, fd, out[0:1])
    assert abs(out[0].item() - v.astype(L) @ f0) <= tol


@pytest.mark.parametrize("pol", [False, True])
def test_hotelling_term_either_way(pol, monkeypatch):
    """Operator.apply below and above the line of the two-launch form: the same to rounding."""
    from inching_amd import chebyshev, hessian
    from inching_amd.operator import Operator
    rng = np.random.default_rng(11)
    A = hessian.build_hessian(rng.uniform(0.0, 30.0, (1500, 3)), 8.0, precision=())
    Q = torch.linalg.qr(torch.as_tensor(rng.standard_normal((4500, 6)), device="cuda"))[0].T.contiguous()
    design = chebyshev.design_filter(1.0, 3.0, (1.0, 80.0), 5120, 5, 0.7) if pol else None
    op = Operator(A, "mf64", pol=design, Q=Q, shift=-40.0)
    v = torch.as_tensor(rng.standard_normal(4500), device="cuda")
    a, b = torch.empty_like(v), torch.empty_like(v)
    op.apply(v, a)
    monkeypatch.setattr(ops, "SHIFT_MAX_DOF", 4499)
    op.apply(v, b)
    h = Q.abs() @ v.abs()
    assert ((a - b).abs() <= 1e-13 * (a.abs().max() + 40.0 * (Q.abs().T @ h))).all()
