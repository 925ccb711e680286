"""Kernels of the warm-start network at odd widths and row counts (edges of the 32-row tiles, the
4-wide output groups and the 16 x 16 weight-gradient grid): dense forward and backward and the
neighbour mean and its adjoint against float64, and the fused layer against their composition,
bit for bit."""
import numpy as np
import pytest
import torch

from helpers import small_globule

pytestmark = pytest.mark.gpu

WIDTHS = [(16, 64), (64, 64), (64, 96), (96, 96), (5, 7), (33, 18), (1, 1)]
EPS32 = 2.0 ** -24


def _call(name, *args):
    from inching_amd import ops
    from inching_amd._lib import call
    call(name, *[ops.P(a) if a is None or isinstance(a, torch.Tensor) else a for a in args], ops.stream_ptr())


def _f32(*shape):
    return torch.full(shape, float("nan"), dtype=torch.float32, device="cuda")


def _dense_bwd(h, W, dY):
    from inching_amd._lib import lib
    (N, Din), Dout = h.shape, W.shape[1]
    work = _f32(int(lib().inch_gnn_work_size(Din, Dout)))
    dX, dW, db = _f32(N, Din), _f32(Din, Dout), _f32(Dout)
    _call("inch_gnn_dense_bwd", N, Din, Dout, h, W, dY, dX, dW, db, work)
    return dX, dW, db


@pytest.mark.parametrize("N", [1, 31, 33, 10001])
@pytest.mark.parametrize("Din,Dout", WIDTHS)
def test_dense_kernels_float64(cuda, Din, Dout, N):
    print("case: dense %d x %d, %d rows" % (Din, Dout, N), flush=True)
    g = torch.Generator(device="cuda")
    g.manual_seed(N + Din)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")    # noqa: E731
    X, W, b, dY = rnd(N, Din).half(), rnd(Din, Dout).half(), rnd(Dout), rnd(N, Dout)
    pre, y, y16 = _f32(N, Dout), _f32(N, Dout), torch.empty((N, Dout), dtype=torch.float16, device="cuda")
    _call("inch_gnn_dense_fwd", N, Din, Dout, X, W, b, 1, pre, y16, y)
    ref = X.double() @ W.double() + b.double()
    # a chain of k roundings of partial sums of at most the sum of the magnitudes
    size = X.double().abs() @ W.double().abs() + b.double().abs()
    assert bool(((pre - ref).abs() <= (Din + 1) * EPS32 * size).all())
    assert torch.equal(y, pre.clamp_min(0.0)) and torch.equal(y16, y.half())
    dX, dW, db = _dense_bwd(X, W, dY)
    for got, a, c, k in ((dX, dY.double(), W.double().T, Dout), (dW, X.double().T, dY.double(), N)):
        assert bool(((got - a @ c).abs() <= (k + 1) * EPS32 * (a.abs() @ c.abs())).all())
    assert bool(((db - dY.double().sum(0)).abs() <= (N + 1) * EPS32 * dY.double().abs().sum(0)).all())


@pytest.mark.parametrize("D", [1, 3, 16, 64, 96, 300])
def test_aggregate_float64(cuda, D):
    from inching_amd import ops
    print("case: aggregate D=%d" % D, flush=True)
    X = np.concatenate([small_globule(1001, seed=9), [[300.0, 0.0, 0.0]]])     # an atom without neighbours
    ip, ix = ops.neighbours(torch.as_tensor(X, device="cuda"), 8.0)
    n = len(X)
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), ip[1:] - ip[:-1])
    M = torch.zeros((n, n), dtype=torch.float64, device="cuda")
    M[rows, ix.long()] = 1.0
    M.fill_diagonal_(0.0)
    deg = M.sum(1).clamp_min(1.0)
    g = torch.Generator(device="cuda")
    g.manual_seed(D)
    F = torch.randn((n, D), generator=g, device="cuda")
    k = int(deg.max())
    for mode, A in ((0, M / deg[:, None]), (1, M / deg[None, :])):
        for x, xdt in ((F, 0), (F.half(), 2)):
            y = _f32(n, D)
            _call("inch_gnn_aggregate", n, D, ip, ix, x, xdt, y, 0, mode)
            assert bool(((y - A @ x.double()).abs() <= (k + 2) * EPS32 * (A @ x.double().abs())).all())
            if xdt == 2:
                y16 = torch.empty((n, D), dtype=torch.float16, device="cuda")
                _call("inch_gnn_aggregate", n, D, ip, ix, x, 2, y16, 2, mode)
                assert torch.equal(y16, y.half())


@pytest.mark.parametrize("Din,Dout", WIDTHS)
def test_fused_layer_equals_its_parts(cuda, Din, Dout):
    from inching_amd import ops
    from inching_amd.warmstart import GraphLayer, _Graph
    print("case: layer %d x %d" % (Din, Dout), flush=True)
    ip, ix = ops.neighbours(torch.as_tensor(small_globule(1001, seed=9), device="cuda"), 8.0)
    N = 1001
    g = torch.Generator(device="cuda")
    g.manual_seed(Din * 100 + Dout)
    rnd = lambda *s: torch.randn(s, generator=g, device="cuda")    # noqa: E731
    h, Ws, Wn, b = (t.requires_grad_() for t in (rnd(N, Din), rnd(Din, Dout), rnd(Din, Dout), rnd(Dout)))
    dout = rnd(N, Dout)
    out = GraphLayer.apply(h, Ws, Wn, b, _Graph(ip, ix))
    got = torch.autograd.grad(out, (h, Ws, Wn, b), dout)
    with torch.no_grad():
        h16, ws, wn = h.half(), Ws.half(), Wn.half()
        agg = torch.empty_like(h16)
        _call("inch_gnn_aggregate", N, Din, ip, ix, h16, 2, agg, 2, 0)
        a, c = _f32(N, Dout), _f32(N, Dout)
        _call("inch_gnn_dense_fwd", N, Din, Dout, h16, ws, b, 0, None, None, a)
        _call("inch_gnn_dense_fwd", N, Din, Dout, agg, wn, None, 0, None, None, c)
        pre = a + c
        assert torch.equal(out, torch.relu(pre))
        dp = torch.where(pre > 0, dout, torch.zeros_like(dout))
        dh, dWs, db = _dense_bwd(h16, ws, dp)
        dagg, dWn, _ = _dense_bwd(agg, wn, dp)
        back = _f32(N, Din)
        _call("inch_gnn_aggregate", N, Din, ip, ix, dagg, 0, back, 0, 1)
        for x, y in zip(got, (dh + back, dWs, dWn, db)):
            assert torch.equal(x, y)


@pytest.mark.parametrize("n", [1, 255, 257, 4096 * 256 + 3])
def test_relu_backward(cuda, n):
    from inching_amd import ops
    print("case: relu backward %d" % n, flush=True)
    pre, dy = torch.randn(n, device="cuda"), torch.randn(n, device="cuda")
    pre[0] = 0.0
    out = torch.full((n,), float("nan"), device="cuda")
    ops.call("inch_gnn_relu_bwd", n, ops.P(pre), ops.P(dy), ops.P(out), ops.stream_ptr())
    assert torch.equal(out, torch.where(pre > 0, dy, torch.zeros_like(dy)))
