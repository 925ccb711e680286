"""The stored-block product on tiles of rows against the plain product and a float64 dense reference: sizes around
a tile's 16 rows and the lanes' passes of 64 blocks, scattered and clustered atoms, both types, the fused epilogue,
periodic images, empty rows, and the refusals. Row sums of m terms are off by at most (m + 4) eps of the sum of
magnitudes in either order."""
import numpy as np
import pytest
import torch

from inching_amd import hessian, ops
from inching_amd.autotune import BSR_TILE, bsr_launch

pytestmark = pytest.mark.gpu

RC = 8.0


def _matrix(n, seed, density=0.05):
    rng = np.random.default_rng(seed)
    side = (n / density) ** (1.0 / 3.0)
    xyz = rng.uniform(0.0, side, (n, 3))
    return hessian.build_hessian(xyz, RC, plus_i=1.0, precision=("f32", "f64"))


def _dense_abs(A, vals, xa, xs):
    """(sum, sum of magnitudes) of every row's products in float64."""
    rowptr, col = A.rowptr.cpu().numpy(), A.col.cpu().numpy()
    v = vals.cpu().numpy().astype(np.float64).reshape(-1, 3, 3)
    X, S = xa.reshape(-1, 3), xs.reshape(-1, 3)
    y, m = np.zeros_like(X), np.zeros_like(X)
    rows = np.repeat(np.arange(rowptr.size - 1), np.diff(rowptr))
    np.add.at(y, rows, np.einsum("bij,bj->bi", v, X[col]))
    np.add.at(m, rows, np.einsum("bij,bj->bi", np.abs(v), S[col]))
    return y.ravel(), m.ravel()


@pytest.mark.parametrize("n,density", [(2, 0.05), (15, 0.05), (16, 0.01), (17, 0.2), (300, 0.06), (1500, 0.001),
                                       (4001, 0.1)])
@pytest.mark.parametrize("precision", ["f32", "f64"])
def test_tile_product(n, density, precision):
    A = _matrix(n, n, density)
    T = A.bsr_tiles()
    assert T is not None
    vals = A.vals(precision)
    dt = torch.float32 if precision == "f32" else torch.float64
    eps = np.finfo(np.float32 if precision == "f32" else np.float64).eps
    g = np.random.default_rng(n)
    x, z, acc = (torch.as_tensor(g.standard_normal(3 * n), dtype=dt, device="cuda") for _ in range(3))
    kw = dict(s1=0.7, c0=1.3, z=z, c2=0.4, mu=0.3)
    y, acc2 = torch.empty_like(x), acc.clone()
    ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, vals, x, y, acc=acc2, lanes=T.LANES, col16=T, **kw)
    xh, zh = x.cpu().numpy().astype(np.float64), z.cpu().numpy().astype(np.float64)
    s, m = _dense_abs(A, vals, xh, np.abs(xh))
    ref = 0.7 * (s - 1.3 * xh) - 0.4 * zh
    mag = 0.7 * (m + 1.3 * np.abs(xh)) + 0.4 * np.abs(zh)
    longest = int(np.diff(A.rowptr.cpu().numpy()).max()) * 3
    tol = (longest + 8) * eps
    assert np.all(np.abs(y.cpu().numpy() - ref) <= tol * mag)
    ah = acc.cpu().numpy().astype(np.float64)
    assert np.all(np.abs(acc2.cpu().numpy() - (ah + 0.3 * ref)) <= tol * (np.abs(ah) + 0.3 * mag))
    # every option off, mixed vector type, and a Hotelling term
    y2, y3 = torch.empty_like(x), torch.empty_like(x)
    Q = torch.as_tensor(g.standard_normal((2, 3 * n)), device="cuda")
    h = torch.tensor([0.5, -2.0], dtype=torch.float64, device="cuda")
    ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, vals, x, y2, Q=Q, qcoef=h, lanes=T.LANES, col16=T)
    ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, vals, x, y3, Q=Q, qcoef=h, lanes=32)
    qmag = (np.abs(Q.cpu().numpy()) * np.abs(h.cpu().numpy())[:, None]).sum(0)
    assert np.all(np.abs((y2 - y3).double().cpu().numpy()) <= 2 * tol * (m + qmag))
    if precision == "f32":
        xd, yd = x.double(), torch.empty(3 * n, dtype=torch.float64, device="cuda")
        ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, vals, xd, yd, lanes=T.LANES, col16=T)
        assert np.all(np.abs(yd.cpu().numpy() - s) <= tol * m)


def test_tile_lists():
    """Every tile lists exactly its rows' columns, ascending; every row stands in one place."""
    A = _matrix(777, 5)
    T = A.bsr_tiles()
    slots = T.slots.cpu().numpy().reshape(T.ntile, T.TILE, 4)
    ulen, ulist = T.ulen.cpu().numpy(), T.ulist.cpu().numpy().reshape(T.ntile, T.stride)
    uidx = T.uidx.cpu().numpy().view(np.uint16)
    rowptr, col = A.rowptr.cpu().numpy(), A.col.cpu().numpy()
    assert np.array_equal(np.sort(slots[..., 0][slots[..., 0] >= 0]), np.arange(777))
    for t in range(T.ntile):
        rows = slots[t][slots[t, :, 0] >= 0]
        cols = np.unique(np.concatenate([col[rowptr[r[0]]:rowptr[r[0] + 1]] for r in rows]))
        assert np.array_equal(ulist[t, :ulen[t]], cols)
        for r in rows:
            b0, b1 = rowptr[r[0]], rowptr[r[0] + 1]
            assert r[1] == b1 - b0 and r[2] == b0 and r[3] == 0
            assert np.array_equal(cols[uidx[b0:b1]], col[b0:b1])


def test_tile_empty_rows_and_refusals():
    """Rows without blocks (also the last one) give the epilogue alone; a column span beyond the
    bits of a tile is refused, and a matrix that has no tiles takes another shape."""
    n = 40
    A = _matrix(n, 9, 0.02)
    rowptr, col = A.rowptr.clone(), A.col
    keep = torch.ones(n, dtype=torch.bool, device="cuda")
    keep[[3, 20, n - 1]] = False
    cnt = torch.where(keep, rowptr.diff(), torch.zeros_like(rowptr[1:]))
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), rowptr.diff())
    sel = keep[rows]
    col2, vals2 = col[sel].contiguous(), A.vals64.reshape(-1, 9)[sel].contiguous()
    rp2 = torch.cat([torch.zeros(1, dtype=rowptr.dtype, device="cuda"), cnt.cumsum(0)]).to(rowptr.dtype)
    T = ops.BsrTiles(A.xyz, rp2, col2, 5.0)
    x = torch.randn(3 * n, dtype=torch.float64, device="cuda")
    y, y2 = torch.empty_like(x), torch.empty_like(x)
    ops.bsr_spmv(n, rp2, col2, vals2, x, y, s1=2.0, c0=1.0, lanes=T.LANES, col16=T)
    ops.bsr_spmv(n, rp2, col2, vals2, x, y2, s1=2.0, c0=1.0, lanes=16)
    assert torch.allclose(y, y2, rtol=1e-12, atol=1e-12 * float(y2.abs().max()))
    assert torch.equal(y.view(n, 3)[~keep], (-2.0 * x).view(n, 3)[~keep])
    with pytest.raises(ValueError):
        ops.bsr_spmv(n, A.rowptr, A.col, A.vals64, x, y, lanes=T.LANES, col16=T)
    m = 300000     # one row of each tile names both ends of the numbering
    rp = torch.arange(0, 2 * m + 1, 2, dtype=torch.int64, device="cuda")
    far = torch.tensor([0, m - 1], dtype=torch.int32, device="cuda").repeat(m)
    xyz = torch.rand((m, 3), dtype=torch.float64, device="cuda") * 170.0
    with pytest.raises(ops.InchingError):
        ops.BsrTiles(xyz, rp, far, 6.0)
    A._bsr_tiles = None
    lanes, c16 = bsr_launch(A, BSR_TILE)
    assert not isinstance(c16, ops.BsrTiles) and lanes in (32, 1032)


def test_tile_periodic():
    rng = np.random.default_rng(2)
    box = (30.0, 32.0)
    xyz = np.column_stack([rng.uniform(0, box[0], 1500), rng.uniform(0, box[1], 1500), rng.uniform(0, 25.0, 1500)])
    A = hessian.build_hessian(xyz, RC, plus_i=1.0, precision=("f64",), box=box)
    T = A.bsr_tiles()
    assert T is not None
    x = torch.randn(4500, dtype=torch.float64, device="cuda")
    y, y2 = torch.empty_like(x), torch.empty_like(x)
    ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, A.vals64, x, y, lanes=T.LANES, col16=T)
    ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, A.vals64, x, y2, lanes=16)
    assert torch.allclose(y, y2, rtol=1e-12, atol=1e-12 * float(y2.abs().max()))


def test_tile_lists_on_another_stream():
    """Lists laid out on one stream are whole for a product on another without a wait in between."""
    A = _matrix(3000, 4)
    x = torch.randn(9000, dtype=torch.float64, device="cuda")
    y, y2 = torch.empty_like(x), torch.empty_like(x)
    ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, A.vals64, x, y2, lanes=16)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        T = A.bsr_tiles()
    with torch.cuda.stream(s2):
        ops.bsr_spmv(A.n_atoms, A.rowptr, A.col, A.vals64, x, y, lanes=T.LANES, col16=T)
    torch.cuda.synchronize()
    assert torch.allclose(y, y2, rtol=1e-12, atol=1e-12 * float(y2.abs().max()))
