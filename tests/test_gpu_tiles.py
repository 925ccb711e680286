"""Tile form of the matrix-free operator: the layout's pairs equal the neighbour CSR's (open and
periodic, padded tiles, isolated and coincident atoms), one recurrence step equals the oracle's
blocks, and what does not fit falls back to the record form."""
import numpy as np
import pytest
import torch

from helpers import small_globule
from oracle import hessian as OH
from test_gpu_pbc import _dense, _slab

pytestmark = pytest.mark.gpu

SHAPES = [(64, 8), (32, 16), (16, 32)]
CASES = ["globule", "isolated_coincident", "pbc_narrow", "pbc_slab"]


def _matrix(case):
    """Coordinates, box, device pattern and the oracle's dense matrix."""
    from inching_amd import ops
    if case == "globule":
        X, box = small_globule(1003, seed=23), None
    elif case == "isolated_coincident":
        X = small_globule(130, seed=5)
        X = np.concatenate([X, X[:3], [[400.0, 400.0, 60.0 * k] for k in range(9)]])
        box = None
    elif case == "pbc_narrow":       # a pair has several images within the cutoff
        box = (15.0, 15.0)
        X = _slab(90, box, 8.0, seed=3)
    else:
        box = (40.0, 36.0)
        X = _slab(700, box, 12.0, seed=3)
    xyz = torch.as_tensor(X, device="cuda")
    if box is None:
        rp, col, vals = OH.block_hessian(X, 8.0, 1.0)
        D = OH.block_to_scipy(rp, col, vals, len(X)).toarray()
        ip, ix = ops.neighbours(xyz, 8.0)
        return X, box, xyz, ip, ix, None, D
    rp, col, vals, _ = OH.block_hessian_pbc(X, 8.0, 1.0, box)
    ip, ix, im = ops.neighbours_pbc(xyz, 8.0, box, (0.0, 0.0))
    return X, box, xyz, ip, ix, im, _dense(rp, col, vals, len(X))


def _terms(T, X, box, n):
    """Every (atom, neighbour, image) that the layout's lists hold, by walking them as the product does."""
    tile, lanes = T.shape
    atoms = T.atoms.cpu().numpy()
    ulen, ulist = T.ulen.cpu().numpy(), T.ulist.cpu().numpy().view(np.uint32).reshape(T.ntile, -1).astype(np.int64)
    waves = T.waves.cpu().numpy().reshape(-1, 2)
    pairs = T.pairs.cpu().numpy().view(np.uint16).reshape(-1, 64, 8).astype(np.int64)
    per = 64 // lanes
    got = []
    for w, (blk, passes) in enumerate(waves):
        t = w * per // tile
        u = ulist[t, :ulen[t]]
        assert np.all(np.diff(u) > 0)
        for a in range(per):
            place = (w * per + a) % tile
            at = atoms[t * tile + place]
            for b in range((passes + 7) // 8):
                off = pairs[blk + b, a * lanes:(a + 1) * lanes]
                assert np.all(off % 48 == 0)
                real = off[off < 48 * ulen[t]] // 48
                assert np.all(off[off >= 48 * ulen[t]] == 48 * (ulen[t] + place))
                assert at >= 0 or real.size == 0
                got += [(at, atoms[u[r] // 48], u[r] & 15) for r in real]
    return got


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("case", CASES)
def test_tile_layout_and_product(cuda, case, shape):
    from inching_amd import ops
    print("case: tiles %s %s" % (case, shape), flush=True)
    X, box, xyz, ip, ix, im, D = _matrix(case)
    n = len(X)
    T = ops.Tiles(xyz, ip, ix, 8.0 * (shape[0] / 117.0) ** (1 / 3) * 1.6, shape, images=im, box=box)
    atoms = T.atoms.cpu().numpy()
    assert np.array_equal(np.sort(atoms[atoms >= 0]), np.arange(n))
    rp, col = ip.cpu().numpy(), ix.cpu().numpy()
    masks = np.full(len(col), 16) if im is None else im.cpu().numpy().astype(int)
    want = []
    for i in range(n):
        for e in range(rp[i], rp[i + 1]):
            for bit in range(9):
                s = np.zeros(3) if box is None else np.array([(bit // 3 - 1) * box[0], (bit % 3 - 1) * box[1], 0.0])
                if masks[e] >> bit & 1 and np.any(X[col[e]] + s != X[i]):
                    want.append((i, col[e], bit))
    assert sorted(_terms(T, X, box, n)) == sorted(want)
    # one step with every epilogue term: sums of at most a few hundred terms of size |x| each
    rng = np.random.default_rng(4)
    x, z, a0 = (rng.standard_normal(3 * n) for _ in range(3))
    out = 0.3 * (D @ x - 2.0 * x) - z
    dev = lambda v: torch.as_tensor(v, device="cuda")    # noqa: E731
    rin, rz, ro = T.buffers(3)
    acc = torch.empty(3 * T.slots, dtype=torch.float64, device="cuda")
    y = torch.empty_like(acc)
    back = torch.full((3 * n,), float("nan"), dtype=torch.float64, device="cuda")
    ops.rec_pack(T.atoms, dev(a0), ro, acc, 1.0)
    ops.rec_pack(T.atoms, dev(z), rz)
    ops.rec_pack(T.atoms, dev(x), rin)
    T.product(rin, rz, ro, 1.0, s1=0.3, c0=2.0, c2=1.0, acc=acc, mu=0.5, y=y)
    tol = 1e-12 * np.abs(out).max()
    assert torch.equal(ro.view(-1, 6)[:, 3:].reshape(-1), y) and torch.equal(ro.view(-1, 6)[:, :3], T.rec.view(-1, 6)[:, :3])
    ops.rec_unpack(T.atoms, y, back)
    assert np.abs(back.cpu().numpy() - out).max() <= tol
    ops.rec_unpack(T.atoms, acc, back)
    assert np.abs(back.cpu().numpy() - (a0 + 0.5 * out)).max() <= tol
    assert not bool(y.view(-1, 3)[T.atoms < 0].any())
    # the recurrence in one call equals its steps
    mu = np.array([0.2, 0.7, -0.4, 0.1])
    recs = T.buffers(3)
    ops.rec_pack(T.atoms, dev(x), recs[0], acc, mu[0])
    T.chebyshev(recs, mu, 30.0, 29.0, 1.0, acc)
    Ah = (D - 30.0 * np.eye(3 * n)) / 29.0
    t = [x, Ah @ x]
    t += [2.0 * Ah @ t[1] - t[0]]
    t += [2.0 * Ah @ t[2] - t[1]]
    ref = sum(m * v for m, v in zip(mu, t))
    ops.rec_unpack(T.atoms, acc, back)
    assert np.abs(back.cpu().numpy() - ref).max() <= 1e-12 * max(np.abs(v).max() for v in t)


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("case", CASES)
def test_tile_block_product(cuda, case, shape):
    """Several right-hand sides: column counts around the groups of 4 and the 64 of the packing."""
    from inching_amd import ops
    print("case: tile block %s %s" % (case, shape), flush=True)
    X, box, xyz, ip, ix, im, D = _matrix(case)
    T = ops.Tiles(xyz, ip, ix, 8.0 * (shape[0] / 117.0) ** (1 / 3) * 1.6, shape, images=im, box=box)
    rng = np.random.default_rng(7)
    for r in (1, 2, 3, 4, 5, 63, 64, 67):
        V = rng.standard_normal((3 * len(X), r))
        Y = torch.full(V.shape, float("nan"), dtype=torch.float64, device="cuda")
        T.apply(torch.as_tensor(V, device="cuda"), Y, 1.0)
        ref = D @ V
        assert np.abs(Y.cpu().numpy() - ref).max() <= 1e-12 * np.abs(ref).max(), r
    v = torch.as_tensor(V[:, 0].copy(), device="cuda")
    y = torch.empty_like(v)
    T.apply(v, y, 1.0)
    assert np.abs(y.cpu().numpy() - ref[:, 0]).max() <= 1e-12 * np.abs(ref).max()
    with pytest.raises(ValueError):
        T.apply(Y.T, Y.T, 1.0)


def test_periodic_filter_in_slot_order_matches_matrix_order(cuda):
    from inching_amd import chebyshev as CH
    from inching_amd.hessian import build_hessian
    from inching_amd.operator import Operator
    print("case: periodic filter", flush=True)
    box = (40.0, 36.0)
    A = build_hessian(_slab(700, box, 12.0, seed=3), 8.0, precision=(), box=box)
    pol = CH.design_filter(1.0, 3.0, (1.0, 80.0), 5120, 5, 0.7)
    v = torch.randn(A.shape[0], dtype=torch.float64, device="cuda")
    a, b = torch.empty_like(v), torch.empty_like(v)
    op = Operator(A, "mf64", pol=pol)
    assert op.rec is A.tiles() is not None
    op.apply(v, a)
    Operator(A, "mf64", pol=pol, records=False).apply(v, b)
    assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())
    op.apply(v, v)       # in place
    assert torch.equal(v, a)


def test_tiles_fall_back(cuda):
    """Dense rows leave every tile shape (the record form or the matrix's order takes over), and so
    do distances outside the range of the product's float32 seed."""
    from inching_amd import ops
    from inching_amd.hessian import RecordForm, build_hessian
    print("case: tile fallbacks", flush=True)
    X = np.random.default_rng(5).uniform(0.0, 12.0, size=(1500, 3))
    A = build_hessian(X, 30.0, precision=())
    assert A.tiles() is None and A.slot_form() is None
    G = build_hessian(small_globule(2000, seed=21), 18.0, precision=())    # too dense for the clusters too
    assert G.tiles() is None and G.slot_form() is None
    M = build_hessian(small_globule(2000, seed=21), 15.0, precision=())
    assert M.tiles() is None and isinstance(M.slot_form(), RecordForm)
    tiny = build_hessian(small_globule(300, seed=2) * 1e-18, 8e-18, precision=())
    assert tiny.tiles() is None and isinstance(tiny.slot_form(), RecordForm)
    with pytest.raises(ops.InchingError):
        ops.Tiles(A.xyz, A.rowptr, A.col, 5.0, (8, 8))


@pytest.mark.parametrize("columns", [1, 5])
def test_block_product_lays_out_tiles_only_where_they_pay(cuda, columns, monkeypatch):
    """A fresh matrix: below the line the product leaves the tiles out, at it or with tiles at hand it takes them;
    both agree to rounding (124 terms a row)."""
    from inching_amd import hessian
    print("case: block product rule %d" % columns, flush=True)
    rng = np.random.default_rng(3)
    xyz = rng.uniform(0.0, 30.0, (1500, 3))
    X = torch.as_tensor(rng.standard_normal((4500, columns)), device="cuda")
    A = hessian.build_hessian(xyz, 8.0, precision=())
    plain = A.matfree(X)
    assert "_tiles" not in A.__dict__
    monkeypatch.setattr(hessian, "TILE_APPLY_TERMS", A.nnzb * columns + 1)
    A.matfree(X)
    assert "_tiles" not in A.__dict__
    monkeypatch.setattr(hessian, "TILE_APPLY_TERMS", A.nnzb * columns)
    tiled = A.matfree(X)
    assert A.__dict__["_tiles"] is not None
    monkeypatch.setattr(hessian, "TILE_APPLY_TERMS", float("inf"))
    assert torch.equal(A.matfree(X), tiled)
    assert (plain - tiled).abs().max() <= 1e-11 * plain.abs().max()
