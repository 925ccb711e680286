"""What the tile form's construction refuses, and what it takes at its limits."""
import numpy as np
import pytest
import torch

from inching_amd.synth import globule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("times", [1, 2, 11, 12, 60])
def test_tile_rows_with_repeated_columns(cuda, times):
    """A repeated column counts as often as it is listed, up to the 1,349 terms of a row that a tile of 16 atoms has
    places for (119 others x 11 = 1,309); longer rows are refused."""
    from inching_amd import ops
    print("case: columns repeated %d times" % times, flush=True)
    n = 120
    xyz = torch.as_tensor(globule(n, seed=2), device="cuda")
    rows = [np.repeat(np.arange(n), times) if i % 7 == 0 else np.arange(n) for i in range(n)]
    ip = torch.as_tensor(np.concatenate([[0], np.cumsum([len(r) for r in rows])]), device="cuda")
    ix = torch.as_tensor(np.concatenate(rows).astype(np.int32), device="cuda")
    if times > 11:
        with pytest.raises(ops.InchingError) as e:
            ops.Tiles(xyz, ip, ix, 6.0, (16, 32))
        assert e.value.status == -3
        return
    T = ops.Tiles(xyz, ip, ix, 6.0, (16, 32))
    x = torch.randn(3 * n, dtype=torch.float64, device="cuda")
    y, want = torch.empty_like(x), torch.empty_like(x)
    T.apply(x, y, 1.0)
    ops.matfree_apply(xyz, ip, ix, 1.0, x, want)
    # row sums of at most 1,309 terms
    assert float((y - want).abs().max()) <= 1e-11 * float(want.abs().max())


@pytest.mark.parametrize("shape", [(64, 8), (32, 16), (16, 32)])
@pytest.mark.parametrize("value", [float("inf"), float("-inf"), float("nan"), 1e300])
def test_tile_entries_that_are_not_finite(cuda, shape, value):
    """An entry that is not finite reaches its own row and its neighbours' alone, as in the record form: an atom without
    neighbours that shares its wave with others has plus_i times it, not a NaN from the wave's empty passes."""
    from inching_amd import ops
    from inching_amd.hessian import RecordForm, build_hessian
    print("case: entries of %g, tiles %s" % (value, shape), flush=True)
    r = np.random.default_rng(6)
    X = np.concatenate([r.uniform(0.0, 4.0, (21, 3)), [[2.0, 2.0, 100.0 + 30.0 * k] for k in range(6)],
                        [[2.0, 2.0, 300.0], [3.0, 1.0, 303.0], [2.5, 1.5, 306.0]]])
    n = len(X)
    A = build_hessian(X, 8.0, precision=(), reorder=False)
    T = ops.Tiles(A.xyz, A.rowptr, A.col, 50.0, shape)
    F = RecordForm(A)
    for at in (3, 21, 23, 26, 27, 29):       # in the cloud, without neighbours, in the chain of three
        x = r.standard_normal((n, 3))
        x[at, at % 3] = value
        x = torch.as_tensor(x.reshape(-1), device="cuda")
        out = []
        for form in (T, F):
            rec = form.buffers(1)[0]
            ops.rec_pack(form.atoms, x, rec)
            y = torch.empty(3 * form.slots, dtype=torch.float64, device="cuda")
            u = torch.empty_like(x)
            form.product(rec, None, None, 2.0, y=y)
            ops.rec_unpack(form.atoms, y, u)
            out.append(u.cpu().numpy())
        a, b = out
        kind = lambda v: np.where(np.isnan(v), 2, np.where(np.isinf(v), np.sign(v), 0))    # noqa: E731
        assert np.array_equal(kind(a), kind(b)), at
        ok = np.isfinite(b)
        assert np.all(np.abs(a[ok] - b[ok]) <= 1e-12 * np.abs(b[ok]).max())
        if 21 <= at < 27:
            assert np.array_equal(a.reshape(n, 3)[at], 2.0 * x.cpu().numpy().reshape(n, 3)[at], equal_nan=True)


@pytest.mark.parametrize("axis", [0, 1, 2])
@pytest.mark.parametrize("far,status", [(1.5e308, -3), (float("inf"), -5), (float("nan"), -5), (1e300, 0)])
def test_tile_order_of_far_coordinates(cuda, axis, far, status):
    """Columns widen until their numbers fit; a span that overflows has none (and is refused; along z it only loses the
    order), a huge one has."""
    import ctypes as C
    from inching_amd import ops
    print("case: tile order, span %g along %d" % (far, axis), flush=True)
    X = np.random.default_rng(1).uniform(0.0, 5.0, (40, 3))
    X[0, axis], X[1, axis] = -far, far
    xyz = torch.as_tensor(X, device="cuda")
    order, start = (torch.empty(41, dtype=torch.int32, device="cuda") for _ in range(2))
    nt = C.c_int64(0)
    args = (40, ops.P(xyz), 6.0, 16, ops.P(order), ops.P(start), C.byref(nt), ops.stream_ptr())
    if status and (status == -5 or axis < 2):
        with pytest.raises(ops.InchingError) as e:
            ops.call("inch_anm_tile_order", *args)
        assert e.value.status == status
        return
    ops.call("inch_anm_tile_order", *args)
    cut = start.cpu().numpy()[:nt.value + 1]
    assert np.array_equal(np.sort(order.cpu().numpy()[:40]), np.arange(40))
    assert cut[0] == 0 and cut[-1] == 40 and np.all(np.diff(cut) >= 1) and np.all(np.diff(cut) <= 16)


@pytest.mark.parametrize("case", ["stride", "span"])
def test_row_tiles_refuse_lists_without_room(cuda, case):
    """The second call finds longer lists, or columns further apart, than the first call's stride allows."""
    import ctypes as C
    from inching_amd import ops
    print("case: row tiles, %s" % case, flush=True)
    n = 40 if case == "stride" else 300000
    i32 = dict(dtype=torch.int32, device="cuda")
    per = 20 if case == "stride" else 2
    rowptr = torch.arange(0, per * n + 1, per, dtype=torch.int64, device="cuda")
    cols = torch.arange(20, **i32) if case == "stride" else torch.tensor([0, n - 1], **i32)
    col = cols.repeat(n)
    order, start = torch.arange(n, **i32), torch.arange(0, n + 1, 10, **i32)
    nt = n // 10
    slots, ulen, uidx = torch.empty(64 * nt, **i32), torch.empty(nt, **i32), torch.empty(per * n, dtype=torch.int16, device="cuda")
    for stride, ok in ((19, False),) + (((20, True),) if case == "stride" else ()):
        ulist = torch.empty(stride * nt, **i32)
        args = (n, ops.P(rowptr), ops.P(col), nt, ops.P(order), ops.P(start), 16, stride, ops.P(slots), ops.P(ulen),
                ops.P(ulist), ops.P(uidx), None, ops.stream_ptr())
        if ok:
            ops.call("inch_bsr_tiles", *args)
            assert torch.equal(ulist.view(nt, 20), cols.repeat(nt, 1))
        else:
            with pytest.raises(ops.InchingError) as e:
                ops.call("inch_bsr_tiles", *args)
            assert e.value.status == -3


def test_tile_lists_keep_no_spare_room(cuda):
    from inching_amd.hessian import build_hessian
    print("case: tile lists' stride", flush=True)
    T = build_hessian(globule(2000, seed=3), 8.0, precision=()).tiles()
    assert T.ulist.numel() == T.ntile * int(T.ulen.max())


@pytest.mark.parametrize("what", ["dimers", "chain", "globule", "few_dimers"])
def test_tiles_that_would_be_padding_are_left_out(cuda, what):
    """Structures spread thin keep the record form; dense ones, and as many slots as the chip holds at once, the tiles."""
    from inching_amd import chebyshev as CH
    from inching_amd.hessian import RecordForm, build_hessian
    from inching_amd.operator import Operator
    print("case: sparse structure %s" % what, flush=True)
    r = np.random.default_rng(2)
    if what == "globule":
        X = globule(4000, seed=3)
    elif what == "chain":
        t = 3.8 * np.arange(20000)
        X = np.stack([t, np.sin(t), np.cos(t)], 1)
    else:
        k = 5000 if what == "dimers" else 500
        d = r.uniform(0.0, 1.0, (k, 3)) * [80.0 * k ** 0.5, 80.0 * k ** 0.5, 5.0]
        X = np.concatenate([d, d + 1.5])
    A = build_hessian(X, 8.0, precision=())
    assert (A.tiles() is None) == (what in ("dimers", "chain"))
    assert isinstance(A.slot_form(), RecordForm) == (A.tiles() is None)
    v = torch.randn(A.shape[0], dtype=torch.float64, device="cuda")
    a, b = torch.empty_like(v), torch.empty_like(v)
    pol = CH.design_filter(1.0, 3.0, (1.0, 80.0), 5120, 5, 0.7)
    Operator(A, "mf64", pol=pol).apply(v, a)
    Operator(A, "mf64", pol=pol, records=False).apply(v, b)
    assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


@pytest.mark.parametrize("degree", [0, 1, 2])
@pytest.mark.parametrize("shift", [0.0, -40.0])
def test_filters_of_the_smallest_degrees(cuda, degree, shift):
    """A filter without a product is its constant, on the tiles as in the matrix's order."""
    from types import SimpleNamespace
    from inching_amd.hessian import build_hessian, rigid_body_basis
    from inching_amd.operator import Operator
    print("case: filter of degree %d, shift %g" % (degree, shift), flush=True)
    A = build_hessian(globule(300, seed=3), 8.0, precision=())
    pol = SimpleNamespace(AdjustedCoefficients=np.array([0.3, -0.7, 0.2]), AdjustedDegree=degree, cc=40.0, dd=39.0)
    Q = rigid_body_basis(A.xyz)
    v = torch.randn(900, dtype=torch.float64, device="cuda")
    a, b = torch.empty_like(v), torch.empty_like(v)
    op = Operator(A, "mf64", pol=pol, Q=Q, shift=shift)
    assert op.rec is A.tiles() is not None
    op.apply(v, a)
    Operator(A, "mf64", pol=pol, Q=Q, shift=shift, records=False).apply(v, b)
    assert float((a - b).abs().max()) <= 1e-12 * float(b.abs().max())


@pytest.mark.parametrize("x,ok", [(1e149, True), (1e151, False)])
def test_tiles_of_an_atom_out_of_range(cuda, x, ok):
    """An atom by itself so far out that its empty passes would overflow leaves the tiles to the other forms."""
    from inching_amd import ops
    print("case: an atom at x = %g" % x, flush=True)
    X = np.random.default_rng(6).uniform(0.0, 4.0, (20, 3))
    X[7, 0] = x
    xyz = torch.as_tensor(X, device="cuda")
    keep = [i for i in range(20) if i != 7]
    rows = [keep if i != 7 else [7] for i in range(20)]
    ip = torch.as_tensor(np.concatenate([[0], np.cumsum([len(r) for r in rows])]), device="cuda")
    ix = torch.as_tensor(np.concatenate(rows).astype(np.int32), device="cuda")
    if not ok:
        with pytest.raises(ops.InchingError) as e:
            ops.Tiles(xyz, ip, ix, 1e160, (32, 16))
        assert e.value.status == -3
        return
    T = ops.Tiles(xyz, ip, ix, 1e160, (32, 16))
    v = torch.randn(60, dtype=torch.float64, device="cuda")
    rec, y, u = T.buffers(1)[0], torch.empty(3 * T.slots, dtype=torch.float64, device="cuda"), torch.empty_like(v)
    ops.rec_pack(T.atoms, v, rec)
    T.product(rec, None, None, 2.0, y=y)
    ops.rec_unpack(T.atoms, y, u)
    assert T.ntile == 1 and torch.equal(u.view(20, 3)[7], 2.0 * v.view(20, 3)[7])
    assert bool(torch.isfinite(u).all())
