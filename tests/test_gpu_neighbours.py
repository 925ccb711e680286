"""Neighbour search where its workgroups can go wrong: runs of 32 atoms at their edges and across
columns of cells, more candidates than one LDS stage, the unordered rows, and row sorting at the
edges of its 64- and 256-entry forms and with equal entries."""
import numpy as np
import pytest
import torch

from helpers import small_globule

pytestmark = pytest.mark.gpu


def _rows(ip, ix):
    ip, ix = ip.cpu().numpy(), ix.cpu().numpy()
    return [ix[ip[i]:ip[i + 1]] for i in range(len(ip) - 1)]


def _brute(X, rc):
    d = X[None, :, :] - X[:, None, :]
    return ((d[..., 0] * d[..., 0] + d[..., 1] * d[..., 1]) + d[..., 2] * d[..., 2]) <= rc * rc


CASES = {
    "one": lambda r: r.uniform(0, 5, (1, 3)),
    "run_edge_31": lambda r: r.uniform(0, 20, (31, 3)),
    "run_edge_33": lambda r: r.uniform(0, 20, (33, 3)),
    "many_columns": lambda r: r.uniform(0, 1, (700, 3)) * [300, 300, 4],
    "one_column": lambda r: r.uniform(0, 1, (700, 3)) * [4, 4, 900],
    "one_cell_two_stages": lambda r: r.uniform(0, 7, (1500, 3)),
    "coincident": lambda r: np.repeat(r.uniform(0, 12, (60, 3)), 3, axis=0),
    "globule": lambda r: small_globule(1500, seed=11) - 40.0,
}


@pytest.mark.parametrize("case", list(CASES))
def test_neighbours_equal_brute_force(cuda, case):
    from inching_amd import ops
    print("case: neighbours %s" % case, flush=True)
    X = CASES[case](np.random.default_rng(8))
    want = _brute(X, 8.0)
    xyz = torch.as_tensor(X, device="cuda")
    ip, ix = ops.neighbours(xyz, 8.0)
    for i, row in enumerate(_rows(ip, ix)):
        assert np.array_equal(row, np.nonzero(want[i])[0]), i
    ip2, ix2 = ops.neighbours(xyz, 8.0, ascending=False)
    assert torch.equal(ip, ip2)
    for a, b in zip(_rows(ip, ix), _rows(ip2, ix2)):
        assert np.array_equal(a, np.sort(b))


def test_neighbours_reject_rows_over_the_limit(cuda):
    from inching_amd import ops
    print("case: 2,049 neighbours", flush=True)
    X = np.random.default_rng(8).uniform(0, 2, (2049, 3))
    for ascending in (True, False):
        with pytest.raises(ops.InchingError) as e:
            ops.neighbours(torch.as_tensor(X, device="cuda"), 8.0, ascending=ascending)
        assert e.value.status == -3


@pytest.mark.parametrize("equal", [False, True])
def test_row_sort_at_its_edges(cuda, equal):
    """Rows of 0 to 2048 entries through the renumbering, also with repeated columns."""
    from inching_amd import ops
    print("case: row sort, equal entries %s" % equal, flush=True)
    r = np.random.default_rng(3)
    lens = [0, 1, 3, 4, 63, 64, 65, 127, 128, 129, 192, 255, 256, 257, 700, 2048]
    n = 4096
    lens = lens + [1] * (n - len(lens))
    rows = [r.choice(n, k, replace=False) if not equal else r.integers(0, max(1, k // 2), k) for k in lens]
    ip = np.concatenate([[0], np.cumsum(lens)]).astype(np.int64)
    order = r.permutation(n).astype(np.int32)
    undo = np.empty(n, np.int64)
    undo[order] = np.arange(n)
    dev = lambda a: torch.as_tensor(a, device="cuda")    # noqa: E731
    op, oi = ops.csr_permute(dev(ip), dev(np.concatenate(rows).astype(np.int32)), dev(order), dev(undo))
    for i, row in enumerate(_rows(op, oi)):
        assert np.array_equal(row, np.sort(undo[rows[order[i]]])), i


@pytest.mark.parametrize("rc,lo,step", [(49.0, 0.0, 49.0), (7.3, 0.0, 7.3), (8.0, 5.3, 8.0), (0.8, 0.1, 0.8)])
@pytest.mark.parametrize("axis", [0, 1, 2])
def test_pairs_at_the_cutoff_across_rounded_cells(cuda, rc, lo, step, axis):
    """Atoms one cutoff apart along an axis: (v - lo) / rc rounds to either side of a whole number, so that with cells
    of the cutoff itself two such atoms could lie two cells apart, and a row held the other while its own did not."""
    from inching_amd import ops
    print("case: pairs at the cutoff %g, axis %d" % (rc, axis), flush=True)
    X = np.zeros((200, 3))
    X[:, axis] = lo + step * np.arange(200)
    X[100:, (axis + 1) % 3] = 0.25 * rc
    X[100:, axis] = X[:100, axis]
    want = _brute(X, rc)
    ip, ix = ops.neighbours(torch.as_tensor(X, device="cuda"), rc)
    for i, row in enumerate(_rows(ip, ix)):
        assert np.array_equal(row, np.nonzero(want[i])[0]), i


@pytest.mark.parametrize("case", ["one", "run_edge_33", "one_cell_two_stages", "globule"])
def test_one_call_search_equals_the_steps(cuda, case):
    """inch_neighbors_celllist: the count pass, the fill pass, a buffer one short, and rows over 2,048 entries."""
    import ctypes as C
    from inching_amd import ops
    print("case: one-call search %s" % case, flush=True)
    X = CASES[case](np.random.default_rng(8))
    xyz = torch.as_tensor(X, device="cuda")
    n = len(X)
    want = ops.neighbours(xyz, 8.0)
    ip = torch.full((n + 1,), -1, dtype=torch.int64, device="cuda")
    nnz = C.c_int64(-1)
    call = lambda ix, cap: ops.call("inch_neighbors_celllist", n, ops.P(xyz), 8.0, ops.P(ip), ops.P(ix), cap,    # noqa: E731
                                    C.byref(nnz), ops.stream_ptr())
    call(None, 0)
    assert nnz.value == want[1].numel() and torch.equal(ip, want[0])
    ix = torch.full((nnz.value + 1,), -7, dtype=torch.int32, device="cuda")
    with pytest.raises(ops.InchingError) as e:
        call(ix, nnz.value - 1)
    assert e.value.status == -3 and bool((ix == -7).all())
    call(ix, nnz.value)
    assert torch.equal(ix[:-1], want[1]) and int(ix[-1]) == -7
    if case == "one":
        xyz, n = torch.rand((2049, 3), dtype=torch.float64, device="cuda"), 2049
        ip = torch.empty(n + 1, dtype=torch.int64, device="cuda")
        call(None, 0)
        assert nnz.value == 2049 * 2049
        ix = torch.empty(nnz.value, dtype=torch.int32, device="cuda")
        with pytest.raises(ops.InchingError) as e:
            call(ix, nnz.value)
        assert e.value.status == -3


@pytest.mark.parametrize("far", [1e5, 1e25, 1e300, 1.5e308])
@pytest.mark.parametrize("axis", [0, 2])
def test_neighbours_across_any_span(cuda, far, axis):
    """Atoms a few cells or any distance apart, the span's overflow included: brute force, and built either way."""
    from inching_amd import ops
    from inching_amd.hessian import build_hessian
    print("case: atoms %g apart along %d" % (far, axis), flush=True)
    X = np.random.default_rng(4).uniform(0.0, 6.0, (40, 3))
    X[3, axis], X[20, axis] = far, -far
    with np.errstate(over="ignore", invalid="ignore"):
        want = _brute(X, 8.0)
    ip, ix = ops.neighbours(torch.as_tensor(X, device="cuda"), 8.0)
    for i, row in enumerate(_rows(ip, ix)):
        assert np.array_equal(row, np.nonzero(want[i])[0]), i
    A = build_hessian(X, 8.0, precision=())
    assert A.nnzb == int(want.sum())
