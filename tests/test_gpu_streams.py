"""Results that a call hands out are whole on every stream, and its scratch is neither given back while
kernels still read it nor taken while earlier work still writes it."""
import numpy as np
import pytest
import torch

from inching_amd.synth import globule

pytestmark = pytest.mark.gpu

LONG = 50_000_000     # cycles of a wait that outlasts the launches after it (0.02 s or more)


def _cloud(n, seed):
    return torch.as_tensor(np.random.default_rng(seed).uniform(0.0, (n / 0.05) ** (1.0 / 3.0), (n, 3)), device="cuda")


@pytest.mark.parametrize("own", [False, True])
@pytest.mark.parametrize("ascending", [True, False])
def test_neighbours_are_whole_on_return(cuda, own, ascending):
    from inching_amd import ops
    print("case: neighbours whole on return, stream %s, ascending %s" % (own, ascending), flush=True)
    xyz = _cloud(60000, 1)
    s = torch.cuda.Stream() if own else None
    torch.cuda.synchronize()
    ip, ix = ops.neighbours(xyz, 8.0, stream=s, ascending=ascending)
    assert (s or torch.cuda.current_stream()).query()
    other = torch.cuda.Stream()
    with torch.cuda.stream(other):      # no wait between: the list is symmetric, every row names itself
        total = ip[-1].item()
        rows = torch.repeat_interleave(torch.arange(60000, device="cuda"), ip.diff(), output_size=total)
        assert int((rows == ix).sum()) == 60000
        assert int((rows * 131071 + ix).sum() - (ix.long() * 131071 + rows).sum()) == 0
    torch.cuda.synchronize()


def test_neighbours_wait_for_a_reused_block(cuda):
    """The result's memory comes from the current stream, where a write to the block's former tensor may still be
    queued: the search on another stream follows it, and coordinates still being written there too."""
    from inching_amd import ops
    print("case: neighbours after a reused block", flush=True)
    n = 20000
    xyz = _cloud(n, 2)
    ip, ix = ops.neighbours(xyz, 8.0)
    want = ip.clone(), ix.clone()
    later = torch.full_like(xyz, 1.0)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda._sleep(LONG)
    later.copy_(xyz)
    ip.fill_(0)
    ix.fill_(0)
    del ip, ix
    ip, ix = ops.neighbours(later, 8.0, stream=s)
    torch.cuda.synchronize()
    assert torch.equal(ip, want[0]) and torch.equal(ix, want[1])


def test_build_without_ordering_on_another_stream(cuda):
    from inching_amd.hessian import build_hessian
    print("case: build_hessian on one stream, product on another", flush=True)
    X = globule(3000, seed=4)
    x = torch.randn(9000, dtype=torch.float64, device="cuda")
    ref = build_hessian(X, 8.0, reorder=False, precision=()).matfree(x)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        A = build_hessian(X, 8.0, reorder=False, precision=())
    with torch.cuda.stream(s2):
        y = A.matfree(x)
    torch.cuda.synchronize()
    assert torch.equal(y, ref)


def test_block_product_keeps_its_scratch(cuda, monkeypatch):
    """The packed columns of a block product on another stream are not handed to the current stream while that product
    has still to run."""
    from inching_amd import ops
    from inching_amd.hessian import build_hessian
    print("case: block product's scratch", flush=True)
    A = build_hessian(globule(3000, seed=5), 8.0, precision=())
    T = A.tiles()
    X = torch.randn(9000, 16, dtype=torch.float64, device="cuda")
    Y, want = torch.empty_like(X), torch.empty_like(X)
    T.apply(X, want, 1.0)
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    work, call = [], ops.call

    def spy(name, *args):
        if name == "inch_anm_matfree_tile_apply":
            work.append(args[-2])
        return call(name, *args)

    monkeypatch.setattr(ops, "call", spy)
    with torch.cuda.stream(s):
        torch.cuda._sleep(LONG)
    T.apply(X, Y, 1.0, stream=s)
    junk = [torch.empty(12 * T.slots * 4, dtype=torch.float64, device="cuda") for _ in range(4)]
    assert len(work) == 1 and all(t.data_ptr() != work[0] for t in junk)
    torch.cuda.synchronize()
    assert torch.equal(Y, want)


def test_filter_on_another_stream_than_its_operator(cuda):
    """The record buffers of an Operator are whole when it is made: its first application may run elsewhere."""
    from inching_amd import chebyshev as CH
    from inching_amd.hessian import build_hessian
    from inching_amd.operator import Operator
    print("case: operator made on one stream, applied on another", flush=True)
    A = build_hessian(globule(3000, seed=5), 8.0, precision=())
    pol = CH.design_filter(1.0, 3.0, (1.0, 80.0), 5120, 5, 0.7)
    v = torch.randn(9000, dtype=torch.float64, device="cuda")
    u, want = torch.empty_like(v), torch.empty_like(v)
    Operator(A, "mf64", pol=pol).apply(v, want)
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(s1):
        torch.cuda._sleep(LONG)
        op = Operator(A, "mf64", pol=pol)
    assert s1.query()
    with torch.cuda.stream(s2):
        op.apply(v, u)
    torch.cuda.synchronize()
    assert torch.equal(u, want)


@pytest.mark.parametrize("layout", ["Tiles", "BsrTiles"])
def test_layouts_wait_for_reused_blocks(cuda, layout):
    """The layouts' arrays come from the current stream's pool too, with writes to their former tensors still queued."""
    from inching_amd import ops
    from inching_amd.hessian import build_hessian
    print("case: %s after reused blocks" % layout, flush=True)
    A = build_hessian(globule(3000, seed=5), 8.0, precision=())
    names = {"Tiles": ["atoms", "waves", "pairs", "ulen", "ulist", "rec"], "BsrTiles": ["slots", "ulen", "ulist", "uidx"]}

    def make(stream):
        args = ((32, 16),) if layout == "Tiles" else ()
        return getattr(ops, layout)(A.xyz, A.rowptr, A.col, 10.0, *args, stream=stream)

    want = make(None)
    want = {k: getattr(want, k).clone() for k in names[layout]}
    s = torch.cuda.Stream()
    torch.cuda.synchronize()
    old = make(None)
    torch.cuda._sleep(LONG)
    for k in names[layout]:
        getattr(old, k).fill_(0)
    del old
    got = make(s)
    torch.cuda.synchronize()
    n = getattr(got, "ntile")
    for k in names[layout]:
        a, b = getattr(got, k), want[k]
        if k == "ulist":          # entries past a tile's union are not written
            keep = torch.arange(a.numel() // n, device="cuda")[None, :] < want["ulen"][:, None]
            a, b = a.view(n, -1)[keep], b.view(n, -1)[keep]
        assert torch.equal(a, b), k
