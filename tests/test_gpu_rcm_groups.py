"""Device ordering where a parent has very many children (a star, a hub above 2,048 children), many levels (a path,
longer than one batch of rounds) and many components, against the host ordering, which is bit-exact."""
import numpy as np
import pytest
import torch

from inching_amd import ops

pytestmark = pytest.mark.gpu


def _csr(n, edges):
    rows = [[] for _ in range(n)]
    for a, b in edges:
        rows[a].append(b)
        rows[b].append(a)
    rows = [sorted(set(r + [i])) for i, r in enumerate(rows)]
    ptr = np.concatenate([[0], np.cumsum([len(r) for r in rows])]).astype(np.int64)
    return ptr, np.concatenate(rows).astype(np.int32)


def _graph(kind):
    rng = np.random.default_rng(7)
    if kind == "star":
        return 300, [(17, j) for j in range(300) if j != 17]
    if kind == "hub":
        n = 3000
        return n, [(0, j) for j in range(1, n)] + [tuple(e) for e in rng.integers(1, n, (4000, 2)) if e[0] != e[1]]
    if kind == "path":
        p = rng.permutation(100)
        return 100, [(int(a), int(b)) for a, b in zip(p[:-1], p[1:])]
    if kind == "islands":
        return 500, [(i, i + 1) for i in range(499) if i % 5 != 4]
    if kind == "single":
        return 1, []
    n = 700
    return n, [tuple(e) for e in rng.integers(0, n, (2500, 2)) if e[0] != e[1]]


@pytest.mark.parametrize("kind", ["star", "hub", "path", "islands", "single", "random"])
@pytest.mark.parametrize("reverse", [True, False])
def test_rcm_device_groups(kind, reverse):
    n, edges = _graph(kind)
    ptr, idx = _csr(n, edges)
    host = ops.rcm_host(ptr, idx, reverse=reverse)
    dev = ops.rcm_device(torch.as_tensor(ptr, device="cuda"), torch.as_tensor(idx, device="cuda"), reverse=reverse)
    assert np.array_equal(host[0], dev[0].cpu().numpy()) and np.array_equal(host[1], dev[1].cpu().numpy())
