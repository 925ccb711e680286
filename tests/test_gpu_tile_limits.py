"""What the tile form's construction refuses, and what it takes at its limits."""
import numpy as np
import pytest
import torch

from helpers import small_globule

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("times", [1, 2, 11, 12, 60])
def test_tile_rows_with_repeated_columns(cuda, times):
    """A repeated column counts as often as it is listed, up to the 1,349 terms of a row that a tile of 16 atoms has
    places for (119 others x 11 = 1,309); longer rows are refused."""
    from inching_amd import ops
    print("case: columns repeated %d times" % times, flush=True)
    n = 120
    xyz = torch.as_tensor(small_globule(n, seed=2), device="cuda")
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
