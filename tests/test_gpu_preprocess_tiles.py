"""The preprocessing's LDS tile sort at the edges of its tiles: the workset
gather against numpy's stable sort, index arrays equal, values bitwise."""
import numpy as np
import pytest

import powersparse_amd as ps
from powersparse_amd import _native
from gpu_util import say, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gs", [64, 128, 512, 2048, 4096, 8192])
@pytest.mark.parametrize("groups", [1, 3, 33])
@pytest.mark.parametrize("cols", [1, 70, 1 << 20, (1 << 31) - 1])
def test_gather_tiles(gs, groups, cols):
    # groups per tile: whole tiles, a remainder, one group; columns from one
    # value (every key ties: nothing to sort) to all 31 bits (one group a tile)
    setup()
    say(f"gather gs={gs} groups={groups} cols={cols}")
    rng = np.random.default_rng(gs + groups + cols % 1000)
    n = gs * groups
    col = rng.integers(0, cols, n).astype(np.int32)
    if groups == 33:  # some groups in order already, some reversed
        for k in range(0, 33, 3):
            col[k * gs:(k + 1) * gs].sort()
        for k in range(1, 33, 3):
            col[k * gs:(k + 1) * gs][::-1].sort()
    val = rng.uniform(-1, 1, n).astype(np.float32)
    start = (rng.permutation(groups) * gs).astype(np.int32)
    perm = rng.permutation(groups).astype(np.uint32)
    ranked = np.concatenate([k * gs + rng.permutation(gs) for k in range(groups)]).astype(np.uint32)
    d = [ps.DeviceBuffer(host=a) for a in (perm, start, ranked, col, val)]
    out = [ps.DeviceBuffer(n * 4) for _ in range(3)]
    ps._hip_call(_native.hip().ps_pre_gather_workset_cols(
        gs, cols, d[0].ptr, groups, d[1].ptr, None, d[2].ptr, d[3].ptr, d[4].ptr, out[0].ptr,
        out[1].ptr, out[2].ptr, None))
    pos = np.empty(n, np.int32)
    for k in range(groups):
        p = ranked[start[perm[k]]:start[perm[k]] + gs]
        pos[k * gs:(k + 1) * gs] = p[np.argsort(col[p], kind="stable")]
    np.testing.assert_array_equal(out[2].download(np.int32), pos)
    np.testing.assert_array_equal(out[0].download(np.int32), col[pos])
    np.testing.assert_array_equal(out[1].download(np.uint32), val[pos].view(np.uint32))
