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


@pytest.mark.parametrize("length", [1, 33, 3488, (1 << 31) - 1])
@pytest.mark.parametrize("worksets", [1, 2, 9])
def test_group_lists(length, worksets):
    # each group's distinct signature bits: residue groups of 1..31 members, one
    # and several groups per tile, all bits equal, none equal, already sorted
    import ctypes
    setup()
    say(f"group lists L={length} worksets={worksets}")
    rng = np.random.default_rng(length % 1000 + worksets)
    num = [70] + [int(rng.choice([0, 1, 5, 67])) for _ in range(worksets - 1)]
    if worksets == 9:
        num[2], num[7], num[8] = 67, 3, 2  # 64: several a tile; 2048 and 4096
    sizes = [rng.integers(1, 32, num[0])] + [np.full(num[s], 32 << (s - 1)) for s in range(1, worksets)]
    begin = np.concatenate([[0], np.cumsum(np.concatenate(sizes))])
    n = int(begin[-1])
    cols = max(1, n // 3)
    sigbit = rng.integers(0, length, cols).astype(np.int32)
    if length == 3488:
        sigbit.sort()  # sorted columns then give sorted bits
    col = rng.integers(0, cols, n).astype(np.int32)
    bounds = np.concatenate([[0], np.cumsum(num)])
    starts = [begin[bounds[s]:bounds[s + 1]].astype(np.int32) for s in range(worksets)]
    if length == 3488:
        for a, b in zip(begin[:-1:2], begin[1::2]):
            col[a:b].sort()
    ranked = rng.permutation(n).astype(np.uint32)
    by_rank = np.empty(n, np.int32)
    by_rank[ranked] = col  # col_ind such that ranked position i holds column col[i]
    d = [ps.DeviceBuffer(host=a) for a in (ranked, by_rank, sigbit, sizes[0].astype(np.int32))]
    ds = [ps.DeviceBuffer(host=a if a.size else np.zeros(1, np.int32)) for a in starts]
    total = int(bounds[-1])
    lists, at, end = ps.DeviceBuffer(n * 4), ps.DeviceBuffer(total * 4), ps.DeviceBuffer(total * 4)
    counts = (ctypes.c_int * worksets)(*num)
    ptrs = (ctypes.c_void_p * worksets)(*[x.ptr for x in ds])
    ps._hip_call(_native.hip().ps_pre_group_lists(
        worksets, counts, ptrs, d[3].ptr, d[0].ptr, d[1].ptr, d[2].ptr, length, lists.ptr, at.ptr,
        end.ptr, None))
    got, a, e = lists.download(np.uint32), at.download(np.uint32), end.download(np.uint32)
    for g in range(total):
        want = np.unique(sigbit[col[begin[g]:begin[g + 1]]])
        assert a[g] == begin[g]
        np.testing.assert_array_equal(got[a[g]:e[g]], want, err_msg=f"group {g}")


@pytest.mark.parametrize("cols", [1, 255, 256, 257, 100000, (1 << 23), (1 << 23) + 1])
@pytest.mark.parametrize("nnz", [1, 2047, 2049, 1 << 20, (1 << 26) + 5])
def test_col_histogram(cols, nnz):
    # one class, all classes, the most columns the split takes and one beyond;
    # one nonzero, chunk remainders, more than one slab
    setup()
    say(f"column histogram cols={cols} nnz={nnz}")
    rng = np.random.default_rng(cols + nnz)
    if nnz > 1 << 21 and cols < 100000:
        pytest.skip("the slab edge needs one column range")
    c = rng.integers(0, cols, nnz, dtype=np.int32)
    c[::3] //= 1 + cols // 50  # popular columns
    c[-1] = cols - 1
    d, out = ps.DeviceBuffer(host=c), ps.DeviceBuffer.zeros(cols * 4)
    ps._hip_call(_native.hip().ps_pre_col_histogram_cols(d.ptr, nnz, cols, out.ptr, None))
    np.testing.assert_array_equal(out.download(np.int32), np.bincount(c, minlength=cols))


@pytest.mark.parametrize("at", [0, (1 << 24) - 1, 1 << 24, (1 << 24) + 4])
@pytest.mark.parametrize("what", ["column", "negative", "nan", "inf"])
def test_large_csr_is_checked_on_the_device(at, what):
    # a matrix large enough for the device's checks, one bad entry: refused with
    # the host check's message; the same matrix without it is built
    setup()
    rows, cols, n = 1 << 18, 1000, (1 << 24) + 5
    rp = np.minimum(np.arange(rows + 1, dtype=np.int64) * 65, n).astype(np.int32)
    rp[-1] = n
    ci = (np.arange(n, dtype=np.int64) * 7 % cols).astype(np.int32)
    va = np.ones(n, np.float32)
    say(f"check {what} at {at}")
    ok = (ci[at], va[at])
    if what == "column":
        ci[at] = cols
    elif what == "negative":
        ci[at] = -1
    else:
        va[at] = np.nan if what == "nan" else -np.inf
    with pytest.raises(ValueError, match="Invalid CSR column index or sparse value"):
        ps.PowerSparseMatrixGPU(rows, cols, n, rp, ci, va)
    ci[at], va[at] = ok
    if at == 0:
        m = ps.PowerSparseMatrixGPU(rows, cols, n, rp, ci, va)
        assert m.MatrixNNZ() == n
        m.close()
