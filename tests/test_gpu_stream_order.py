"""SpMM and SDDMM with work queued on the null stream and on the supplied
streams before the call: the launch comes after all of it, for blocking and
non-blocking streams, busy and idle ones."""
import numpy as np
import pytest

import oracle
import powersparse_amd as ps
import tolerance
from gpu_util import random_graph, say, setup

pytestmark = pytest.mark.gpu

N = 64
HEAVY = 256 << 20


class Torch:
    """A non-blocking stream of the default priority."""

    def __init__(self):
        import torch
        self.stream = torch.cuda.Stream()
        self.ptr = self.stream.cuda_stream


@pytest.fixture(scope="module")
def case():
    setup()
    rng = np.random.default_rng(8)
    csr = random_graph(rng, 3000, 2000, 60, hubs=4, hub_deg=700)
    m = ps.PowerSparseMatrixGPU.from_csr(csr, cu_count=1)
    X = rng.uniform(-1, 1, (csr.rows, N)).astype(np.float32)
    Y = rng.uniform(-1, 1, (csr.cols, N)).astype(np.float32)
    return csr, m, X, Y, ps.DeviceBuffer(HEAVY)


def late(heavy, stream):
    """A few milliseconds of work on the stream (fills of 256 MB)."""
    for _ in range(20):
        heavy.zero(stream)


# who has work left: the null stream (the outputs' clearing), and which of the
# supplied streams (an operand's copy)
@pytest.mark.parametrize("op", ["spmm", "sddmm"])
@pytest.mark.parametrize("first", ["blocking", "non-blocking", "null"])
@pytest.mark.parametrize("other", ["blocking", "non-blocking"])
@pytest.mark.parametrize("work", ["null", "first", "other", "null+first", "null+other", "none"])
def test_behind_queued_work(case, op, first, other, work):
    csr, m, X, Y, heavy = case
    S = m.GroupTypeNum()
    assert S >= 3
    kinds = {"blocking": ps.Stream, "non-blocking": Torch, "null": lambda: None}
    streams = [kinds[first]()] + [kinds[other]() for _ in range(S - 1)]
    say(f"{op} streams[0] {first}, others {other}, work on {work}")
    x, y = ps.DeviceBuffer(host=X), ps.DeviceBuffer(host=Y)
    late_y = ps.DeviceBuffer(host=np.full_like(Y, np.nan))
    sizes = [csr.rows * N] if op == "spmm" else m.sddmm_output_sizes()
    outs = [ps.DeviceBuffer(host=np.full(max(n, 1), np.nan, np.float32)) for n in sizes]
    ps.synchronize()
    on = {"first": streams[0], "other": streams[1]}
    queued = [k for k in work.split("+") if k in on]
    if "null" in work:
        late(heavy, None)
    for o in outs:
        o.zero()
    if "null" not in work:
        ps.synchronize()
    for k in queued:
        late(heavy, on[k])
        ps._hip_call(ps._native.hip().ps_memcpy_dtod_async(late_y.ptr, y.ptr, Y.nbytes,
                                                           ps._ptr(on[k])))
    rhs = late_y if queued else y
    if op == "spmm":
        ps.SpMM(m, N, rhs, outs[0], S, streams)
        got = outs[0].download(np.float32).reshape(csr.rows, N)
        E, M = oracle.spmm(csr.row_ptr, csr.col_ind, csr.values, N, Y, with_mag=True)
        tolerance.check(got, E, M, "SpMM")
        return
    ps.SDDMM(m, N, x, rhs, outs, S, streams)
    offs0 = m.residue_offset()
    for s in range(S):
        if not sizes[s]:
            continue
        col, val, des = m.download_workset(s)
        offs = offs0 if s == 0 else np.arange(m.GroupNum()[s] + 1) * ps.GROUP_SIZE(s)
        E, M = oracle.sddmm(des, offs, col, val, N, X, Y, with_mag=True)
        tolerance.check(outs[s].download(np.float32, sizes[s]), E, M, f"SDDMM {s}")
