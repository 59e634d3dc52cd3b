"""SDDMM in feature slices (widths beyond one launch): workset order, CSR order
and the row-ordered copy, whose outputs the later slices add to, against the
oracle; outputs left dirty before the call, and residue outputs that
accumulate over calls."""
import numpy as np
import pytest

import oracle
import powersparse_amd as ps
import tolerance
from gpu_util import random_graph, say, setup

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("order", ["signature", "row"])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("N", [256, 288, 320, 352, 480, 512])
def test_slices(N, wide, order):
    # wide: Y beyond 48 MB, where slices hold 128 features, else 256 (CSR
    # order: 320); N a multiple of the slice, one slice less or more. At least
    # 8.2 k tasks of 64, so that the gathers pass 512 MB at every N
    setup()
    rng = np.random.default_rng(N + wide)
    cols = 60000 if wide else 700
    csr = random_graph(rng, 20000, cols, 90, hubs=4, hub_deg=650)
    m = ps.PowerSparseMatrixGPU.from_csr(csr, cu_count=1, csr_positions=True, task_order=order)
    say(f"SDDMM slices N={N} cols={cols} {order}: S={m.GroupTypeNum()} groups={m.GroupNum()}")
    X = rng.uniform(-1, 1, (csr.rows, N)).astype(np.float32)
    Y = rng.uniform(-1, 1, (cols, N)).astype(np.float32)
    dX, dY = ps.DeviceBuffer(host=X), ps.DeviceBuffer(host=Y)
    w = oracle.preprocess(csr.rows, csr.cols, csr.row_ptr, csr.col_ind, csr.values, 1)
    sizes = m.sddmm_output_sizes()
    outs = [ps.DeviceBuffer(host=np.full(max(n, 1), np.nan if s else 0.0, np.float32))
            for s, n in enumerate(sizes)]
    for _ in range(2):  # block outputs stored, the residue's added
        ps.SDDMMAsync(m, N, dX, dY, outs)
    ps.synchronize()
    for s in range(m.GroupTypeNum()):
        if not sizes[s]:
            continue
        E, M = oracle.sddmm(w.des[s], w.offsets(s), w.col[s], w.val[s], N, X, Y, with_mag=True)
        k = 1 if s else 2
        tolerance.check(outs[s].download(np.float32, sizes[s]), k * E, k * M, f"workset {s}")
    flat = ps.DeviceBuffer(host=np.full(csr.nnz, np.nan, np.float32))
    ps.SDDMMToCSR(m, N, dX, dY, flat)
    ps.synchronize()
    row = np.repeat(np.arange(csr.rows), np.diff(csr.row_ptr))
    x64, y64 = X.astype(np.float64)[row], Y.astype(np.float64)[csr.col_ind]
    E = (x64 * y64).sum(1) * csr.values
    M = (np.abs(x64) * np.abs(y64)).sum(1) * np.abs(csr.values)
    tolerance.check(flat.download(np.float32, csr.nnz), E, M, "CSR order")
    m.close()
