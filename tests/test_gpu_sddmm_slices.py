"""SDDMM in feature slices (widths beyond one launch): workset order, CSR order
and the row-ordered copy, whose outputs the later slices add to, against the
oracle; outputs left dirty before the call, and residue outputs that
accumulate over calls; values whose product with a part of the dot overflows."""
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


@pytest.mark.parametrize("order", ["signature", "row"])
@pytest.mark.parametrize("wide,N", [(False, 288), (False, 416), (False, 512), (True, 288),
                                    (True, 352), (True, 480)])
def test_values_above_one(N, wide, order):
    # the added-to residue computed whole in the last slice: windows of its
    # width, the last one short (288: 160 + 128; 416: 224 + 192) or not
    setup()
    rng = np.random.default_rng(N + wide)
    cols = 60000 if wide else 700
    csr = random_graph(rng, 20000, cols, 90, hubs=4, hub_deg=650)
    csr = ps.HostCsr(csr.rows, csr.cols, csr.row_ptr, csr.col_ind, csr.values * np.float32(5))
    m = ps.PowerSparseMatrixGPU.from_csr(csr, cu_count=1, task_order=order)
    say(f"SDDMM slices, values up to 5: N={N} cols={cols} {order}")
    X = rng.uniform(-1, 1, (csr.rows, N)).astype(np.float32)
    Y = rng.uniform(-1, 1, (cols, N)).astype(np.float32)
    dX, dY = ps.DeviceBuffer(host=X), ps.DeviceBuffer(host=Y)
    w = oracle.preprocess(csr.rows, csr.cols, csr.row_ptr, csr.col_ind, csr.values, 1)
    sizes = m.sddmm_output_sizes()
    outs = [ps.DeviceBuffer(host=np.full(max(n, 1), np.nan if s else 0.0, np.float32))
            for s, n in enumerate(sizes)]
    for _ in range(2):
        ps.SDDMMAsync(m, N, dX, dY, outs)
    ps.synchronize()
    for s in range(m.GroupTypeNum()):
        if sizes[s]:
            E, M = oracle.sddmm(w.des[s], w.offsets(s), w.col[s], w.val[s], N, X, Y, with_mag=True)
            k = 1 if s else 2
            tolerance.check(outs[s].download(np.float32, sizes[s]), k * E, k * M, f"workset {s}")
    m.close()


def test_unbounded_operands():
    # an infinite or NaN feature reaches the dots that read it and no others,
    # also through the last, shorter window (whose shared features are left out)
    setup()
    rng = np.random.default_rng(4)
    N = 288
    csr = random_graph(rng, 20000, 700, 90, hubs=4, hub_deg=650)
    csr = ps.HostCsr(csr.rows, csr.cols, csr.row_ptr, csr.col_ind, csr.values * np.float32(5))
    m = ps.PowerSparseMatrixGPU.from_csr(csr, cu_count=1, csr_positions=True, hub_block="off")
    X = np.ones((csr.rows, N), np.float32)
    Y = np.ones((csr.cols, N), np.float32)
    places = [0, 31, 127, 128, 159, 160, 255, 256, 287]
    for i, f in enumerate(places):
        Y[i, f] = np.inf
        Y[100 + i, f] = np.nan
    dX, dY = ps.DeviceBuffer(host=X), ps.DeviceBuffer(host=Y)
    outs = [ps.DeviceBuffer.zeros(max(n, 1) * 4) for n in m.sddmm_output_sizes()]
    ps.SDDMMAsync(m, N, dX, dY, outs)
    flat = ps.DeviceBuffer.zeros(csr.nnz * 4)
    csr_order = ps.DeviceBuffer.zeros(csr.nnz * 4)
    ps.WorksetToCSR(m, outs, flat)
    ps.SDDMMToCSR(m, N, dX, dY, csr_order)
    ps.synchronize()
    with np.errstate(invalid="ignore"):
        want = csr.values * Y.sum(1)[csr.col_ind]
    for got in (flat, csr_order):
        got = got.download(np.float32, csr.nnz)
        np.testing.assert_array_equal(np.isnan(got), np.isnan(want))
        np.testing.assert_array_equal(np.isinf(got), np.isinf(want))
        ok = np.isfinite(want)
        np.testing.assert_allclose(got[ok], want[ok], rtol=1e-6)
    m.close()


@pytest.mark.parametrize("order", ["signature", "row"])
@pytest.mark.parametrize("wide", [False, True])
@pytest.mark.parametrize("N", [288, 512])
def test_values_near_the_limit(N, wide, order):
    # each dot is 2^30, of halves near +-2^37: every sum is exact, and 2^95
    # times the whole dot is finite while 2^95 times a slice's part is not
    setup()
    rng = np.random.default_rng(N)
    cols = 60000 if wide else 700
    csr = random_graph(rng, 20000, cols, 90, hubs=4, hub_deg=650)
    csr = ps.HostCsr(csr.rows, csr.cols, csr.row_ptr, csr.col_ind,
                     np.full(csr.nnz, 2.0**95, np.float32))
    m = ps.PowerSparseMatrixGPU.from_csr(csr, cu_count=1, csr_positions=True, task_order=order)
    say(f"SDDMM slices near the limit N={N} cols={cols} {order}: S={m.GroupTypeNum()}")
    Y = np.full((cols, N), 2.0**30, np.float32)
    Y[:, N // 2:] *= -1
    Y[:, N - 1] = 0
    dX = ps.DeviceBuffer(host=np.ones((csr.rows, N), np.float32))
    dY = ps.DeviceBuffer(host=Y)
    sizes = m.sddmm_output_sizes()
    outs = [ps.DeviceBuffer.zeros(max(n, 1) * 4) for n in sizes]
    ps.SDDMMAsync(m, N, dX, dY, outs)
    flat = ps.DeviceBuffer(host=np.full(csr.nnz, np.nan, np.float32))
    ps.SDDMMToCSR(m, N, dX, dY, flat)
    ps.synchronize()
    for s, n in enumerate(sizes):
        assert (outs[s].download(np.float32, n) == np.float32(2.0**125)).all(), s
    assert (flat.download(np.float32, csr.nnz) == np.float32(2.0**125)).all()
    m.close()


@pytest.mark.parametrize("degree,rows", [(6, 90000), (40, 20000)])
@pytest.mark.parametrize("scale", [1, 5])
@pytest.mark.parametrize("N", [192, 256])
def test_one_launch_where_slices_cost_more(N, scale, degree, rows):
    # two of: fewer than 256 features, values above 1, nearly all nonzeros in
    # the residue. CSR order is one launch up to 256 features, so workset order
    # gives its dots bit for bit exactly when it is one launch too
    setup()
    one = (N < 256) + (scale > 1) + (degree < 32) >= 2
    rng = np.random.default_rng(N + degree + scale)
    cols = 70000
    ci = (rng.integers(0, cols, (rows, 1)) + np.arange(degree) * 1313) % cols
    rp = np.arange(rows + 1, dtype=np.int32) * degree
    values = (rng.uniform(0.5, 1, rows * degree) * scale).astype(np.float32)
    csr = ps.HostCsr(rows, cols, rp, np.sort(ci, 1).reshape(-1).astype(np.int32), values)
    m = ps.PowerSparseMatrixGPU.from_csr(csr, cu_count=1, csr_positions=True, hub_block="off")
    say(f"SDDMM N={N} values up to {scale} degree {degree}: groups={m.GroupNum()}")
    assert (sum(m.GroupNum()[1:]) > 0) == (degree > 32)
    X = rng.uniform(-1, 1, (rows, N)).astype(np.float32)
    Y = rng.uniform(-1, 1, (cols, N)).astype(np.float32)
    dX, dY = ps.DeviceBuffer(host=X), ps.DeviceBuffer(host=Y)
    outs = [ps.DeviceBuffer.zeros(max(n, 1) * 4) for n in m.sddmm_output_sizes()]
    ps.SDDMMAsync(m, N, dX, dY, outs)
    flat, csr_order = ps.DeviceBuffer.zeros(csr.nnz * 4), ps.DeviceBuffer.zeros(csr.nnz * 4)
    ps.WorksetToCSR(m, outs, flat)
    ps.SDDMMToCSR(m, N, dX, dY, csr_order)
    ps.synchronize()
    got, want = flat.download(np.float32, csr.nnz), csr_order.download(np.float32, csr.nnz)
    assert np.array_equal(got, want) == one
    row = np.repeat(np.arange(rows), degree)
    E, M = np.empty(csr.nnz), np.empty(csr.nnz)
    for b in range(0, csr.nnz, 1 << 16):
        s = slice(b, b + (1 << 16))
        xy = X[row[s]].astype(np.float64) * Y[csr.col_ind[s]]
        E[s], M[s] = xy.sum(1) * values[s], np.abs(xy).sum(1) * np.abs(values[s])
    tolerance.check(got, E, M, "workset order")
    tolerance.check(want, E, M, "CSR order")
    m.close()
