"""The workloads this framework's performance is followed on, and how one pass of each is run.

A case is a graph (its family and size), an operation and a feature width. The
operations are the three things a user's program does: build the block/residue
worksets of a CSR matrix, aggregate node features (SpMM), and score edges
(SDDMM, in workset order or in the input CSR's order). Sizes are the
synthetic benchmark graphs' (powersparse_amd/host/synth.cpp: C0, C1, C3, C4)
and reduced or ragged ones between them; the reference's own widths are 32 and
128, the others are accepted too. Graphs are drawn on the GPU from the seed
alone, with the distributions of synth.cpp: degrees that vary uniformly,
Chung-Lu power laws whose rows keep their degree, and communities with
empty and single-entry rows.
"""
import math

import torch

import powersparse_amd as ps

# ------------------------------------------------------------------ cases


def _case(name, op, graph, rows, N, **more):
    return dict(name=name, op=op, graph=graph, rows=rows, N=N, **more)


def listed():
    return [
        # A small graph (a few citations per paper), one layer of 32 features:
        # the smallest call, through the synchronising drop-in entry point.
        _case("spmm_small_n32", "spmm", "uniform", 4096, 32, cols=4096, deg_lo=1, deg_hi=31,
              sync=True),
        # Edge scores of a 10 k-node social graph, the same entry point; several worksets.
        _case("sddmm_small_n32", "sddmm", "power", 10000, 32, gamma=2.1, mean=50.0, clip=2500,
              shuffled=False, sync=True),
        # Its preprocessing: what a program that loads many small graphs pays for each.
        _case("build_small", "build", "power", 10000, 0, gamma=2.1, mean=50.0, clip=2500,
              shuffled=False),
        # A bipartite graph of ragged shape (users x items), a width between the usual ones.
        _case("spmm_rect_n96", "spmm", "uniform", 200003, 96, cols=77777, deg_lo=0, deg_hi=60),
        # Attention scores with many heads, handed back in the caller's CSR order;
        # a power law with node ids in no order.
        _case("sddmm_csr_n256", "sddmm_csr", "power", 100003, 256, gamma=2.1, mean=50.0, clip=25000,
              shuffled=True),
        # The million-node power-law graph at the reference's two widths.
        _case("spmm_power_n32", "spmm", "power", 1000000, 32, gamma=2.1, mean=50.0, clip=50000,
              shuffled=False),
        _case("sddmm_power_n128", "sddmm", "power", 1000000, 128, gamma=2.1, mean=50.0, clip=50000,
              shuffled=False),
        # Its preprocessing.
        _case("build_power", "build", "power", 1000000, 0, gamma=2.1, mean=50.0, clip=50000,
              shuffled=False),
        # The community graph: local neighbourhoods, empty and single-entry rows.
        _case("spmm_community_n64", "spmm", "community", 2048 * 1024, 64, block=1024, p_intra=0.02,
              inter=8.0, empty=0.05, single=0.05),
        # The headline graph, 264 M nonzeros with dense hubs: both operators at N = 128.
        _case("spmm_hub_n128", "spmm", "power", 1600000, 128, gamma=1.8, mean=165.0, clip=100000,
              shuffled=False),
        _case("sddmm_hub_n128", "sddmm", "power", 1600000, 128, gamma=1.8, mean=165.0, clip=100000,
              shuffled=False),
        # Its preprocessing, dense hub block included.
        _case("build_hub", "build", "power", 1600000, 0, gamma=1.8, mean=165.0, clip=100000,
              shuffled=False),
    ]


# A drawn case's nonzeros, and nonzeros times width, stay below half of the
# largest listed case's.
_DRAW_NNZ = 130e6
_DRAW_WORK = 130e6 * 128


def _log_between(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(["spmm", "spmm", "sddmm", "sddmm_csr", "build"])
    graph = rng.choice(["uniform", "power", "power", "community"])
    rows = _log_between(rng, 2000, 1600000)
    mean = math.exp(rng.uniform(math.log(4.0), math.log(165.0)))
    mean = min(mean, _DRAW_NNZ / rows, rows / 16.0)
    N = 0 if op == "build" else 32 * _log_between(rng, 1, 16)
    while N > 32 and mean * rows * N > _DRAW_WORK:
        N -= 32
    case = dict(op=op, graph=graph, rows=rows, N=N)
    if graph == "uniform":
        lo = int(rng.uniform(0.0, 0.7) * mean)
        case.update(cols=_log_between(rng, 1000, 1600000), deg_lo=lo,
                    deg_hi=max(lo + 1, int(2 * mean) - lo))
        case["deg_hi"] = min(case["deg_hi"], case["cols"] // 2)
        case["deg_lo"] = min(case["deg_lo"], case["deg_hi"])
    elif graph == "power":
        case.update(gamma=round(rng.uniform(1.8, 2.6), 3), mean=round(mean, 2),
                    clip=max(8, rows // rng.choice([4, 8, 16])), shuffled=rng.random() < 0.5)
    else:
        block = rng.choice([128, 256, 512, 1024])
        case["rows"] = max(4, rows // block) * block
        inter = round(rng.uniform(0.1, 0.5) * mean, 2)
        case.update(block=block, p_intra=round(min(0.5, (mean - inter) / block), 5), inter=inter,
                    empty=0.05, single=0.05)
    if op in ("spmm", "sddmm"):
        case["sync"] = rng.random() < 0.3
    return case


# ------------------------------------------------------------------ graphs


def _weights(n, gamma, mean, clip, dev):
    """Chung-Lu weights c * i^(-1 / (gamma - 1)) cut at `clip`, c set for the mean."""
    base = torch.arange(1, n + 1, dtype=torch.float64, device=dev) ** (-1.0 / (gamma - 1.0))
    lo, hi = 1e-3, 1e13
    for _ in range(80):
        mid = math.sqrt(lo * hi)
        if float((mid * base).clamp(max=clip).mean()) < mean:
            lo = mid
        else:
            hi = mid
    return (hi * base).clamp(max=clip)


def _present(sorted_keys, keys):
    """Which of `keys` are among `sorted_keys`."""
    at = torch.searchsorted(sorted_keys, keys).clamp_(max=sorted_keys.numel() - 1)
    return sorted_keys[at] == keys


def _distinct(rows, cols, deg, sample):
    """Sorted keys row * cols + column, deg[r] distinct columns for row r.

    sample(row, k) draws a column for each row id of round k; a row's repeats
    are drawn again until it has its degree.
    """
    every = torch.arange(rows, device=deg.device)
    taken, missing, k = [], deg, 0
    while True:
        row = torch.repeat_interleave(every, missing)
        if row.numel() == 0:
            break
        new = torch.unique(row * cols + sample(row, k))
        for t in taken:
            new = new[~_present(t, new)]
        if new.numel():
            taken.append(new)
            missing = missing - torch.bincount(new // cols, minlength=rows)
        k += 1
    return torch.sort(torch.cat(taken)).values


def _degrees(case):
    """The rows' degrees (and the power law's weights): the case's own, whatever the seed.

    Worksets are made of whole rows' pieces, so every seed's outputs have one shape.
    """
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(977)
    rows = case["rows"]
    if case["graph"] == "uniform":
        return torch.randint(case["deg_lo"], case["deg_hi"] + 1, (rows,), generator=gen,
                             device=dev), None
    if case["graph"] == "power":
        w = _weights(rows, case["gamma"], case["mean"], case["clip"], dev)
        return torch.poisson(w, generator=gen).long().clamp_(max=rows // 2), w
    mean = case["p_intra"] * case["block"] + case["inter"]
    deg = torch.poisson(torch.full((rows,), mean, device=dev), generator=gen).long()
    u = torch.rand(rows, generator=gen, device=dev)
    deg[u < case["empty"]] = 0
    deg[(u >= case["empty"]) & (u < case["empty"] + case["single"])] = 1
    return deg.clamp_(max=rows // 2), None


def _graph(case, seed):
    """(rows, cols, row_ptr, col_ind, values) on the GPU: int32, int32, float32."""
    dev = torch.device("cuda")
    gen = torch.Generator(device=dev)
    gen.manual_seed(seed)
    rows = case["rows"]
    cols = case.get("cols", rows)
    deg, w = _degrees(case)

    def uniform(n, dtype=torch.float32):
        return torch.rand(n, generator=gen, device=dev, dtype=dtype)

    def anywhere(row):
        return torch.randint(0, cols, row.shape, generator=gen, device=dev)

    low = 0.0 if case["graph"] == "power" else -1.0
    if case["graph"] == "uniform":
        keys = _distinct(rows, cols, deg, lambda row, k: anywhere(row))
    elif case["graph"] == "power":
        # in whole numbers: a parallel sum of floats may round differently each time
        ends = torch.cumsum((w * 2.0**20).long(), 0)
        total = int(ends[-1])

        def by_weight(row, k):
            if k >= 40:  # rows that hold nearly all of the weight already
                return anywhere(row)
            u = (uniform(row.numel(), torch.float64) * total).long()
            return torch.searchsorted(ends, u, right=True)

        keys = _distinct(rows, cols, deg, by_weight)
        if case["shuffled"]:
            name = torch.randperm(rows, generator=gen, device=dev)
            keys = torch.sort(name[keys // cols] * cols + name[keys % cols]).values
    else:
        block = case["block"]
        share = case["inter"] / (case["p_intra"] * block + case["inter"])

        def near_or_far(row, k):
            near = row // block * block + torch.randint(0, block, row.shape, generator=gen,
                                                        device=dev)
            return torch.where(uniform(row.numel()) < share, anywhere(row), near)

        keys = _distinct(rows, cols, deg, near_or_far)
    row_ptr = torch.zeros(rows + 1, dtype=torch.int64, device=dev)
    row_ptr[1:] = torch.cumsum(torch.bincount(keys // cols, minlength=rows), 0)
    values = uniform(keys.numel()) * (1.0 - low) + low
    return rows, cols, row_ptr.int(), (keys % cols).int(), values


def _dense(case, seed, rows, cols):
    """The operands: B or Y (cols x N), and X (rows x N) for SDDMM. U(-1, 1)."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed ^ 0x5DEECE66D)
    y = torch.rand(cols, case["N"], generator=gen, device="cuda") * 2 - 1
    if case["op"] == "spmm":
        return y, None
    return y, torch.rand(rows, case["N"], generator=gen, device="cuda") * 2 - 1


# ------------------------------------------------------------------ a pass


class _View:
    """A device array of a matrix as torch takes it; keeps the matrix alive."""

    def __init__(self, owner, ptr, count, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (count,), "typestr": typestr,
                                         "data": (ptr, False), "version": 2, "strides": None}


def _view(owner, ptr, count, typestr, dtype):
    if count == 0:
        return torch.empty(0, dtype=dtype, device="cuda")
    return torch.as_tensor(_View(owner, ptr, count, typestr), device="cuda")


def _worksets(m):
    """(column ids, values, group rows) of every workset and the residue offsets and flags."""
    col, val, des = m.WorksetColInd(), m.WorksetSpData(), m.GroupDestination()
    num = m.GroupNum()
    nnz = m.MatrixNNZ()
    length = [0] + [num[s] * ps.GROUP_SIZE(s) for s in range(1, len(num))]
    length[0] = nnz - sum(length)
    out = [{"col": _view(m, col[s], length[s], "<i4", torch.int32),
            "val": _view(m, val[s], length[s], "<f4", torch.float32),
            "des": _view(m, des[s], num[s], "<i4", torch.int32)} for s in range(len(num))]
    return out, {"offset": _view(m, m.ResidueOffset(), num[0] + 1, "<i4", torch.int32),
                 "atomic": _view(m, m.ResidueAtomic(), num[0], "|u1", torch.uint8)}


def prepare(case, seed):
    ps.set_device(torch.cuda.current_device())
    rows, cols, rp, ci, v = _graph(case, seed)
    host = [a.cpu().numpy() for a in (rp, ci, v)]
    state = dict(case=case, rows=rows, cols=cols, host=host)
    del rp, ci, v
    torch.cuda.empty_cache()  # the matrix allocates beside torch's cache
    if case["op"] == "build":
        return state
    m = ps.PowerSparseMatrixGPU(rows, cols, host[1].size, *host,
                                csr_positions=case["op"] == "sddmm_csr")
    del state["host"]
    state["m"] = m
    state["y"], state["x"] = _dense(case, seed, rows, cols)
    if case["op"] == "spmm":
        state["out"] = torch.empty(rows, case["N"], device="cuda")
    elif case["op"] == "sddmm_csr":
        state["out"] = torch.empty(m.MatrixNNZ(), device="cuda")
    else:
        state["out"] = [torch.empty(n, device="cuda") for n in m.sddmm_output_sizes()]
    if case.get("sync"):
        state["streams"] = [ps.Stream() for _ in range(m.GroupTypeNum())]
    state["handles"] = dict(
        y=state["y"].data_ptr(), x=state["x"].data_ptr() if state["x"] is not None else 0,
        out=[t.data_ptr() for t in state["out"]] if case["op"] == "sddmm"
        else state["out"].data_ptr())
    return state


def run(state):
    case = state["case"]
    op, N = case["op"], case["N"]
    if op == "build":
        rp, ci, v = state["host"]
        m = ps.PowerSparseMatrixGPU(state["rows"], state["cols"], ci.size, rp, ci, v)
        worksets, residue = _worksets(m)
        return {"worksets": worksets, "residue": residue}
    m, out, h = state["m"], state["out"], state["handles"]
    # the caller clears what the operator adds to (C; the residue's scores)
    if op == "spmm":
        out.zero_()
        if "streams" in state:
            ps.SpMM(m, N, h["y"], h["out"], m.GroupTypeNum(), state["streams"])
        else:
            ps.SpMMAsync(m, N, h["y"], h["out"])
    elif op == "sddmm":
        out[0].zero_()
        if "streams" in state:
            ps.SDDMM(m, N, h["x"], h["y"], h["out"], m.GroupTypeNum(), state["streams"])
        else:
            ps.SDDMMAsync(m, N, h["x"], h["y"], h["out"])
    else:
        ps.SDDMMToCSR(m, N, h["x"], h["y"], h["out"])
    return out


# ------------------------------------------------------------------ what it takes


def _nnz(case):
    rows = case["rows"]
    if case["graph"] == "uniform":
        return rows * (case["deg_lo"] + case["deg_hi"]) / 2.0
    if case["graph"] == "power":
        return rows * case["mean"]
    full = case["p_intra"] * case["block"] + case["inter"]
    return rows * ((1.0 - case["empty"] - case["single"]) * full + case["single"])


def work(case):
    nnz, rows, cols, N = _nnz(case), case["rows"], case.get("cols", case["rows"]), case["N"]
    if case["op"] == "build":  # the CSR in, the worksets out (column, value; a row per group)
        return {"bytes": 16.0 * nnz + 8.0 * rows, "flops": 0.0}
    each = 8.0 if case["op"] == "spmm" else 12.0
    return {"bytes": each * nnz + 4.0 * (rows + 1) + 4.0 * N * (rows + cols),
            "flops": 2.0 * nnz * N}


def tolerance(case):
    if case["op"] == "build":
        return "exact"
    # 32-bit sums: rows of up to 1e5 terms (SpMM; two calls on one input, whose
    # atomic additions fall in another order, differ by rel 2.1e-7, max 2.6e-5)
    # and dot products of N terms (SDDMM; rel 1.6e-7 from 64 bits)
    return {"rel": 1e-6, "max": 1e-4}


def _dots(x, y, row, col, val):
    """val * <x[row], y[col]> in 64 bits, in pieces that bound the gathered rows to 4 GB."""
    out = torch.empty(row.numel(), dtype=torch.float64, device=x.device)
    step = max(1, (1 << 28) // x.shape[1])
    for b in range(0, row.numel(), step):
        e = b + step
        out[b:e] = (x[row[b:e]].double() * y[col[b:e]].double()).sum(1) * val[b:e].double()
    return out


def exact(case, seed):
    if case["op"] == "build":
        return None  # the worksets hold the input's own numbers, rearranged
    if case["op"] == "sddmm":
        # The order of the scores is the worksets', which are part of the
        # inputs here; the scores are plain torch in 64 bits.
        state = prepare(case, seed)
        worksets, residue = _worksets(state["m"])
        out = []
        for s, w in enumerate(worksets):
            des = w["des"].long()
            size = residue["offset"].long().diff() if s == 0 else \
                torch.full_like(des, ps.GROUP_SIZE(s))
            row = torch.repeat_interleave(des, size)
            out.append(_dots(state["x"], state["y"], row, w["col"].long(), w["val"]))
        return out
    rows, cols, rp, ci, v = _graph(case, seed)
    y, x = _dense(case, seed, rows, cols)
    row = torch.repeat_interleave(torch.arange(rows, device="cuda"), rp.long().diff())
    ci = ci.long()
    if case["op"] == "sddmm_csr":
        return _dots(x, y, row, ci, v)
    out = torch.zeros(rows, case["N"], dtype=torch.float64, device="cuda")
    step = max(1, (1 << 28) // case["N"])
    for b in range(0, row.numel(), step):
        e = b + step
        out.index_add_(0, row[b:e], y[ci[b:e]].double() * v[b:e, None].double())
    return out
