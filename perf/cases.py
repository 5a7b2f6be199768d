"""The calls whose speed matters, as data: what a program does with the sparse products.

Two ways of calling are in use and both are here: a matrix prepared once and multiplied many
times (solvers, propagation, attention over a fixed pattern), and a plain call with the arrays
of a matrix that was just built (assembly loops, sampled graphs, one product per matrix), which
pays for its own checks, ordering and planning every time.

A case is a dict of plain values; ``op`` names the entry point, ``pattern`` how the non-zeros
lie, ``prepared`` which way of calling.  Everything is made on the GPU from the seed.
"""

import torch

import flagsparse_amd as fs

_DTYPES = {"f32": torch.float32, "f64": torch.float64}
_INDEX = {"i32": torch.int32, "i64": torch.int64}
_BAND = 512  # columns of the band of pattern "band": half of a row's entries lie in it


def listed():
    return [
        # one step of an iterative solver on a small system: latency and launches are all of it
        {"name": "spmv_small", "op": "spmv_csr", "prepared": True, "pattern": "regular",
         "rows": 4096, "cols": 4096, "mean": 16, "dtype": "f32", "index": "i32", "opt": False},
        # conjugate gradients on a 5-point stencil: the double precision stream
        {"name": "spmv_stencil", "op": "spmv_csr", "prepared": True, "pattern": "stencil",
         "rows": 2048 * 2048, "cols": 2048 * 2048, "mean": 5, "dtype": "f64", "index": "i32",
         "opt": False},
        # propagation over a web-like graph, the headline size: short rows, a few huge ones
        {"name": "spmv_powerlaw", "op": "spmv_csr", "prepared": True, "pattern": "powerlaw",
         "rows": 8 << 20, "cols": 8 << 20, "mean": 12, "dtype": "f32", "index": "i64",
         "opt": False},
        # the same kind of graph, smaller, multiplied once with no prepared object
        {"name": "spmv_call_powerlaw", "op": "spmv_csr", "prepared": False,
         "pattern": "powerlaw", "rows": 1000003, "cols": 1000003, "mean": 12, "dtype": "f32",
         "index": "i64", "opt": False},
        # COO triplets sorted by row, prepared once
        {"name": "coo_spmv_uniform", "op": "spmv_coo", "prepared": True, "pattern": "random",
         "rows": 2 << 20, "cols": 2 << 20, "mean": 20, "dtype": "f32", "index": "i32",
         "sorted": True},
        # triplets as an assembly leaves them (any order, repeats), multiplied once
        {"name": "coo_spmv_call_unsorted", "op": "spmv_coo", "prepared": False,
         "pattern": "random", "rows": 150001, "cols": 120007, "mean": 11, "dtype": "f64",
         "index": "i64", "sorted": False},
        # feature propagation on a large graph, half of each row near the diagonal
        {"name": "spmm_opt_n64", "op": "spmm_csr_opt", "prepared": True, "pattern": "band",
         "rows": 1 << 20, "cols": 1 << 20, "mean": 32, "dtype": "f32", "index": "i32", "n": 64},
        # the output layer of a graph network: a skewed graph, a class count for a width
        {"name": "spmm_opt_n47", "op": "spmm_csr_opt", "prepared": True, "pattern": "powerlaw",
         "rows": 200003, "cols": 200003, "mean": 24, "dtype": "f32", "index": "i32", "n": 47},
        # one product with a matrix that was just sampled, float32 summed in float64
        {"name": "spmm_call_n16", "op": "spmm_csr", "prepared": False, "pattern": "ragged",
         "rows": 100003, "cols": 90001, "mean": 16, "dtype": "f32", "index": "i64", "n": 16},
        # the same from unsorted triplets with repeats
        {"name": "coo_spmm_call_n32", "op": "spmm_coo", "prepared": False, "pattern": "random",
         "rows": 60013, "cols": 50021, "mean": 20, "dtype": "f32", "index": "i64", "n": 32,
         "sorted": False},
        # attention scores on a fixed pattern
        {"name": "sddmm_k64", "op": "sddmm", "prepared": True, "pattern": "band",
         "rows": 1 << 20, "cols": 1 << 20, "mean": 32, "dtype": "f32", "index": "i32", "k": 64,
         "scaled": False},
        # a sampled residual alpha x y^T + beta data, double precision, the pattern used once
        {"name": "sddmm_call_k50", "op": "sddmm", "prepared": False, "pattern": "powerlaw",
         "rows": 40009, "cols": 50021, "mean": 24, "dtype": "f64", "index": "i32", "k": 50,
         "scaled": True},
    ]


def _log_int(rng, lo, hi):
    """An integer of [lo, hi], even on a logarithmic scale."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random()))))


def draw(rng):
    """One more case of the ranges above: sizes from a thousand rows to the listed ones, any
    width, both value and index types.  The caps keep a draw below the largest listed case."""
    op = rng.choice(["spmv_csr", "spmv_csr", "spmv_coo", "spmm_csr_opt", "spmm_csr", "spmm_coo",
                     "sddmm"])
    prepared = {"spmm_csr_opt": True, "spmm_csr": False, "spmm_coo": False}.get(
        op, rng.random() < 0.5)
    case = {"op": op, "prepared": prepared, "dtype": rng.choice(["f32", "f32", "f64"]),
            "index": rng.choice(["i32", "i64"])}
    mean = _log_int(rng, 3, 60)
    if op in ("spmv_csr", "spmv_coo"):
        rows = _log_int(rng, 1000, 4000000)
        cap = 48000000 if prepared else 12000000
    else:
        rows = _log_int(rng, 1000, 1000000)
        width = _log_int(rng, 1, 256)
        cap = min(32000000 if prepared else 6000000, (1 << 30) // width)
        case["k" if op == "sddmm" else "n"] = width
    case["mean"] = mean
    case["rows"] = rows = max(1000, min(rows, cap // mean))
    case["cols"] = rows if rng.random() < 0.5 else _log_int(rng, max(512, rows // 4), 2 * rows)
    if op in ("spmv_coo", "spmm_coo"):
        case["pattern"] = "random"
        case["sorted"] = rng.random() < 0.5
    else:
        case["pattern"] = rng.choice(["regular", "ragged", "powerlaw", "band", "random"])
        if op == "spmv_csr" and rng.random() < 0.2:
            side = max(32, int(rows ** 0.5))
            case.update(pattern="stencil", rows=side * side, cols=side * side, mean=5)
    if op == "spmv_csr":
        case["opt"] = rng.random() < 0.5
    if op == "sddmm":
        case["index"] = "i32"  # the only index type the entry point takes
        case["scaled"] = rng.random() < 0.5
    return case


# ------------------------------------------------------------------------------------------
# Inputs
# ------------------------------------------------------------------------------------------


def _lengths(case, gen):
    """Entries per row of the patterns that are built row by row; rows * mean in all."""
    n, mean = case["rows"], case["mean"]
    pattern = case["pattern"]
    if pattern == "ragged":  # 0 .. 2 * mean, empty rows among them
        half = torch.randint(0, 2 * mean + 1, (n // 2,), generator=gen, device="cuda")
        middle = torch.full((n % 2,), mean, dtype=torch.int64, device="cuda")
        return torch.cat([half, middle, 2 * mean - half.flip(0)])
    if pattern != "powerlaw":
        return torch.full((n,), mean, dtype=torch.int64, device="cuda")
    # min(ceil(c Z), cap) with Z Pareto-like of exponent 1.8, c fitted to the mean
    u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64).clamp_min_(1e-12)
    z = torch.floor(u.pow(-1.0 / 0.8))
    cap = min(200000, case["cols"] // 4)
    lo, hi = 0.0, float(2 * mean)
    for _ in range(40):
        mid = 0.5 * (lo + hi)
        if float(torch.ceil(mid * z).clamp_(max=cap).sum()) <= float(mean) * n:
            lo = mid
        else:
            hi = mid
    length = torch.ceil(lo * z).clamp_(max=cap).to(torch.int64)
    short = mean * n - int(length.sum())
    while short > 0:  # the few entries left over, one to a row
        rows = torch.nonzero(length < cap).flatten()[:short]
        length[rows] += 1
        short -= rows.numel()
    return length


def _spread(gen, k, parts, span):
    """A column of the k-th of ``parts`` equal pieces of [0, span): distinct and rising in k."""
    lo = k * span // parts
    width = (k + 1) * span // parts - lo
    u = torch.rand(k.numel(), generator=gen, device="cuda", dtype=torch.float64)
    return lo + (u * width).to(torch.int64)


def _stencil(case):
    side = int(round(case["rows"] ** 0.5))
    i = torch.arange(side * side, dtype=torch.int64, device="cuda")
    r, c = i // side, i % side
    valid = torch.stack([r > 0, c > 0, r >= 0, c < side - 1, r < side - 1], 1)
    cols = (i[:, None] + torch.tensor([-side, -1, 0, 1, side], device="cuda")[None, :])[valid]
    return i[:, None].expand(-1, 5)[valid], cols


def _entries(case, gen):
    """(row, col) int64, in the order the case supplies them."""
    n, cols, mean = case["rows"], case["cols"], case["mean"]
    if case["pattern"] == "stencil":
        return _stencil(case)
    if case["pattern"] == "random":  # independent draws, repeats possible
        nnz = n * mean
        row = torch.randint(0, n, (nnz,), generator=gen, device="cuda")
        col = torch.randint(0, cols, (nnz,), generator=gen, device="cuda")
        if case.get("sorted"):
            key = torch.sort(row * cols + col).values
            return key // cols, key % cols
        if "sorted" in case:
            return row, col
        return torch.sort(row).values, col  # CSR: rows in order, columns as drawn
    length = _lengths(case, gen)
    row = torch.repeat_interleave(torch.arange(n, device="cuda"), length)
    length = length[row]
    k = torch.arange(row.numel(), device="cuda") - torch.searchsorted(row, row)
    if case["pattern"] != "band":
        return row, _spread(gen, k, length, cols)
    near = length // 2  # a row's first half: a window about its diagonal position
    width = min(_BAND, cols)
    start = (row * cols // n - width // 2).clamp_(0, cols - width)
    inside = start + _spread(gen, k, near.clamp_min(1), width)
    col = torch.where(k < near, inside, _spread(gen, k - near, length - near, cols))
    key = torch.sort(row * cols + col.clamp_(0, cols - 1)).values
    return key // cols, key % cols


def _values(gen, dtype, *size):
    return torch.randn(*size, generator=gen, device="cuda", dtype=dtype)


def _inputs(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    dtype = _DTYPES[case["dtype"]]
    row, col = _entries(case, gen)
    s = {"row": row, "col": col, "shape": (case["rows"], case["cols"]),
         "data": _values(gen, dtype, row.numel())}
    op = case["op"]
    if op in ("spmv_csr", "spmv_coo"):
        s["x"] = _values(gen, dtype, case["cols"])
    elif op == "sddmm":
        s["x"] = _values(gen, dtype, case["rows"], case["k"])
        s["y"] = _values(gen, dtype, case["cols"], case["k"])
    else:
        s["B"] = _values(gen, dtype, case["cols"], case["n"])
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    index = _INDEX[case["index"]]
    op, shape = case["op"], s["shape"]
    row, col = s.pop("row"), s.pop("col")
    if op in ("spmv_coo", "spmm_coo"):
        s["row"], s["col"] = row.to(index), col.to(index)
        if case["prepared"]:
            s["plan"] = fs.prepare_spmv_coo(s["data"], s["row"], s["col"], shape)
    else:
        bounds = torch.arange(case["rows"] + 1, device="cuda")
        s["indptr"] = torch.searchsorted(row, bounds).to(index)
        s["indices"] = col.to(index)
        if case["prepared"]:
            if op == "spmv_csr":
                s["plan"] = fs.prepare_spmv_csr(s["data"], s["indices"], s["indptr"], shape)
            elif op == "spmm_csr_opt":
                s["plan"] = fs.prepare_spmm_csr_opt(s["data"], s["indices"], s["indptr"], shape)
            else:
                s["plan"] = fs.prepare_sddmm_csr(s["indices"], s["indptr"], shape,
                                                 k_hint=case["k"])
    s["case"] = case
    return s


# ------------------------------------------------------------------------------------------
# The pass, its work and its accuracy
# ------------------------------------------------------------------------------------------


def run(s):
    case = s["case"]
    op = case["op"]
    if op == "spmv_csr":
        if case["prepared"]:
            return fs.flagsparse_spmv_csr(x=s["x"], prepared=s["plan"], use_opt=case["opt"])
        return fs.flagsparse_spmv_csr(s["data"], s["indices"], s["indptr"], s["x"], s["shape"],
                                      use_opt=case["opt"])
    if op == "spmv_coo":
        if case["prepared"]:
            return fs.flagsparse_spmv_coo(x=s["x"], prepared=s["plan"])
        return fs.flagsparse_spmv_coo(s["data"], s["row"], s["col"], s["x"], s["shape"])
    if op == "spmm_csr_opt":
        return fs.flagsparse_spmm_csr_opt(B=s["B"], prepared=s["plan"])
    if op == "spmm_csr":
        return fs.flagsparse_spmm_csr(s["data"], s["indices"], s["indptr"], s["B"], s["shape"])
    if op == "spmm_coo":
        return fs.flagsparse_spmm_coo(s["data"], s["row"], s["col"], s["B"], s["shape"])
    scaled = {"data": s["data"], "alpha": 0.5, "beta": 2.0} if case["scaled"] else {}
    if case["prepared"]:
        return fs.flagsparse_sddmm_csr(x=s["x"], y=s["y"], prepared=s["plan"], **scaled)
    return fs.flagsparse_sddmm_csr(indices=s["indices"], indptr=s["indptr"], x=s["x"], y=s["y"],
                                   shape=s["shape"], **scaled)


def work(case):
    """Each array once: a prepared matrix at the width its columns need (four bytes), a plain
    call at the widths supplied."""
    v = 4 if case["dtype"] == "f32" else 8
    i = 8 if case["index"] == "i64" and not case["prepared"] else 4
    n, cols = case["rows"], case["cols"]
    nnz = n * case["mean"]
    op = case["op"]
    rows = nnz * i if op in ("spmv_coo", "spmm_coo") and not case["prepared"] else (n + 1) * i
    index = nnz * i + rows
    if op in ("spmv_csr", "spmv_coo"):
        return {"bytes": nnz * v + index + (n + cols) * v, "flops": 2 * nnz}
    if op == "sddmm":
        k = case["k"]
        return {"bytes": index + nnz * v * (2 if case["scaled"] else 1) + (n + cols) * k * v,
                "flops": 2 * nnz * k}
    return {"bytes": nnz * v + index + (n + cols) * case["n"] * v, "flops": 2 * nnz * case["n"]}


def tolerance(case):
    """Four times the error against exact() that was measured.  Sums of float32 taken in
    float64 and rounded once (default CSR SpMV, base and COO SpMM): 2.5e-8, half an ulp.  Sums
    taken in the values' own type: 4e-8 to 2.4e-7 in float32, 5e-17 to 5e-16 in float64, the
    largest of each where a power law's rows are long."""
    if case["dtype"] == "f64":
        return {"rel": 2e-15}
    op = case["op"]
    once = op in ("spmm_csr", "spmm_coo") or (op == "spmv_csr" and not case["opt"])
    return {"rel": 1e-7 if once else 1e-6}


def exact(case, seed):
    s = _inputs(case, seed)
    row, col, op = s["row"], s["col"], case["op"]
    data = s["data"].double()
    if op in ("spmv_csr", "spmv_coo"):
        out = torch.zeros(case["rows"], dtype=torch.float64, device="cuda")
        return out.index_add_(0, row, data * s["x"].double()[col])
    step = 1 << 21
    if op == "sddmm":
        x, y = s["x"].double(), s["y"].double()
        out = torch.empty(row.numel(), dtype=torch.float64, device="cuda")
        for a in range(0, row.numel(), step):
            b = a + step
            out[a:b] = (x[row[a:b]] * y[col[a:b]]).sum(1)
        return 0.5 * out + 2.0 * data if case["scaled"] else out
    B = s["B"].double()
    out = torch.zeros(case["rows"], case["n"], dtype=torch.float64, device="cuda")
    for a in range(0, row.numel(), step):
        b = a + step
        out.index_add_(0, row[a:b], data[a:b, None] * B[col[a:b]])
    return out
