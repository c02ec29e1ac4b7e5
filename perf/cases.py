"""Timed cases of the sparse operators: one per way a program uses them.

``listed()`` gives the fixed cases, ``draw(rng)`` further ones of the same
ranges.  A case names an operator (``op``), a matrix family and its size, the
dtypes and the dense width; ``prepare`` makes its inputs on the GPU from a
seed, ``run`` makes one call, ``work`` counts the bytes and operations that
call cannot do without and ``exact`` computes the same outputs in fp64 with
torch alone.

Matrix families:
  * poisson  -- n * mean entries at uniform rows and columns (graphs without
    structure, random meshes);
  * powerlaw -- row lengths ~ l^-2 on [1, 1e5] (web and social graphs);
  * banded   -- 7 diagonals plus (mean - 7) random columns per row (stencils
    with long-range couplings).
Values, vectors and dense operands are uniform in [-1, 1).
"""

import math

import torch

from flagsparse_public_amd import (
    flagsparse_sddmm_csr,
    flagsparse_spmm_coo,
    flagsparse_spmm_csr,
    flagsparse_spmm_csr_opt,
    flagsparse_spmv_coo,
    flagsparse_spmv_csr,
    prepare_sddmm_csr,
    prepare_spmm_csr_opt,
    prepare_spmv_csr,
)
from flagsparse_public_amd.batched import BatchedCsr

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32,
          "f64": torch.float64, "c64": torch.complex64}
INDEX = {"i32": torch.int32, "i64": torch.int64}
MAX_ROW = 100_000  # longest row of the power-law family


def listed():
    return [
        # a small system inside a solver loop: the matrix prepared once, launch latency counts
        {"name": "spmv_small_f32", "op": "spmv", "matrix": "poisson", "n": 16_384, "mean": 16,
         "dtype": "f32", "index": "i32", "mode": "opt", "trans": "non"},
        # the largest: an iterative method (PageRank, power iteration) on a web-like graph
        {"name": "spmv_powerlaw_f32", "op": "spmv", "matrix": "powerlaw", "n": 4_000_000,
         "mean": 12, "dtype": "f32", "index": "i32", "mode": "opt", "trans": "non"},
        # the adjoint product of a complex operator (A^H x), prepared, default accumulation
        {"name": "spmv_adjoint_c64", "op": "spmv", "matrix": "poisson", "n": 400_003, "mean": 18,
         "dtype": "c64", "index": "i32", "mode": "default", "trans": "conj"},
        # the plain operator call on CSR arrays, nothing prepared by the caller, double precision
        {"name": "spmv_call_f64", "op": "spmv_call", "matrix": "banded", "n": 300_007, "mean": 15,
         "dtype": "f64", "index": "i32", "mode": "default", "trans": "non"},
        # unsorted triplets as an assembly loop leaves them, one product
        {"name": "spmv_coo_f32", "op": "spmv_coo", "matrix": "poisson", "n": 150_001, "mean": 12,
         "dtype": "f32", "index": "i32"},
        # many right-hand sides on a large stencil-like matrix, prepared
        {"name": "spmm_prepared_f32", "op": "spmm_prepared", "matrix": "banded", "n": 1_048_576,
         "mean": 15, "dtype": "f32", "index": "i32", "cols": 64},
        # a block of eight vectors (block Krylov) in double precision, prepared
        {"name": "spmm_prepared_f64", "op": "spmm_prepared", "matrix": "poisson", "n": 200_000,
         "mean": 24, "dtype": "f64", "index": "i32", "cols": 8},
        # a graph layer's aggregation with an odd output width, torch's own int64 CSR arrays
        {"name": "spmm_call_f32", "op": "spmm_call", "matrix": "powerlaw", "n": 170_000,
         "mean": 12, "dtype": "f32", "index": "i64", "cols": 47},
        # the same aggregation in half precision at a hidden width of 128
        {"name": "spmm_call_bf16", "op": "spmm_call", "matrix": "poisson", "n": 250_000,
         "mean": 20, "dtype": "bf16", "index": "i32", "cols": 128},
        # aggregation over an edge list in arrival order
        {"name": "spmm_coo_f32", "op": "spmm_coo", "matrix": "poisson", "n": 100_000, "mean": 16,
         "dtype": "f32", "index": "i64", "cols": 32},
        # edge scores of graph attention (and the gradient of an SpMM's values)
        {"name": "sddmm_f32", "op": "sddmm", "matrix": "poisson", "n": 200_003, "mean": 16,
         "dtype": "f32", "index": "i32", "cols": 64},
        # a batch of uneven matrices, one SpMV and one 8-column SpMM each
        {"name": "batched_f32", "op": "batched", "matrix": "poisson", "n": 200_000, "count": 32,
         "mean": 34, "dtype": "f32", "index": "i32", "cols": 8},
    ]


def draw(rng):
    op = rng.choice(("spmv", "spmv", "spmv_call", "spmv_coo", "spmm_prepared", "spmm_call",
                     "spmm_call", "spmm_coo", "sddmm", "batched"))
    n = int(round(math.exp(rng.uniform(math.log(2_000), math.log(1_000_000)))))
    family = rng.choice(("poisson", "powerlaw", "banded"))
    mean = {"poisson": rng.randint(3, 40), "powerlaw": 12, "banded": rng.randint(8, 24)}[family]
    case = {"op": op, "matrix": family, "n": n, "mean": mean,
            "index": rng.choice(("i32", "i32", "i64"))}
    if op in ("spmv", "spmv_call"):
        case["dtype"] = rng.choice(("f32", "f32", "f64", "f16", "bf16", "c64"))
        case["mode"] = rng.choice(("opt", "default"))
        case["trans"] = rng.choice(("non", "non", "trans")) if op == "spmv" else "non"
    elif op == "spmv_coo":
        case["dtype"] = rng.choice(("f32", "f64", "c64"))
    elif op == "spmm_prepared" or op == "sddmm":
        case["dtype"] = rng.choice(("f32", "f32", "f64"))
    elif op == "batched":
        case["dtype"] = "f32"
        case["count"] = rng.randint(4, 32)
        case["n"] = min(n, 200_000)
        case["matrix"], case["mean"], case["index"] = "poisson", rng.randint(4, 34), "i32"
    else:
        case["dtype"] = rng.choice(("f32", "f32", "f64", "bf16", "f16", "c64"))
    if op == "sddmm":
        case["index"] = "i32"
    if op in ("spmm_prepared", "spmm_call", "spmm_coo", "sddmm"):
        case["cols"] = rng.choice((3, 8, 16, 32, 40, 64, 100, 128, rng.randint(1, 160)))
    if op == "batched":
        case["cols"] = rng.choice((4, 8, 16, rng.randint(1, 16)))
    # no larger than the largest listed case
    while work(case)["bytes"] > 4e8 or work(case)["flops"] > 1.5e9:
        case["n"] = int(case["n"] * 0.7)
    return case


# ------------------------------------------------------------------ inputs

def _gen(seed, device):
    g = torch.Generator(device=device)
    g.manual_seed(int(seed))
    return g


def _uniform(shape, dtype, g, device):
    if dtype.is_complex:
        return torch.view_as_complex(torch.rand((*shape, 2), generator=g, device=device) * 2 - 1)
    wide = torch.float64 if dtype == torch.float64 else torch.float32
    return (torch.rand(shape, generator=g, device=device, dtype=wide) * 2 - 1).to(dtype)


def _entries(family, n, mean, g, device):
    """(rows, columns) of the entries, int64, sorted by row and column."""
    if family == "powerlaw":  # the quantiles of the length distribution in random order
        u = (torch.randperm(n, generator=g, device=device).double() + 0.5) / n
        lens = torch.ceil(1.0 / (1.0 - u * (1.0 - 1.0 / min(n, MAX_ROW)))).long()
        rows = torch.repeat_interleave(torch.arange(n, device=device), lens.clamp_(1, n))
    elif family == "poisson":  # entries thrown into the rows at random: Poisson row lengths
        rows = torch.randint(0, n, (n * mean,), generator=g, device=device)
    else:
        rows = torch.arange(n, device=device).repeat_interleave(mean - 7)
    cols = torch.randint(0, n, (rows.numel(),), generator=g, device=device)
    if family == "banded":
        r = torch.arange(n, device=device)
        band = r[:, None] + torch.arange(-3, 4, device=device)[None, :]
        keep = (band >= 0) & (band < n)
        rows = torch.cat([rows, r[:, None].expand_as(band)[keep]])
        cols = torch.cat([cols, band[keep]])
    key = torch.sort(rows * n + cols)[0]
    rows = torch.div(key, n, rounding_mode="floor")
    return rows, key - rows * n


def _csr(case, n, g, device):
    index = INDEX[case["index"]]
    rows, cols = _entries(case["matrix"], n, case["mean"], g, device)
    indptr = torch.zeros(n + 1, dtype=torch.int64, device=device)
    torch.cumsum(torch.bincount(rows, minlength=n), 0, out=indptr[1:])
    values = _uniform((rows.numel(),), DTYPES[case["dtype"]], g, device)
    return values, cols.to(index), indptr.to(index)


def _inputs(case, seed, device):
    """The tensors a program holds before the call."""
    g = _gen(seed, device)
    op, n, dtype = case["op"], case["n"], DTYPES[case["dtype"]]
    if op == "batched":
        mats = []
        for k in range(case["count"]):
            # sizes log-uniform over two decades, the largest last
            m = max(50, int(n * 0.005 ** (1.0 - (k + 1) / case["count"])))
            values, cols, indptr = _csr(case, m, g, device)
            mats.append({"data": values, "indices": cols, "indptr": indptr, "shape": (m, m),
                         "x": _uniform((m,), dtype, g, device),
                         "B": _uniform((m, case["cols"]), dtype, g, device)})
        return mats
    if op in ("spmv_coo", "spmm_coo"):
        rows, cols = _entries(case["matrix"], n, case["mean"], g, device)
        order = torch.randperm(rows.numel(), generator=g, device=device)
        index = INDEX[case["index"]]
        s = {"data": _uniform((rows.numel(),), dtype, g, device), "row": rows[order].to(index),
             "col": cols[order].to(index)}
    else:
        values, cols, indptr = _csr(case, n, g, device)
        s = {"data": values, "indices": cols, "indptr": indptr}
    s["shape"] = (n, n)
    if op == "sddmm":
        del s["data"]
        s["x"] = _uniform((n, case["cols"]), dtype, g, device)
        s["y"] = _uniform((n, case["cols"]), dtype, g, device)
    elif op in ("spmv", "spmv_call", "spmv_coo"):
        s["x"] = _uniform((n,), dtype, g, device)
    else:
        s["B"] = _uniform((n, case["cols"]), dtype, g, device)
    return s


def prepare(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    op, s = case["op"], _inputs(case, seed, device)
    if op == "batched":
        return {"op": op, "batch": BatchedCsr(s)}
    if op == "spmv":
        p = prepare_spmv_csr(s["data"], s["indices"], s["indptr"], s["shape"], op=case["trans"])
        return {"op": op, "prepared": p, "x": s["x"], "opt": case["mode"] == "opt"}
    if op == "spmm_prepared":
        p = prepare_spmm_csr_opt(s["data"], s["indices"], s["indptr"], s["shape"])
        return {"op": op, "prepared": p, "B": s["B"]}
    if op == "sddmm":
        p = prepare_sddmm_csr(s["indices"], s["indptr"], s["shape"], k_hint=case["cols"])
        return {"op": op, "prepared": p, "x": s["x"], "y": s["y"]}
    s["op"] = op
    s["opt"] = case.get("mode") == "opt"
    return s


def run(state):
    s, op = state, state["op"]
    if op == "spmv":
        return flagsparse_spmv_csr(x=s["x"], prepared=s["prepared"], use_opt=s["opt"])
    if op == "spmv_call":
        return flagsparse_spmv_csr(s["data"], s["indices"], s["indptr"], s["x"], s["shape"],
                                   use_opt=s["opt"])
    if op == "spmv_coo":
        return flagsparse_spmv_coo(s["data"], s["row"], s["col"], s["x"], s["shape"])
    if op == "spmm_prepared":
        return flagsparse_spmm_csr_opt(B=s["B"], prepared=s["prepared"])
    if op == "spmm_call":
        return flagsparse_spmm_csr(s["data"], s["indices"], s["indptr"], s["B"], s["shape"])
    if op == "spmm_coo":
        return flagsparse_spmm_coo(s["data"], s["row"], s["col"], s["B"], s["shape"])
    if op == "sddmm":
        return flagsparse_sddmm_csr(x=s["x"], y=s["y"], prepared=s["prepared"])
    s["batch"].run()
    return {"y": s["batch"].y, "C": s["batch"].C}


# -------------------------------------------------------------------- work

def _mean_row(case, n):
    if case["matrix"] == "powerlaw":  # of ceil(l), density ~ l^-2 on [1, max]
        return math.log(min(n, MAX_ROW)) + 0.58
    return float(case["mean"])


def _work_of(case, n):
    item = torch.empty(0, dtype=DTYPES[case["dtype"]]).element_size()
    idx = 4 if case["index"] == "i32" else 8
    nnz, op = n * _mean_row(case, n), case["op"]
    mul = 8.0 if case["dtype"] == "c64" else 2.0
    width = case.get("cols", 1)
    matrix = nnz * (2 * idx + item) if op.endswith("coo") else nnz * (idx + item) + (n + 1) * idx
    if op == "sddmm":  # pattern and both operands read, one value per entry written
        return (n + 1) * idx + nnz * (idx + item) + 2 * n * width * item, mul * nnz * width
    if op == "batched":  # one SpMV and one SpMM over the same matrix
        return matrix + 2 * n * (width + 1) * item, mul * nnz * (width + 1)
    return matrix + 2 * n * width * item, mul * nnz * width


def work(case):
    if case["op"] != "batched":
        b, f = _work_of(case, case["n"])
        return {"bytes": b, "flops": f}
    sizes = [max(50, int(case["n"] * 0.005 ** (1.0 - (k + 1) / case["count"])))
             for k in range(case["count"])]
    each = [_work_of(case, m) for m in sizes]
    return {"bytes": sum(e[0] for e in each), "flops": sum(e[1] for e in each)}


# ------------------------------------------------------------------- exact

def _sum_rows(indptr, terms):
    """Sums of the rows' terms ([nnz, k] fp64), one row after another."""
    return torch.segment_reduce(terms, "sum", offsets=indptr.long(), axis=0, initial=0.0)


def _product(values, cols, indptr, dense):
    """A @ dense in fp64, a few columns of the dense operand at a time."""
    width = max(1, int(2e8 // max(values.numel(), 1)))
    out = []
    for k in range(0, dense.shape[1], width):
        terms = values[:, None] * dense[:, k:k + width][cols]
        if terms.is_complex():
            sums = _sum_rows(indptr, torch.view_as_real(terms).flatten(1))
            out.append(torch.view_as_complex(sums.unflatten(1, (-1, 2))))
        else:
            out.append(_sum_rows(indptr, terms))
    return torch.cat(out, 1)


def exact(case, seed):
    device = torch.device("cuda", torch.cuda.current_device())
    op, s = case["op"], _inputs(case, seed, device)
    wide = torch.complex128 if DTYPES[case["dtype"]].is_complex else torch.float64
    if op == "batched":
        y, C = [], []
        for m in s:
            both = _product(m["data"].to(wide), m["indices"].long(), m["indptr"],
                            torch.cat([m["x"][:, None], m["B"]], 1).to(wide))
            y.append(both[:, 0].contiguous())
            C.append(both[:, 1:].contiguous())
        return {"y": y, "C": C}
    if op == "sddmm":
        lens = s["indptr"][1:] - s["indptr"][:-1]
        rows = torch.repeat_interleave(torch.arange(case["n"], device=device), lens.long())
        step = 1 << 20
        return torch.cat([(s["x"][rows[k:k + step]].to(wide)
                           * s["y"][s["indices"][k:k + step].long()].to(wide)).sum(1)
                          for k in range(0, rows.numel(), step)])
    values = s["data"].to(wide)
    dense = s["x"][:, None] if "x" in s else s["B"]
    if op in ("spmv_coo", "spmm_coo"):
        rows, cols = s["row"].long(), s["col"].long()
    else:
        lens = s["indptr"][1:] - s["indptr"][:-1]
        rows = torch.repeat_interleave(torch.arange(case["n"], device=device), lens.long())
        cols = s["indices"].long()
    if case.get("trans", "non") != "non":
        rows, cols = cols, rows
        values = values.conj().resolve_conj() if case["trans"] == "conj" else values
    order = torch.sort(rows, stable=True)[1]
    indptr = torch.zeros(case["n"] + 1, dtype=torch.int64, device=device)
    torch.cumsum(torch.bincount(rows, minlength=case["n"]), 0, out=indptr[1:])
    out = _product(values[order], cols[order], indptr, dense.to(wide))
    return out[:, 0].contiguous() if "x" in s else out
