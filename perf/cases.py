"""The performance cases of this library: the work its users have it do, through the public entry points.

listed() names the cases, draw() gives further ones of the same ranges.  prepare() makes, on the GPU and from the seed
alone, what a program holds before the call: the matrix, the operands, the handle and descriptors, the buffer of the
size the library asks for and, where a program would make it, the preprocess call.  run() is one pass.
"""
import functools
import math

import numpy as np
import torch

from mcsparse_amd import api

# A case is a task on a matrix:
#   task    spmv, spmm, csr2csc, csr2coo or assemble
#   matrix  laplacian  5-point stencil on a grid x by y (values 4 / -1)
#           stencil    27-point stencil on a grid x by y by z, values U[-1, 1]
#           uniform    per_row distinct, sorted, uniformly drawn columns in every row, values N(0, 1)
#           powerlaw   row lengths of a Zipf law (exponent 1.8, at most longest), distinct sorted uniform columns,
#                      values U[-1, 1]
#           mesh       (assemble) the 16 triples of every four-node element of a mesh of x by y elements, element by element
#           edges      (assemble) nnz triples, each with a uniformly drawn row and column
#   dtype   float32 or float64
_POWERLAW_EXPONENT = 1.8

_LISTED = [
    # The smallest call: one product with the matrix of a 512 x 512 grid inside an iteration whose matrix changes from
    # step to step (no preprocess call).  What it costs is mostly the call: host work, one launch, one pass of latencies.
    {"name": "spmv-laplacian-small", "task": "spmv", "matrix": "laplacian", "x": 512, "y": 512, "dtype": "float32",
     "op": "N", "prepared": False, "alpha": 1.0, "beta": 0.0},
    # Conjugate gradients on a three-dimensional finite-element or finite-difference matrix: double precision, a
    # preprocess call before the loop, a grid whose sides are no round numbers.
    {"name": "spmv-stencil-f64-prepared", "task": "spmv", "matrix": "stencil", "x": 101, "y": 97, "z": 89,
     "dtype": "float64", "op": "N", "prepared": True, "alpha": 1.0, "beta": 0.0},
    # An unstructured matrix with equal rows under an iterative solver: y = alpha A x + beta y with A prepared once
    # (the headline configuration of bench.py).
    {"name": "spmv-uniform-f64-prepared", "task": "spmv", "matrix": "uniform", "rows": 1 << 20, "per_row": 16,
     "dtype": "float64", "op": "N", "prepared": True, "alpha": 1.5, "beta": 0.5},
    # The same product by a program that knows the buffer-size and compute calls only.
    {"name": "spmv-uniform-f64-direct", "task": "spmv", "matrix": "uniform", "rows": 1 << 20, "per_row": 16,
     "dtype": "float64", "op": "N", "prepared": False, "alpha": 1.5, "beta": 0.5},
    # A graph's matrix applied again and again (ranking, propagation): a few rows of 10^5 and many of one nonzero.
    {"name": "spmv-powerlaw-f32-prepared", "task": "spmv", "matrix": "powerlaw", "rows": 1 << 22, "longest": 200000,
     "dtype": "float32", "op": "N", "prepared": True, "alpha": 1.0, "beta": 0.0},
    # The transposed product with a matrix whose values change between calls: no preprocess call.
    {"name": "spmv-powerlaw-f32-transposed", "task": "spmv", "matrix": "powerlaw", "rows": 1 << 22, "longest": 200000,
     "dtype": "float32", "op": "T", "prepared": False, "alpha": 1.0, "beta": 0.0},
    # A stencil applied to a block of 64 vectors held row by row, prepared once (bench.py's SpMM configuration).
    {"name": "spmm-stencil-f32-n64", "task": "spmm", "matrix": "stencil", "x": 128, "y": 128, "z": 128,
     "dtype": "float32", "columns": 64, "order": "row", "prepared": True},
    # Aggregation over a graph: 32 features per node, the two calls every program knows.
    {"name": "spmm-powerlaw-f32-n32", "task": "spmm", "matrix": "powerlaw", "rows": 1 << 20, "longest": 50000,
     "dtype": "float32", "columns": 32, "order": "row", "prepared": False},
    # A block eigensolver: double precision, 16 vectors as the columns of a column-major array, prepared once.
    {"name": "spmm-stencil-f64-colmajor", "task": "spmm", "matrix": "stencil", "x": 101, "y": 97, "z": 89,
     "dtype": "float64", "columns": 16, "order": "col", "prepared": True},
    # Transposing a graph's matrix, values included.
    {"name": "csr2csc-powerlaw-f32", "task": "csr2csc", "matrix": "powerlaw", "rows": 1 << 22, "longest": 200000,
     "dtype": "float32"},
    # The row of every nonzero of the same kind of matrix.
    {"name": "csr2coo-powerlaw", "task": "csr2coo", "matrix": "powerlaw", "rows": 1 << 22, "longest": 200000,
     "dtype": "float32"},
    # Assembly of a finite-element matrix from its elements' triples: sort by row and column with the permutation, the
    # values brought into that order, the row offsets.
    {"name": "assemble-mesh-f64", "task": "assemble", "matrix": "mesh", "x": 701, "y": 643, "dtype": "float64"},
]


def listed():
    return [dict(c) for c in _LISTED]


def _log_between(rng, low, high):
    """A whole number between low and high, evenly spread over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def _size(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


@functools.lru_cache(maxsize=None)
def _largest_listed():
    return max(_size(c) for c in _LISTED)


def draw(rng):
    """One more case of the ranges the listed ones stand for: one of their kinds, at other sizes."""
    while True:
        case = _draw(rng)
        if _size(case) <= _largest_listed():
            return case


def _draw(rng):
    case = dict(rng.choice(_LISTED))
    del case["name"]
    case["dtype"] = rng.choice(["float32", "float64"])
    matrix = case["matrix"]
    if matrix == "laplacian":
        case["x"], case["y"] = _log_between(rng, 512, 2000), _log_between(rng, 512, 2000)
    elif matrix == "stencil":
        for side in "xyz":
            case[side] = _log_between(rng, 30, 150)
    elif matrix == "uniform":
        case["rows"] = _log_between(rng, 100000, 4000000)
        case["per_row"] = rng.randint(4, 40)
    elif matrix == "powerlaw":
        case["rows"] = _log_between(rng, 100000, 4500000)
        case["longest"] = max(64, case["rows"] // rng.randint(20, 100))
    elif rng.random() < 0.5:
        case["x"], case["y"] = _log_between(rng, 150, 1000), _log_between(rng, 150, 1000)
    else:
        case = {"task": "assemble", "matrix": "edges", "rows": _log_between(rng, 50000, 4000000),
                "nnz": _log_between(rng, 500000, 16000000), "dtype": case["dtype"]}
    if case["task"] == "spmm":
        case["columns"] = _log_between(rng, 4, 128)
    return case


# ---- sizes --------------------------------------------------------------------------------------

@functools.lru_cache(maxsize=8)
def _powerlaw_lengths(rows, longest):
    """Row lengths at the quantiles of the Zipf law: the same ones, and as many nonzeros, for every seed."""
    cdf = np.cumsum(np.arange(1, longest + 1, dtype=np.float64) ** -_POWERLAW_EXPONENT)
    lengths = np.searchsorted(cdf, cdf[-1] * (np.arange(rows) + 0.5) / rows) + 1
    return np.minimum(lengths, longest).astype(np.int64)


def _shape(case):
    """(rows, nonzeros) of the case's square matrix."""
    matrix = case["matrix"]
    if matrix == "laplacian":
        x, y = case["x"], case["y"]
        return x * y, 5 * x * y - 2 * x - 2 * y
    if matrix == "stencil":
        x, y, z = case["x"], case["y"], case["z"]
        return x * y * z, (3 * x - 2) * (3 * y - 2) * (3 * z - 2)
    if matrix == "uniform":
        return case["rows"], case["rows"] * case["per_row"]
    if matrix == "powerlaw":
        return case["rows"], int(_powerlaw_lengths(case["rows"], case["longest"]).sum())
    if matrix == "mesh":
        return (case["x"] + 1) * (case["y"] + 1), 16 * case["x"] * case["y"]
    return case["rows"], case["nnz"]


def work(case):
    m, nnz = _shape(case)
    s = 4 if case["dtype"] == "float32" else 8
    offsets, task = 4 * (m + 1), case["task"]
    if task == "spmv":
        reads_y = m * s if case["beta"] != 0 else 0
        return {"bytes": offsets + nnz * (4 + s) + 2 * m * s + reads_y, "flops": 2 * nnz}
    if task == "spmm":
        return {"bytes": offsets + nnz * (4 + s) + 2 * m * case["columns"] * s, "flops": 2 * nnz * case["columns"]}
    if task == "csr2csc":
        return {"bytes": 2 * offsets + 2 * nnz * (4 + s), "flops": 0}
    if task == "csr2coo":
        return {"bytes": offsets + 4 * nnz, "flops": 0}
    # triples read (rows, columns, values), columns, values and permutation written, and the offsets
    return {"bytes": nnz * (8 + s) + nnz * (8 + s) + offsets, "flops": 0}


def tolerance(case):
    if case["task"] in ("spmv", "spmm"):
        return {"rel": 1e-5} if case["dtype"] == "float32" else {"rel": 1e-13}
    return "exact"  # orders, offsets and moved values


# ---- matrices -----------------------------------------------------------------------------------

def _uniform_values(gen, size, dtype):
    return torch.rand(size, generator=gen, dtype=dtype, device="cuda").mul_(2).sub_(1)


def _offsets(lengths):
    ptr = torch.zeros(lengths.numel() + 1, dtype=torch.int64, device="cuda")
    torch.cumsum(lengths, 0, out=ptr[1:])
    return ptr.to(torch.int32)


def _grid_matrix(sides, reach):
    """Offsets and columns of a stencil on a grid, numbered with the first side fastest; reach: the steps to take."""
    strides = [1]
    for side in sides[:-1]:
        strides.append(strides[-1] * side)
    index = torch.arange(strides[-1] * sides[-1], device="cuda")
    at = [index // stride % side for side, stride in zip(sides, strides)]
    columns, kept = [], []
    for step in reach:
        ok = torch.ones_like(index, dtype=torch.bool)
        for position, side, d in zip(at, sides, step):
            if d != 0:
                ok &= (position + d >= 0) & (position + d < side)
        columns.append((index + sum(d * stride for d, stride in zip(step, strides))).to(torch.int32))
        kept.append(ok)
    kept = torch.stack(kept, 1)
    return _offsets(kept.sum(1)), torch.stack(columns, 1)[kept]


def _matrix(case, gen):
    """CSR arrays (offsets, columns, values) on the GPU."""
    dtype = getattr(torch, case["dtype"])
    m, nnz = _shape(case)
    if case["matrix"] == "laplacian":
        ptr, col = _grid_matrix([case["x"], case["y"]], [(0, -1), (-1, 0), (0, 0), (1, 0), (0, 1)])
        rows = torch.repeat_interleave(torch.arange(m, device="cuda"), ptr.diff())
        return ptr, col, torch.where(rows == col, 4.0, -1.0).to(dtype)
    if case["matrix"] == "stencil":
        steps = [(dx, dy, dz) for dz in (-1, 0, 1) for dy in (-1, 0, 1) for dx in (-1, 0, 1)]
        ptr, col = _grid_matrix([case["x"], case["y"], case["z"]], steps)
        return ptr, col, _uniform_values(gen, nnz, dtype)
    if case["matrix"] == "uniform":
        k = case["per_row"]
        # sorted draws from [0, m - k] plus 0 .. k-1: strictly increasing and below m
        d = torch.randint(0, m - k + 1, (m, k), generator=gen, dtype=torch.int32, device="cuda").sort(1).values
        d += torch.arange(k, dtype=torch.int32, device="cuda")
        ptr = torch.arange(m + 1, dtype=torch.int32, device="cuda") * k
        return ptr, d.reshape(-1), torch.randn(nnz, generator=gen, dtype=dtype, device="cuda")
    lengths = torch.from_numpy(_powerlaw_lengths(case["rows"], case["longest"])).cuda()
    lengths = lengths[torch.randperm(m, generator=gen, device="cuda")]
    ptr = _offsets(lengths)
    rows = torch.repeat_interleave(torch.arange(m, device="cuda"), lengths)
    d = (torch.rand(nnz, generator=gen, dtype=torch.float64, device="cuda") * (m - lengths + 1)[rows]).to(torch.int64)
    key = ((rows << 32) | torch.minimum(d, (m - lengths)[rows])).sort().values
    col = (key & 0xFFFFFFFF) + torch.arange(nnz, device="cuda") - ptr.to(torch.int64)[rows]
    return ptr, col.to(torch.int32), _uniform_values(gen, nnz, dtype)


def _triples(case, gen):
    """Row and column indices (int32) of the triples to assemble, in the order they come about."""
    if case["matrix"] == "edges":
        m, nnz = _shape(case)
        return [torch.randint(0, m, (nnz,), generator=gen, dtype=torch.int32, device="cuda") for _ in range(2)]
    x, y = case["x"], case["y"]
    element = torch.arange(x * y, device="cuda")
    first = element // x * (x + 1) + element % x
    nodes = torch.stack([first, first + 1, first + x + 2, first + x + 1], 1).to(torch.int32)
    return nodes.repeat_interleave(4, 1).reshape(-1), nodes.repeat(1, 4).reshape(-1)


# ---- prepare and run ----------------------------------------------------------------------------

def _buffer(status, size):
    api.check(status, "buffer size")
    return torch.empty(size, dtype=torch.uint8, device="cuda")


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    state = {"case": case, "handle": api.Handle(stream=torch.cuda.current_stream().cuda_stream)}
    globals()["_prepare_" + case["task"]](case, gen, state)
    return state


def run(state):
    return globals()["_run_" + state["case"]["task"]](state)


def _prepare_spmv(case, gen, s):
    ptr, col, val = _matrix(case, gen)
    m, nnz = _shape(case)
    s["op"] = api.OP_N if case["op"] == "N" else api.OP_T
    s["x"], s["y"] = _uniform_values(gen, m, val.dtype), _uniform_values(gen, m, val.dtype)
    s["mat"], s["vx"], s["vy"] = api.SpMat(m, m, nnz, ptr, col, val), api.DnVec(s["x"]), api.DnVec(s["y"])
    s["type"] = api.maca_type(val.dtype)
    call = (s["handle"], s["op"], case["alpha"], s["mat"], s["vx"], case["beta"], s["vy"], s["type"])
    if case["prepared"]:
        s["buffer"] = _buffer(*api.spmv_preprocess_buffer_size(*call))
        api.check(api.spmv_preprocess(*call, s["buffer"]), "mcsparseSpMV_preprocess")
    else:
        s["buffer"] = _buffer(*api.spmv_buffer_size(*call))


def _run_spmv(s):
    case = s["case"]
    api.check(api.spmv(s["handle"], s["op"], case["alpha"], s["mat"], s["vx"], case["beta"], s["vy"], s["type"],
                       s["buffer"]), "mcsparseSpMV")
    return s["y"]


def _prepare_spmm(case, gen, s):
    ptr, col, val = _matrix(case, gen)
    m, nnz = _shape(case)
    n, row_major = case["columns"], case["order"] == "row"
    shape, ld = ((m, n), n) if row_major else ((n, m), m)
    order = api.ORDER_ROW if row_major else api.ORDER_COL
    s["B"], s["C"] = _uniform_values(gen, shape, val.dtype), torch.zeros(shape, dtype=val.dtype, device="cuda")
    s["mat"] = api.SpMat(m, m, nnz, ptr, col, val)
    s["mB"], s["mC"] = api.DnMat(m, n, ld, s["B"], order=order), api.DnMat(m, n, ld, s["C"], order=order)
    s["type"] = api.maca_type(val.dtype)
    call = (s["handle"], api.OP_N, api.OP_N, 1.0, s["mat"], s["mB"], 0.0, s["mC"], s["type"])
    s["buffer"] = _buffer(*api.spmm_buffer_size(*call))
    if case["prepared"]:
        api.check(api.spmm_preprocess(*call, s["buffer"]), "mcsparseSpMM_preprocess")


def _run_spmm(s):
    api.check(api.spmm(s["handle"], api.OP_N, api.OP_N, 1.0, s["mat"], s["mB"], 0.0, s["mC"], s["type"], s["buffer"]),
              "mcsparseSpMM")
    return s["C"]


def _prepare_csr2csc(case, gen, s):
    s["ptr"], s["col"], s["val"] = _matrix(case, gen)
    m, nnz = _shape(case)
    s["col_ptr"] = torch.zeros(m + 1, dtype=torch.int32, device="cuda")
    s["row"] = torch.zeros(nnz, dtype=torch.int32, device="cuda")
    s["out_val"] = torch.zeros_like(s["val"])
    s["call"] = (s["handle"], m, m, nnz, s["val"], s["ptr"], s["col"], s["out_val"], s["col_ptr"], s["row"],
                 api.maca_type(s["val"].dtype), api.ACTION_NUMERIC, api.BASE_ZERO)
    s["buffer"] = _buffer(*api.csr2csc_buffer_size(*s["call"]))


def _run_csr2csc(s):
    api.check(api.csr2csc(*s["call"], s["buffer"]), "mcsparseCsr2cscEx2")
    return s["col_ptr"], s["row"], s["out_val"]


def _prepare_csr2coo(case, gen, s):
    s["ptr"] = _matrix(case, gen)[0]
    s["m"], s["nnz"] = _shape(case)
    s["rows"] = torch.zeros(s["nnz"], dtype=torch.int32, device="cuda")


def _run_csr2coo(s):
    api.check(api.xcsr2coo(s["handle"], s["ptr"], s["nnz"], s["m"], s["rows"], api.BASE_ZERO), "mcsparseXcsr2coo")
    return s["rows"]


def _prepare_assemble(case, gen, s):
    s["new_rows"], s["new_cols"] = _triples(case, gen)
    s["m"], s["nnz"] = _shape(case)
    s["new_vals"] = _uniform_values(gen, s["nnz"], getattr(torch, case["dtype"]))
    s["rows"], s["cols"], s["perm"] = (torch.empty_like(s["new_rows"]) for _ in range(3))
    s["vals"] = torch.empty_like(s["new_vals"])
    s["ptr"] = torch.empty(s["m"] + 1, dtype=torch.int32, device="cuda")
    s["buffer"] = _buffer(*api.sort_buffer_size(s["handle"], "coo", s["m"], s["m"], s["nnz"], s["rows"], s["cols"]))


def _run_assemble(s):
    handle, m, nnz = s["handle"], s["m"], s["nnz"]
    s["rows"].copy_(s["new_rows"])  # the sort works in place
    s["cols"].copy_(s["new_cols"])
    api.check(api.create_identity_permutation(handle, nnz, s["perm"]), "mcsparseCreateIdentityPermutation")
    api.check(api.xcoosort_by_row(handle, m, m, nnz, s["rows"], s["cols"], s["perm"], s["buffer"]),
              "mcsparseXcoosortByRow")
    api.check(api.gthr(handle, nnz, s["new_vals"], s["vals"], s["perm"], api.BASE_ZERO), "mcsparseXgthr")
    api.check(api.xcoo2csr(handle, s["rows"], nnz, m, s["ptr"], api.BASE_ZERO), "mcsparseXcoo2csr")
    return s["ptr"], s["cols"], s["vals"], s["perm"]
