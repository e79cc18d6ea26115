"""The workloads this library's performance is measured on.

A case is one pass through the public entry points: products of a kept matrix
handle (SpMV in several formats and value types, SpMM, a batch of many small
matrices), the product of a matrix that is new on every call, conversions
there and back, the assembly of shuffled triplets, and conjugate gradients.
The matrices are those of the library's generators, drawn on the GPU: grid
stencils of a variable-coefficient diffusion, power-law rows and banded
matrices with scattered entries.
"""
from __future__ import annotations

import functools
import math

import torch

from morpheus_amd import capi, device
from morpheus_amd import generators as gen
from morpheus_amd.formats import (COO_FORMAT, CSR_FORMAT, DIA_FORMAT, ELL_FORMAT, HDC_FORMAT,
                                  HYB_FORMAT)

FORMATS = {"coo": COO_FORMAT, "csr": CSR_FORMAT, "dia": DIA_FORMAT, "ell": ELL_FORMAT,
           "hyb": HYB_FORMAT, "hdc": HDC_FORMAT}
VALUE_BYTES = {"f64": 8, "f32": 4, "bf16": 2}
VECTOR_BYTES = {"f64": 8, "f32": 4, "bf16": 4}
STENCILS = {"stencil5": (2, 5), "stencil7": (3, 7), "stencil27": (3, 27)}


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # the product of an iterative method on a small grid: launch latency
        {"name": "spmv_csr_f64_small", "kind": "spmv", "matrix": "stencil5", "size": 256,
         "format": "csr", "dtype": "f64"},
        # a large 3D grid's operator (27 points, 127 interior nodes a side: an odd row count)
        # in single precision
        {"name": "spmv_ell_f32_grid", "kind": "spmv", "matrix": "stencil27", "size": 127,
         "format": "ell", "dtype": "f32"},
        # graph / web matrix: power-law rows, columns all over x
        {"name": "spmv_csr_f64_powerlaw", "kind": "spmv", "matrix": "powerlaw", "size": 1000003,
         "exponent": 1.5, "mean": 16.0, "cap": 20000, "format": "csr", "dtype": "f64"},
        # a large banded matrix with some scattered couplings, BF16 storage
        {"name": "spmv_hdc_bf16_banded", "kind": "spmv", "matrix": "banded", "size": 4000000,
         "half_width": 4, "offband": 0.02, "format": "hdc", "dtype": "bf16"},
        # block of right-hand sides on the largest grid (block Krylov, many load cases)
        {"name": "spmm_dia_f64_grid_k16", "kind": "spmm", "matrix": "stencil27", "size": 160,
         "format": "dia", "dtype": "f64", "k": 16},
        # a few feature / rank vectors over a graph; a ragged number of columns
        {"name": "spmm_csr_f32_powerlaw_k5", "kind": "spmm", "matrix": "powerlaw",
         "size": 2000000, "exponent": 1.2, "mean": 30.0, "cap": 200000, "format": "csr",
         "dtype": "f32", "k": 5},
        # many small matrices of mixed structure and format, one launch for all
        {"name": "batch_f32_k8", "kind": "batch", "count": 256, "size": 65536, "dtype": "f32",
         "k": 8},
        # encode and decode: CSR -> DIA -> CSR on a grid
        {"name": "convert_dia_f64_grid", "kind": "convert", "matrix": "stencil7", "size": 128,
         "format": "dia", "dtype": "f64"},
        # encode and decode: CSR -> HYB -> CSR on power-law rows
        {"name": "convert_hyb_f32_powerlaw", "kind": "convert", "matrix": "powerlaw",
         "size": 1000003, "exponent": 1.5, "mean": 16.0, "cap": 20000, "format": "hyb",
         "dtype": "f32"},
        # assembly: triplets in arbitrary order to a sorted CSR matrix
        {"name": "assemble_f64_banded", "kind": "assemble", "matrix": "banded",
         "size": 1000000, "half_width": 4, "offband": 0.02, "dtype": "f64"},
        # a matrix whose structure is new on every call (adaptive meshes, changing graphs)
        {"name": "fresh_csr_f64_powerlaw", "kind": "fresh", "matrix": "powerlaw",
         "size": 1000003, "exponent": 1.5, "mean": 16.0, "cap": 20000, "format": "csr",
         "dtype": "f64"},
        # ten iterations of conjugate gradients on a 3D grid
        {"name": "cg_dia_f64_grid", "kind": "cg", "matrix": "stencil7", "size": 128,
         "format": "dia", "dtype": "f64", "iterations": 10},
    ]


def draw(rng):
    """A case that moves no more than the largest listed one of its kind."""
    most = {}
    for c in listed():
        most[c["kind"]] = max(most.get(c["kind"], 0), work(c)["bytes"])
    while True:
        case = _draw(rng)
        if work(case)["bytes"] <= most[case["kind"]]:
            return case


def _draw(rng):
    kind = rng.choice(["spmv", "spmv", "spmv", "spmm", "spmm", "batch", "convert", "convert",
                       "assemble", "fresh", "cg"])
    case = {"kind": kind}
    if kind == "batch":
        case.update(count=round(_log(rng, 16, 256)), size=round(_log(rng, 4000, 65536)),
                    dtype=rng.choice(["f64", "f32", "bf16"]), k=rng.choice([1, 4, 8, 16]))
        return case
    if kind == "cg":
        case.update(matrix=rng.choice(list(STENCILS)), iterations=rng.randint(5, 15),
                    format=rng.choice(["csr", "dia", "ell"]), dtype=rng.choice(["f64", "f32"]))
    else:
        case.update(matrix=rng.choice(["stencil5", "stencil7", "stencil27", "powerlaw", "banded"]),
                    dtype=rng.choice(["f64", "f32", "bf16"]))
    m = case["matrix"]
    if m in STENCILS:
        case["size"] = round(_log(rng, 5000, 4e6) ** (1.0 / STENCILS[m][0]))
    else:
        case["size"] = round(_log(rng, 5000, 4e6))
    if m == "powerlaw":
        case.update(exponent=rng.choice([1.2, 1.5]), mean=rng.choice([8.0, 16.0, 30.0]),
                    cap=min(200000, max(1000, case["size"] // rng.choice([10, 50]))))
    if m == "banded":
        case.update(half_width=rng.randint(2, 16), offband=rng.choice([0.0, 0.02]))
    if kind in ("spmv", "spmm", "convert"):
        case["format"] = rng.choice([f for f in _admissible(case)
                                     if kind != "convert" or f != "csr"])
    if kind == "convert" and case["format"] == "ell" and m == "banded":
        case["offband"] = 0.0  # the widest row, and with it the width, is the band
    if kind == "spmm":
        case["k"] = rng.choice([2, 3, 4, 5, 8, 16])
    if kind == "fresh":
        case["format"] = rng.choice(["csr", "coo"])
    return case


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _admissible(case):
    """Formats whose fill the library accepts for the case's structure."""
    m = case["matrix"]
    if m == "powerlaw":
        fits = case["size"] * case["mean"] <= 9e7
        return ["csr", "coo", "hdc"] + (["hyb"] if fits else [])
    if m == "banded" and case["offband"] > 0:
        return ["csr", "coo", "ell", "hyb", "hdc"]
    return ["csr", "coo", "dia", "ell", "hyb", "hdc"]


# ------------------------------------------------------------- matrices (CSR)
def _csr_of(rows, cols, n):
    ro = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    ro[1:] = torch.cumsum(torch.bincount(rows, minlength=n), 0)
    return ro, cols.to(torch.int32)


def _stencil_offsets(kind):
    if kind == "stencil5":
        return [(-1, 0), (0, -1), (0, 0), (0, 1), (1, 0)]
    if kind == "stencil7":
        return [(-1, 0, 0), (0, -1, 0), (0, 0, -1), (0, 0, 0), (0, 0, 1), (0, 1, 0), (1, 0, 0)]
    return [(a, b, c) for a in (-1, 0, 1) for b in (-1, 0, 1) for c in (-1, 0, 1)]


def _stencil(kind, g, rg):
    """Diffusion with a coefficient per node, the mean of two nodes' on the
    edge between them; a reaction term makes it definite."""
    dim = STENCILS[kind][0]
    n = g ** dim
    node = torch.arange(n, device="cuda")
    coord = [(node // g ** (dim - 1 - d)) % g for d in range(dim)]
    coef = 0.5 + torch.rand(n, dtype=torch.float64, device="cuda", generator=rg)
    offsets = _stencil_offsets(kind)
    cols, vals, keep = [], [], []
    diag = 0.1 * coef
    for o in offsets:
        step = sum(o[d] * g ** (dim - 1 - d) for d in range(dim))
        ok = torch.ones(n, dtype=torch.bool, device="cuda")
        for d in range(dim):
            if o[d]:
                ok &= coord[d] != (g - 1 if o[d] > 0 else 0)
        to = (node + step).clamp_(0, n - 1)
        w = 0.5 * (coef + coef[to])
        if any(o):
            diag = diag + w  # edges that leave the grid too: fixed values beyond it
        cols.append(to.to(torch.int32))
        vals.append(-w)
        keep.append(ok)
    vals[len(offsets) // 2] = diag
    keep = torch.stack(keep, 1)
    ro = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
    ro[1:] = torch.cumsum(keep.sum(1), 0)
    ci = torch.stack(cols, 1)[keep]
    del cols
    return ro, ci, torch.stack(vals, 1)[keep]


@functools.lru_cache(maxsize=None)
def _powerlaw_range(exponent, mean, cap):
    return gen.powerlaw_parameters(exponent, mean, cap)


def _distinct(rows, n, cols_of):
    """Sorted keys row * n + column of len(rows) entries, cols_of(rows) drawn
    again where a row has the column already."""
    key = (rows * n + cols_of(rows)).sort().values
    while True:
        again = torch.zeros_like(key, dtype=torch.bool)
        again[1:] = key[1:] == key[:-1]
        if not again.any():
            return key
        rows = key[again] // n
        key[again] = rows * n + cols_of(rows)
        key = key.sort().values


def _powerlaw(n, exponent, mean, cap, rg):
    """Row lengths at the quantiles of a power law (at least 1, at most cap) in
    a drawn order, uniform columns."""
    top, a = _powerlaw_range(exponent, mean, cap), 1.0 - exponent
    u = (torch.randperm(n, device="cuda", generator=rg) + 0.5) / n
    r = (1.0 - u.double() * (1.0 - top ** a)) ** (1.0 / a)
    length = (1 + ((r - 1.0) * ((cap - 1) / (top - 1))).floor()).clamp_(max=cap).to(torch.int64)
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), length)
    key = _distinct(rows, n, lambda r: torch.randint(0, n, r.shape, device="cuda", generator=rg))
    ro, ci = _csr_of(key // n, key % n, n)
    return ro, ci, _normal(ci.numel(), rg)


def _banded(n, half_width, offband, rg):
    row = torch.arange(n, device="cuda")
    off = torch.arange(-half_width, half_width + 1, device="cuda")
    col = row[:, None] + off[None, :]
    key = (row[:, None] * n + col)[(col >= 0) & (col < n)]
    if offband > 0:
        far = torch.randint(0, n, (round(offband * key.numel()),), device="cuda", generator=rg)
        key = torch.cat([key, _distinct(far, n, lambda r: (
            r + torch.randint(half_width + 1, n - half_width, r.shape, device="cuda",
                              generator=rg)) % n)]).sort().values
    ro, ci = _csr_of(key // n, key % n, n)
    return ro, ci, _normal(ci.numel(), rg)


def _normal(n, rg):
    return torch.randn(n, dtype=torch.float64, device="cuda", generator=rg)


def _matrix(case, rg):
    """(nrows, row offsets, columns, values in the case's type), on the GPU."""
    m = case["matrix"]
    if m in STENCILS:
        ro, ci, v = _stencil(m, case["size"], rg)
    elif m == "powerlaw":
        ro, ci, v = _powerlaw(case["size"], case["exponent"], case["mean"], case["cap"], rg)
    else:
        ro, ci, v = _banded(case["size"], case["half_width"], case["offband"], rg)
    return ro.numel() - 1, ro, ci, v.to(device.DTYPES[case["dtype"]][0])


def _members(case, rg):
    """The batch: a third each of 5-point grids (DIA), power-law rows (CSR) and
    bands (ELL), their sizes spread over the logarithm up to case["size"]."""
    count, top = case["count"], case["size"]
    out = []
    for i in range(count):
        u, w = i * 0.6180339887 % 1.0, i * 0.4142135623 % 1.0  # evenly spread, in no order
        n = round(math.exp(math.log(1000) + u * (math.log(top) - math.log(1000))))
        if i % 3 == 0:
            g = round(math.sqrt(n))
            out.append(("dia", {"matrix": "stencil5", "size": g, "dtype": case["dtype"]}))
        elif i % 3 == 1:
            out.append(("csr", {"matrix": "powerlaw", "size": n, "exponent": 1.5, "mean": 12.0,
                                "cap": 500 if n < 4000 else 2000, "dtype": case["dtype"]}))
        else:
            out.append(("ell", {"matrix": "banded", "size": n, "half_width": 2 + int(w * 15),
                                "offband": 0.0, "dtype": case["dtype"]}))
    return [(f, _matrix(c, rg)) for f, c in out]


def _starts(sizes):
    """First rows of the members' results in one array, each on 16 bytes, and
    its number of rows."""
    at = [0]
    for n in sizes:
        at.append(at[-1] + -(-n // 4) * 4)
    return at


def _container(fmt, n, ro, ci, v, dtype):
    A = device.DeviceMatrix(CSR_FORMAT, n, n, ci.numel(), dtype, {"ro": ro, "ci": ci, "v": v}, {})
    return A if fmt == "csr" else device.convert(A, FORMATS[fmt])


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _vector(shape, dtype, rg):
    x = torch.rand(shape, dtype=torch.float64, device="cuda", generator=rg) * 2 - 1
    return x.to(device.vector_dtype(dtype))


# ---------------------------------------------------------------- prepare / run
def prepare(case, seed):
    rg = _generator(seed)
    kind, dtype = case["kind"], case["dtype"]
    if kind == "batch":
        mats, X = [], []
        for fmt, (n, ro, ci, v) in _members(case, rg):
            mats.append(_container(fmt, n, ro, ci, v, dtype))
            X.append(_vector((n, case["k"]), dtype, rg))
        at = _starts([m.nrows for m in mats])
        Y = torch.zeros((at[-1], case["k"]), dtype=X[0].dtype, device="cuda")
        parts = [Y[a:a + m.nrows] for a, m in zip(at, mats)]
        return {"kind": kind, "batch": device.Batch(mats, case["k"], X, parts), "Y": Y}
    n, ro, ci, v = _matrix(case, rg)
    if kind == "assemble":
        rows = torch.repeat_interleave(torch.arange(n, dtype=torch.int32, device="cuda"),
                                       (ro[1:] - ro[:-1]).long())
        at = torch.randperm(ci.numel(), device="cuda", generator=rg)
        return {"kind": kind, "n": n, "dtype": dtype, "ri": rows[at], "ci": ci[at], "v": v[at]}
    if kind == "convert":
        return {"kind": kind, "A": _container("csr", n, ro, ci, v, dtype),
                "format": FORMATS[case["format"]]}
    x = _vector((n, case["k"]) if kind == "spmm" else (n,), dtype, rg)
    if kind == "fresh":
        A = _container(case["format"], n, ro, ci, v, dtype)
        return {"kind": kind, "A": A, "x": x, "y": torch.zeros_like(x)}
    A = _container(case["format"], n, ro, ci, v, dtype)
    A.analyse()
    if kind == "cg":
        return {"kind": kind, "A": A, "cg": device.CG(A), "b": x, "x": torch.zeros_like(x),
                "iterations": case["iterations"]}
    return {"kind": kind, "A": A, "x": x, "y": torch.zeros_like(x)}


def run(state):
    kind = state["kind"]
    if kind in ("spmv", "spmm"):
        device.multiply(state["A"], state["x"], state["y"])
        return state["y"]
    if kind == "batch":
        state["batch"].run_graph()
        return state["Y"]
    if kind == "fresh":
        # the one-shot product over raw arrays: it keeps nothing
        A, x, y = state["A"], state["x"], state["y"]
        a = A.arrays
        coo = A.format == COO_FORMAT
        capi.call("mph_coo_multiply" if coo else "mph_csr_multiply", A.nrows, A.ncols, A.nnz,
                  a["ri"].data_ptr() if coo else a["ro"].data_ptr(), a["ci"].data_ptr(),
                  a["v"].data_ptr(), A.vt, x.data_ptr(), y.data_ptr(), 1, device.stream_handle())
        return y
    if kind == "convert":
        B = device.convert(state["A"], state["format"])
        back = device.convert(B, CSR_FORMAT)
        return {"there": [t for _, t in sorted(B.arrays.items())],
                "back": [t for _, t in sorted(back.arrays.items())]}
    if kind == "assemble":
        # the sort is in place; the program keeps its triplets
        ri, ci, v = state["ri"].clone(), state["ci"].clone(), state["v"].clone()
        dtype = state["dtype"]
        capi.call("mph_coo_sort_by_row_and_column", ri.numel(), ri.data_ptr(), ci.data_ptr(),
                  v.data_ptr(), capi.VALUE_TYPES[dtype], device.stream_handle())
        A = device.DeviceMatrix(COO_FORMAT, state["n"], state["n"], ri.numel(), dtype,
                                {"ri": ri, "ci": ci, "v": v}, {})
        return [t for _, t in sorted(device.convert(A, CSR_FORMAT).arrays.items())]
    x = state["x"]
    x.zero_()
    state["cg"].start(state["b"], x)
    state["cg"].iterate(x, state["iterations"])
    return x


# ---------------------------------------------------------------- work
def _shape(case):
    """(rows, entries, entries of a padded DIA / ELL form), entries as expected."""
    m, s = case["matrix"], case["size"]
    if m in STENCILS:
        dim, points = STENCILS[m]
        nnz = (3 * s - 2) ** 3 if points == 27 else s ** dim + 2 * dim * (s - 1) * s ** (dim - 1)
        return s ** dim, nnz, points * s ** dim
    if m == "powerlaw":
        return s, int(s * case["mean"]), int(s * case["mean"])
    h = case["half_width"]
    nnz = int((s * (2 * h + 1) - h * (h + 1)) * (1 + case["offband"]))
    return s, nnz, max(nnz, s * (2 * h + 1))


def _format_bytes(case):
    """Bytes of the matrix in the case's format, no index or value twice."""
    n, nnz, padded = _shape(case)
    v = VALUE_BYTES[case["dtype"]]
    f = case.get("format", "csr")
    if f == "dia":
        return padded * v
    if f == "ell":
        return padded * (4 + v)
    if f == "coo":
        return nnz * (8 + v)
    if f == "hdc" and case["matrix"] != "powerlaw":
        return nnz * v  # nearly all of it on full diagonals
    return nnz * (4 + v) + 4 * (n + 1)


def work(case):
    if case["kind"] == "batch":
        # sizes spread over the logarithm from 1000: their mean, and 5, 12 and
        # on average 19 entries a row in the three kinds
        n = (case["size"] - 1000) / math.log(case["size"] / 1000) * case["count"]
        v, w, k = VALUE_BYTES[case["dtype"]], VECTOR_BYTES[case["dtype"]], case["k"]
        nnz = n * (5 * v + 12 * (4 + v) + 19 * (4 + v)) / 3
        return {"bytes": int(nnz + 2 * n * k * w), "flops": int(2 * n * 12 * k)}
    n, nnz, _ = _shape(case)
    v, w = VALUE_BYTES[case["dtype"]], VECTOR_BYTES[case["dtype"]]
    csr = nnz * (4 + v) + 4 * (n + 1)
    kind = case["kind"]
    if kind == "convert":
        wide = _format_bytes(case)
        return {"bytes": 2 * csr + 2 * wide, "flops": 0}
    if kind == "assemble":
        return {"bytes": nnz * (8 + v) + csr, "flops": 0}
    if kind == "cg":
        # each iteration the matrix, x, r and p read and written, A p kept
        it = case["iterations"]
        return {"bytes": it * (_format_bytes(case) + 8 * n * w), "flops": it * (2 * nnz + 10 * n)}
    k = case.get("k", 1)
    return {"bytes": _format_bytes(case) + 2 * n * k * w, "flops": 2 * nnz * k}


# ---------------------------------------------------------------- accuracy
def tolerance(case):
    if case["kind"] in ("convert", "assemble"):
        return "exact"
    f64 = case["dtype"] == "f64"
    return {"rel": 4e-15 if f64 else 5e-7}


def _exact_product(n, ro, ci, v, x):
    """A x in 64 bits, each row in 32 partial sums (shorter chains: long rows
    round less)."""
    parts = 32
    rows = torch.repeat_interleave(torch.arange(n, device="cuda"), (ro[1:] - ro[:-1]).long())
    at = rows * parts + torch.arange(ci.numel(), device="cuda") % parts
    ci, v, x = ci.long(), v.double(), x.double()
    if x.dim() == 2:
        return torch.stack([_parts_sum(n, parts, at, v * c[ci]) for c in x.t().contiguous()], 1)
    return _parts_sum(n, parts, at, v * x[ci])


def _parts_sum(n, parts, at, products):
    y = torch.zeros(n * parts, dtype=torch.float64, device="cuda")
    return y.index_add_(0, at, products).view(n, parts).sum(1)


def exact(case, seed):
    kind, dtype = case["kind"], case["dtype"]
    if kind in ("convert", "assemble"):
        return None
    rg = _generator(seed)
    if kind == "batch":
        parts = []
        for _, (n, ro, ci, v) in _members(case, rg):
            parts.append(_exact_product(n, ro, ci, v, _vector((n, case["k"]), dtype, rg)))
        at = _starts([len(y) for y in parts])
        Y = torch.zeros((at[-1], case["k"]), dtype=torch.float64, device="cuda")
        for a, y in zip(at, parts):
            Y[a:a + len(y)] = y
        return Y
    n, ro, ci, v = _matrix(case, rg)
    x = _vector((n, case["k"]) if kind == "spmm" else (n,), dtype, rg)
    if kind != "cg":
        return _exact_product(n, ro, ci, v, x)
    b = x.double()
    x = torch.zeros_like(b)
    r, p = b.clone(), b.clone()
    rr = r.dot(r)
    for _ in range(case["iterations"]):
        q = _exact_product(n, ro, ci, v, p)
        a = rr / p.dot(q)
        x += a * p
        r -= a * q
        new = r.dot(r)
        p = r + (new / rr) * p
        rr = new
    return x
