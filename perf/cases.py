"""Workloads that a user of the array layer has it do, for timing: calls of the public entry points over the range of
shapes, element types and options that they are used with.

``listed()`` names a dozen of them, from a call that is all latency to arrays of 2 GiB; ``draw(rng)`` gives further ones
of the same ranges.  A case is a dict of plain values; ``prepare`` makes its inputs on the GPU, ``run`` is one call as a
user's program writes it (results allocated by the call where the entry point allocates them) and ``work`` is what no
implementation can do without.  Sizes come from ``bench.py``, the tests and the reference's own benchmark suite
(perf/array.jl: 512 x 1000 and 3 x 1 000 000) or are generic.
"""
import math

import numpy as np
import torch

from __graft_entry__ import load_package

rk = load_package()

_TORCH = {"Float32": torch.float32, "Float64": torch.float64, "Int32": torch.int32, "Int64": torch.int64,
          "Int16": torch.int16, "Bool": torch.bool}
_NUMPY = {"Float32": np.float32, "Float64": np.float64, "Int32": np.int32, "Int64": np.int64,
          "Int16": np.int16, "Bool": np.bool_}
_BYTES = {name: np.dtype(t).itemsize for name, t in _NUMPY.items()}


def listed():
    return [
        # the reference suite's reductions/reduce/Float32/dims=1: column sums of a small matrix, a call of pure latency
        dict(name="sum_dims1_512x1000", op="reduce", map="identity", fold="sum", dtype="Float32", rows=512, cols=1000, along=1),
        # the reference suite's reductions/mapreduce/Int64/dims=2L: a closure over points stored as 3 x N, folded over the points
        dict(name="mapreduce_dims2_3x1000000", op="reduce", map="x+1", fold="+", dtype="Int64", rows=3, cols=1000000, along=2),
        # a whole integer vector to one host number, widening to Int64: the result is fetched by every call
        dict(name="sum_int32_2p24", op="reduce", map="identity", fold="sum", dtype="Int32", rows=1 << 24, cols=1, along=0),
        # best entry of every column with its CartesianIndex, matrix of 256 MiB
        dict(name="findmax_dims1_8192x8192", op="findmax", dtype="Float32", rows=8192, cols=8192, along=1),
        # running sum of a long integer vector (wraps)
        dict(name="cumsum_int32_2p27", op="scan", dtype="Int32", rows=1 << 27, cols=1, along=1),
        # running sum across the columns of a matrix whose rows start at odd addresses
        dict(name="cumsum_dims2_4097x16000", op="scan", dtype="Float32", rows=4097, cols=16000, along=2),
        # fused elementwise update of large 3-D fields, three inputs: the largest listed case
        dict(name="broadcast_exp_512x512x512", op="axpbyexp", dtype="Float32", n=512 ** 3),
        # matrix against a row and a column vector, ragged extents
        dict(name="broadcast_rowcol_8191x4099", op="rowcol", dtype="Float32", rows=8191, cols=4099),
        # one right-hand side of the DG solver on a mesh of the benchmark's size, accumulated in place
        dict(name="volumerhs_4000", op="volumerhs", nelem=4000),
        # x[mask]: a quarter of a long vector is selected
        dict(name="logical_index_2p26", op="mask", dtype="Float32", n=1 << 26, percent=25),
        # sorted copy of a long float vector (perf/array.jl sorts Float32 vectors)
        dict(name="sort_float32_2p26", op="sort", dtype="Float32", n=1 << 26, bits=32, rev=False),
        # stable permutation by 64-bit keys, odd length of about a million
        dict(name="sortperm_int64_1000003", op="sortperm", dtype="Int64", n=1000003, bits=64, rev=False),
    ]


def _log_uniform(rng, lo, hi):
    """A whole number of [lo, hi], spread over its logarithm; odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _matrix(rng, most):
    """(rows, cols) with 2^12 .. `most` elements: squarish, tall or wide, now and then a few rows (points stored as 3 x N)."""
    n = _log_uniform(rng, 1 << 12, most)
    if rng.random() < 0.25:
        rows = rng.randint(2, 16)
    else:
        rows = _log_uniform(rng, 32, max(33, n // 32))
    return rows, max(1, n // rows)


def draw(rng):
    op = rng.choice(["reduce", "reduce", "findmax", "scan", "scan", "axpbyexp", "rowcol", "volumerhs", "mask", "sort", "sort", "sortperm"])
    if op == "reduce":
        dtype = rng.choice(["Float32", "Float32", "Float64", "Int32", "Int64"])
        along = rng.choice([0, 1, 2])
        rows, cols = (_log_uniform(rng, 1 << 12, 1 << 27), 1) if along == 0 else _matrix(rng, 1 << 26)
        return dict(op=op, map=rng.choice(["identity", "identity", "abs2", "x+1"]), fold=rng.choice(["sum", "+", "max"]), dtype=dtype,
                    rows=rows, cols=cols, along=along)
    if op == "findmax":
        rows, cols = _matrix(rng, 1 << 26)
        return dict(op=op, dtype=rng.choice(["Float32", "Float64", "Int32"]), rows=rows, cols=cols, along=rng.choice([0, 1, 2]))
    if op == "scan":
        dtype = rng.choice(["Float32", "Int32", "Int64", "Int16"])
        along = rng.choice([1, 2])
        rows, cols = (_log_uniform(rng, 1 << 12, (1 << 29) // _BYTES[dtype]), 1) if rng.random() < 0.4 else _matrix(rng, 1 << 26)
        return dict(op=op, dtype=dtype, rows=rows, cols=cols, along=1 if cols == 1 else along)
    if op == "axpbyexp":
        return dict(op=op, dtype=rng.choice(["Float32", "Float32", "Float64"]), n=_log_uniform(rng, 1 << 12, 1 << 26))
    if op == "rowcol":
        rows, cols = _matrix(rng, 1 << 26)
        return dict(op=op, dtype=rng.choice(["Float32", "Float64"]), rows=rows, cols=cols)
    if op == "volumerhs":
        return dict(op=op, nelem=_log_uniform(rng, 100, 100000))
    if op == "mask":
        return dict(op=op, dtype=rng.choice(["Float32", "Int64"]), n=_log_uniform(rng, 1 << 12, 1 << 26), percent=rng.choice([1, 10, 25, 50, 90]))
    dtype = rng.choice(["Float32", "Int32", "Int64", "Float64"])
    width = 8 * _BYTES[dtype]
    most = 1 << 26 if op == "sort" and width == 32 else 1 << 24
    # integer keys are random in all their bits or small numbers; floats are normally distributed
    bits = rng.choice([width, width, 8, 20]) if dtype.startswith("Int") else width
    return dict(op=op, dtype=dtype, n=_log_uniform(rng, 1 << 12, most), bits=bits, rev=rng.random() < 0.25)


def _values(gen, n, dtype, kind):
    """n values on the GPU: "unit" = uniform in [0, 1) (sums and scans), "normal", "count" = whole numbers in [-1000, 1000]."""
    if dtype.startswith("Int"):
        most = 100 if dtype == "Int16" else 1000
        return torch.randint(-most, most + 1, (n,), device="cuda", generator=gen, dtype=_TORCH[dtype])
    make = torch.rand if kind == "unit" else torch.randn
    return make(n, device="cuda", generator=gen, dtype=_TORCH[dtype])


def _wrap(t, dims, dtype):
    return rk.ROCArray(buf=t.view(torch.uint8).reshape(-1), dims=dims, dtype=_NUMPY[dtype])


def _tensor(a):
    """The elements of a ROCArray as a flat torch tensor (a view)."""
    name = {v: k for k, v in _NUMPY.items()}[a.dtype.type]
    return a.buf[a.offset:a.offset + len(a) * a.dtype.itemsize].view(_TORCH[name])


def prepare(case, seed):
    gen = torch.Generator(device="cuda")
    gen.manual_seed(seed)
    op = case["op"]
    dtype = case.get("dtype", "Float32")
    s = dict(op=op)
    if op in ("reduce", "findmax", "scan"):
        rows, cols = case["rows"], case["cols"]
        dims = (rows,) if cols == 1 and case["along"] != 2 else (rows, cols)
        kind = "normal" if op == "findmax" or case.get("map") == "abs2" else "unit"
        s.update(A=_wrap(_values(gen, rows * cols, dtype, kind), dims, dtype), along=case["along"] or None)
        if op == "reduce":
            s.update(f={"identity": rk.identity, "abs2": rk.abs2, "x+1": lambda v: v + 1}[case["map"]],
                     fold={"sum": rk.add_sum, "+": rk.add, "max": rk.max_}[case["fold"]])
    elif op == "axpbyexp":
        n = case["n"]
        x, y, w = (_wrap(_values(gen, n, dtype, "normal"), (n,), dtype) for _ in range(3))
        s.update(a=_NUMPY[dtype](0.5), x=x, y=y, w=w, z=rk.ROCArray(dims=(n,), dtype=_NUMPY[dtype]))
    elif op == "rowcol":
        rows, cols = case["rows"], case["cols"]
        s.update(A=_wrap(_values(gen, rows * cols, dtype, "unit"), (rows, cols), dtype),
                 r=_wrap(_values(gen, cols, dtype, "unit"), (1, cols), dtype),
                 c=_wrap(_values(gen, rows, dtype, "unit"), (rows, 1), dtype),
                 C=rk.ROCArray(dims=(rows, cols), dtype=_NUMPY[dtype]))
    elif op == "volumerhs":
        ne = case["nelem"]
        s.update(Q=_wrap(_values(gen, 625 * ne, "Float32", "unit") + 0.5, (5, 5, 5, 5, ne), "Float32"),
                 vgeo=_wrap(_values(gen, 1750 * ne, "Float32", "unit") * 0.2 + 0.9, (5, 5, 5, 14, ne), "Float32"),
                 D=_wrap(_values(gen, 25, "Float32", "unit"), (5, 5), "Float32"),
                 rhs=rk.zeros(np.float32, 5, 5, 5, 5, ne), nelem=ne)
    elif op == "mask":
        n = case["n"]
        want = n * case["percent"] // 100
        mask = torch.rand(n, device="cuda", generator=gen) < case["percent"] / 100
        surplus = int(mask.sum()) - want                # the share is met to the element, so that every seed selects alike many
        pool = torch.nonzero(mask if surplus > 0 else ~mask).reshape(-1)
        mask[pool[torch.randperm(len(pool), device="cuda", generator=gen)[:abs(surplus)]]] = surplus < 0
        s.update(x=_wrap(_values(gen, n, dtype, "normal"), (n,), dtype), mask=_wrap(mask, (n,), "Bool"))
    else:
        n, bits = case["n"], case["bits"]
        if dtype.startswith("Int"):
            half = 1 << (bits - 1)
            keys = torch.randint(-half, half - 1, (n,), device="cuda", generator=gen, dtype=_TORCH[dtype])
        else:
            keys = _values(gen, n, dtype, "normal")
        s.update(x=_wrap(keys, (n,), dtype), rev=case["rev"])
    return s


def run(s):
    op = s["op"]
    if op == "reduce":
        R = rk.mapreduce(s["f"], s["fold"], s["A"], dims=s["along"])
        return R if s["along"] is None else _tensor(R)
    if op == "findmax":
        v, i = rk.findmax(s["A"], dims=s["along"])
        return (v, i) if s["along"] is None else (_tensor(v), _tensor(i))
    if op == "scan":
        return _tensor(rk.cumsum(s["A"], dims=s["along"]))
    if op == "axpbyexp":
        return _tensor(rk.materialize_(s["z"], s["a"] * rk.lazy(s["x"]) + rk.lazy(s["y"]) * rk.broadcast.exp(rk.lazy(s["w"]))))
    if op == "rowcol":
        return _tensor(rk.materialize_(s["C"], rk.lazy(s["A"]) + rk.lazy(s["r"]) * rk.lazy(s["c"])))
    if op == "volumerhs":
        return _tensor(rk.volumerhs_(s["rhs"], s["Q"], s["vgeo"], 9.81, s["D"], s["nelem"]))
    if op == "mask":
        return _tensor(rk.getindex_mask(s["x"], s["mask"]))
    if op == "sort":
        return _tensor(rk.sort(s["x"], rev=s["rev"]))
    return _tensor(rk.sortperm(s["x"], rev=s["rev"]))


def work(case):
    """Bytes: every input read once, every output written once.  Operations: those of the formula (comparisons included)."""
    op = case["op"]
    size = _BYTES[case.get("dtype", "Float32")]
    if op in ("reduce", "findmax", "scan"):
        rows, cols = case["rows"], case["cols"]
        n = rows * cols
        if op == "scan":
            return {"bytes": 2 * n * size, "flops": n}
        outs = {0: 1, 1: cols, 2: rows}[case["along"]]
        if op == "findmax":
            return {"bytes": n * size + outs * (size + 8 * (1 if cols == 1 else 2)), "flops": n}
        widened = 8 if case["dtype"] == "Int32" and case["fold"] == "sum" else size
        return {"bytes": n * size + outs * widened, "flops": n * (1 if case["map"] == "identity" else 2)}
    if op == "axpbyexp":
        return {"bytes": 4 * case["n"] * size, "flops": 4 * case["n"]}
    if op == "rowcol":
        rows, cols = case["rows"], case["cols"]
        return {"bytes": (2 * rows * cols + rows + cols) * size, "flops": 2 * rows * cols}
    if op == "volumerhs":
        # Q 2500, 12 of the 14 fields of vgeo 6000, rhs read and written 5000 bytes an element of the mesh
        return {"bytes": 13500 * case["nelem"], "flops": 37000 * case["nelem"]}
    n = case["n"]
    if op == "mask":
        return {"bytes": n * (1 + size) + n * case["percent"] // 100 * size, "flops": 0}
    return {"bytes": n * size + n * (size if op == "sort" else 8), "flops": 0}


def tolerance(case):
    """Whole numbers, selected and moved elements are exact; sums and elementwise floats as their type gives."""
    op, dtype = case["op"], case.get("dtype", "Float32")
    if op in ("findmax", "mask", "sort", "sortperm") or dtype.startswith("Int") or case.get("fold") == "max":
        return "exact"
    # about four times the distance from the same path in 64 bits, the largest seen over the ranges of draw()
    f32 = dtype == "Float32"
    if op == "volumerhs":
        return {"rel": 4e-7, "max": 5e-6}
    if op == "axpbyexp":
        return {"rel": 2e-7, "max": 6e-5} if f32 else {"rel": 4e-16, "max": 2e-13}
    if op == "rowcol":
        return {"rel": 1.2e-7} if f32 else {"rel": 3e-16}
    return {"rel": 7e-7 if f32 else 6e-14 if op == "scan" else 1e-15}
