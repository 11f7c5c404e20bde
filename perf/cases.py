"""Timed cases of the sort path: what a program asks of this package through its public functions.

A case names one call (`op`) and the array it is made on.  The listed cases run from the smallest
call, which is all latency, over ordinary arrays to the largest sort of the benchmark; `draw` gives
further cases of the same operations, types, distributions and range of sizes.  Inputs lie in device
memory beforehand and results stay there.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import cupynumeric_amd as num
from cupynumeric_amd._thunk import DeviceArray

# element type -> (NumPy type, torch type that holds its bits in inputs and results)
TYPES = {
    "float16": (np.float16, torch.float16),
    "float32": (np.float32, torch.float32),
    "float64": (np.float64, torch.float64),
    "int32": (np.int32, torch.int32),
    "uint32": (np.uint32, torch.int32),
    "int64": (np.int64, torch.int64),
}


def listed():
    return [
        # a small array sorted in an interactive program or an inner loop: the latency of one call
        {"name": "sort_float32_1k", "op": "sort", "dtype": "float32", "data": "normal", "n": 1000},
        # ranking a column of a table
        {"name": "argsort_float64_100k", "op": "argsort", "dtype": "float64", "data": "normal", "n": 100_000},
        # the reference's example program (examples/sort.py) with its default size and type
        {"name": "sort_uint32_1m", "op": "sort", "dtype": "uint32", "data": "full", "n": 1_000_000},
        # ordering records by an integer id: 64-bit storage, values below 10^9
        {"name": "argsort_int64_10m", "op": "argsort", "dtype": "int64", "data": "ids", "n": 10_000_000},
        # the reference's microbenchmark (examples/sort_bench.py, sort-1D, float64) at 2^26
        {"name": "sort_float64_64m", "op": "sort", "dtype": "float64", "data": "uniform", "n": 1 << 26},
        # the benchmark's headline workload: stable argsort of 2^28 float32 with NaNs and signed zeros
        {"name": "argsort_float32_256m", "op": "argsort", "dtype": "float32", "data": "specials", "n": 1 << 28},
        # ranking the candidates of many queries: a long stack of short rows of no round length
        {"name": "argsort_rows_float32_100", "op": "argsort", "dtype": "float32", "data": "normal", "rows": 1_000_000, "n": 100},
        # the benchmark's row workload: every row of a matrix sorted along the last axis
        {"name": "sort_rows_float64_1024", "op": "sort", "dtype": "float64", "data": "uniform", "rows": 65536, "n": 1024},
        # the benchmark's column workload: a sort along the first axis, transposes included
        {"name": "sort_axis0_float16_8192", "op": "sort_axis0", "dtype": "float16", "data": "normal", "rows": 8192, "n": 8192},
        # distinct values of a column with repetitions
        {"name": "unique_int32_64m", "op": "unique", "dtype": "int32", "n": 1 << 26, "distinct": 1 << 20},
        # looking many values up in a large sorted table
        {"name": "searchsorted_float32_16m_in_256m", "op": "searchsorted", "dtype": "float32", "n": 1 << 28, "values": 1 << 24},
        # order statistics of a sample: five percentiles of one long vector
        {"name": "percentile_float64_10m", "op": "percentile", "dtype": "float64", "data": "normal", "n": 10_000_000},
    ]


def _size(rng, low, high):
    """A size spread evenly over the logarithm of [low, high]; round sizes are as rare as they are odd."""
    n = int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))
    if rng.random() < 0.25:
        n = 1 << max(0, int(round(math.log2(n))))
    return min(max(n, low), high)


def _data(rng, dtype):
    return rng.choice(("uniform", "normal", "specials") if dtype.startswith("float") else ("full", "ids", "few"))


def draw(rng):
    kind = rng.choice(("flat", "flat", "flat", "flat", "rows", "rows", "axis0", "unique", "searchsorted", "percentile"))
    if kind == "flat":
        dtype = rng.choice(("float32", "float64", "int32", "uint32", "int64"))
        largest = 1 << (26 if TYPES[dtype][0]().itemsize == 8 else 28)
        return {"op": rng.choice(("sort", "argsort")), "dtype": dtype, "data": _data(rng, dtype), "n": _size(rng, 1000, largest)}
    if kind == "rows":
        dtype = rng.choice(("float16", "float32", "float64", "int32", "int64"))
        n = _size(rng, 10, 16384)
        volume = _size(rng, 1 << 18, 1 << 26)
        return {"op": rng.choice(("sort", "argsort")), "dtype": dtype, "data": _data(rng, dtype), "rows": max(1, volume // n), "n": n}
    if kind == "axis0":
        dtype = rng.choice(("float16", "float32", "float64"))
        return {"op": "sort_axis0", "dtype": dtype, "data": _data(rng, dtype), "rows": _size(rng, 500, 8192), "n": _size(rng, 500, 8192)}
    if kind == "unique":
        dtype = rng.choice(("int32", "int64"))
        n = _size(rng, 10_000, 1 << (25 if dtype == "int64" else 26))
        return {"op": "unique", "dtype": dtype, "n": n, "distinct": _size(rng, 16, n)}
    if kind == "searchsorted":
        dtype = rng.choice(("float32", "float64"))
        n = _size(rng, 10_000, 1 << (26 if dtype == "float64" else 28))
        return {"op": "searchsorted", "dtype": dtype, "n": n, "values": _size(rng, 1000, 1 << 24)}
    dtype = rng.choice(("float32", "float64"))
    return {"op": "percentile", "dtype": dtype, "data": _data(rng, dtype), "n": _size(rng, 10_000, 1 << 26)}


def _values(case, n, gen):
    """`n` elements of the case's type and distribution, on the GPU."""
    tt = TYPES[case["dtype"]][1]
    data = case.get("data", "uniform")
    if tt.is_floating_point:
        if data == "uniform":
            return torch.rand(n, generator=gen, device="cuda", dtype=tt)
        x = torch.randn(n, generator=gen, device="cuda", dtype=tt)
        if data == "specials":  # one NaN and one zero of either sign in a hundred
            u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float32)
            x.masked_fill_(u < 0.01, math.nan)
            x.masked_fill_((u >= 0.01) & (u < 0.015), 0.0)
            x.masked_fill_((u >= 0.015) & (u < 0.02), -0.0)
        return x
    info = torch.iinfo(tt)
    if data == "full":
        return torch.randint(info.min, info.max, (n,), generator=gen, device="cuda", dtype=tt)
    if data == "ids":
        return torch.randint(0, 1_000_000_000, (n,), generator=gen, device="cuda", dtype=tt)
    few = torch.randint(info.min, info.max, (100,), generator=gen, device="cuda", dtype=tt)
    return few[torch.randint(0, 100, (n,), generator=gen, device="cuda")]


def _array(buf, shape, dtype):
    return num.ndarray(shape, dtype, thunk=DeviceArray.from_device(buf, shape, dtype))


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = TYPES[case["dtype"]][0]
    n = case["n"]
    state = {"op": case["op"], "type": TYPES[case["dtype"]][1]}
    if case["op"] == "unique":
        # `distinct` ids below 10^9, evenly spaced from a first one; each occurs, the repetitions are random
        count = case["distinct"]
        spacing = torch.randint(1, max(2, 1_000_000_000 // count), (1,), generator=gen, device="cuda")
        first = torch.randint(0, 1000, (1,), generator=gen, device="cuda")
        which = torch.randint(0, count, (n,), generator=gen, device="cuda")
        which[:count] = torch.arange(count, device="cuda")
        which = which[torch.randperm(n, generator=gen, device="cuda")]
        state["a"] = _array((first + which * spacing).to(state["type"]), (n,), dtype)
    elif case["op"] == "searchsorted":
        table = torch.sort(_values(case, n, gen)).values
        state["a"] = _array(table, (n,), dtype)
        state["v"] = _array(_values(case, case["values"], gen), (case["values"],), dtype)
    else:
        shape = (case["rows"], n) if "rows" in case else (n,)
        state["a"] = _array(_values(case, math.prod(shape), gen), shape, dtype)
    return state


def _tensor(result, ttype):
    """The device memory of a result under its own shape and type."""
    flat = result._thunk.base.device().view(ttype)[: result.size]
    return flat.reshape(result.shape)


def run(state):
    op, a = state["op"], state["a"]
    if op == "sort":
        return _tensor(num.sort(a), state["type"])
    if op == "argsort":
        return _tensor(num.argsort(a), torch.int64)
    if op == "sort_axis0":
        return _tensor(num.sort(a, axis=0), state["type"])
    if op == "unique":
        return _tensor(num.unique(a), state["type"])
    if op == "searchsorted":
        return _tensor(num.searchsorted(a, state["v"]), torch.int64)
    return _tensor(num.percentile(a, [5.0, 25.0, 50.0, 75.0, 95.0]), torch.float64)


def work(case):
    """Bytes: inputs read once, results written once.  No floating-point arithmetic is needed."""
    kb = TYPES[case["dtype"]][0]().itemsize
    volume = case["n"] * case.get("rows", 1)
    if case["op"] == "argsort":
        return {"bytes": volume * (kb + 8), "flops": 0}
    if case["op"] == "unique":
        return {"bytes": (volume + min(volume, case["distinct"])) * kb, "flops": 0}
    if case["op"] == "searchsorted":  # of the table no more than one 128-byte line per value
        return {"bytes": min(volume * kb, case["values"] * 128) + case["values"] * (kb + 8), "flops": 0}
    if case["op"] == "percentile":
        return {"bytes": volume * kb + 5 * 8, "flops": 0}
    return {"bytes": 2 * volume * kb, "flops": 0}


def tolerance(case):
    """Sorting moves bits: every correct stable sort gives the same values and positions, and the
    percentiles are one fixed float64 expression of two elements of the input."""
    return "exact"
