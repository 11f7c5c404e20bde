"""Quantiles of a long vector by selection: the same bits as by sorting the vector, over types,
distributions and sizes around the ends of the 16-byte loads, the workgroups and the copy."""
from __future__ import annotations

import numpy as np
import pytest
from conftest import assert_same_bits

import cupynumeric_amd as num
from cupynumeric_amd import _stats
from oracle import sort_oracle as oracle

pytestmark = pytest.mark.gpu

TYPES = [np.float32, np.float64, np.int32, np.uint32, np.int64, np.uint64]


def _data(kind, dtype, n, rng):
    dt = np.dtype(dtype)
    if kind == "equal":
        return np.full(n, 7, dtype=dt)
    if kind == "ids":
        return rng.integers(0, 1_000_000_000, n).astype(dt)
    if kind == "few":
        return rng.integers(0, 5, n).astype(dt)
    if dt.kind != "f":
        info = np.iinfo(dt)
        return rng.integers(info.min, info.max, n, dtype=dt, endpoint=True)
    x = rng.standard_normal(n).astype(dt)
    if kind == "specials":  # zeros of either sign, NaNs of several payloads, infinities
        u = rng.random(n)
        bits = x.view(np.uint32 if dt.itemsize == 4 else np.uint64)
        bits[u < 0.2] = np.asarray(-0.0, dt).view(bits.dtype)
        x[(u >= 0.2) & (u < 0.35)] = 0.0
        nans = (u >= 0.35) & (u < 0.6)
        bits[nans] = np.asarray(np.nan, dt).view(bits.dtype) + rng.integers(0, 1000, int(nans.sum())).astype(bits.dtype)
        x[(u >= 0.6) & (u < 0.62)] = -np.inf
        x[(u >= 0.62) & (u < 0.65)] = np.inf
    return x


@pytest.mark.parametrize("dtype", TYPES)
@pytest.mark.parametrize("kind", ["random", "equal", "ids", "few", "specials"])
def test_selection_gives_the_bits_of_the_sorted_order(dtype, kind, monkeypatch):
    monkeypatch.setattr(_stats, "SELECT_MIN_SIZE", 1)
    rng = np.random.default_rng(np.dtype(dtype).num)
    qs = [0.0, 0.05, 0.25, 0.31, 0.5, 0.62, 0.75, 0.95, 1.0]
    for n in (1, 2, 3, 5, 17, 1023, 1025, 4099, 16384, 65537, 300_007):
        x = _data(kind, dtype, n, rng)
        a = num.array(x)
        assert _stats._select_bytes(a, len(qs)) != 0
        for q, method in ((qs, "lower"), (qs, "linear"), (qs + qs[:7], "midpoint"), (0.4, "nearest")):
            got = np.asarray(num.quantile(a, q, method=method))
            assert_same_bits(got, oracle.quantile(x, q, method=method), f"{np.dtype(dtype)} {kind} n={n} {method}")
        assert_same_bits(np.asarray(a), x, "the input was modified")


@pytest.mark.parametrize("dtype", TYPES)
def test_selection_from_a_vector_at_any_element_address(dtype, monkeypatch):
    monkeypatch.setattr(_stats, "SELECT_MIN_SIZE", 1)
    rng = np.random.default_rng(5)
    x = _data("random", dtype, 6 * 9001, rng).reshape(6, 9001)  # rows of odd length: every alignment
    a = num.array(x)
    a._thunk.base.device()  # (uploaded as a whole: the rows below are views of it)
    for i in range(6):
        row = num.ndarray((9001,), x.dtype, thunk=a._thunk.slice_first_axis(i, 9001, (9001,)))
        got = np.asarray(num.percentile(row, [5.0, 50.0, 95.0]))
        assert_same_bits(got, oracle.percentile(x[i], [5.0, 50.0, 95.0]), f"row {i}")


def test_which_quantiles_are_selected():
    big = num.array(np.zeros(_stats.SELECT_MIN_SIZE, dtype=np.float32))
    assert _stats._select_bytes(big, 16) != 0 and _stats._select_bytes(big, 17) == 0 and _stats._select_bytes(big, 0) == 0
    for dtype in (np.bool_, np.int8, np.float16, np.complex64):
        assert _stats._select_bytes(num.array(np.zeros(8, dtype=dtype)), 1) == 0
    x = np.random.default_rng(1).standard_normal(100_000)
    qs = np.linspace(0, 1, 17)
    assert_same_bits(np.asarray(num.quantile(num.array(x), qs)), oracle.quantile(x, qs), "17 quantiles are read from the sorted vector")


@pytest.mark.parametrize("dtype, n", [(np.float32, 8_500_007), (np.float64, 4_300_003), (np.int64, 4_300_003)])
@pytest.mark.parametrize("kind", ["random", "specials", "few", "ids", "signed", "half"])
def test_selection_from_vectors_longer_than_one_sweep_of_the_grid(dtype, n, kind):
    """Every workgroup takes several strides: the loops with four loads in flight, the copy in several pieces, counters
    with copies by lane, and a tied NaN or zero that is searched for over several steps of a chunk."""
    rng = np.random.default_rng(n)
    if kind == "signed":
        x = rng.integers(-2, 3, n).astype(dtype)
    elif kind == "half":  # one value for half of the vector, in one bin with the others
        x = rng.integers(1, 1000, n).astype(dtype) if np.dtype(dtype).kind == "i" else (1 + rng.random(n)).astype(dtype)
        x[rng.random(n) < 0.5] = 1
    elif kind == "specials" and np.dtype(dtype).kind == "i":
        x = np.where(rng.random(n) < 0.001, rng.integers(-(10**12), 10**12, n), rng.integers(1, 6, n)).astype(dtype)
    else:
        x = _data(kind, dtype, n, rng)
    a = num.array(x)
    assert _stats._select_bytes(a, 9) != 0
    ordered = oracle.sort(x)
    for q in ([0.5], [0.0, 0.05, 0.25, 0.31, 0.5, 0.62, 0.75, 0.95, 1.0], np.linspace(0.01, 0.99, 16)):
        got = np.asarray(num.quantile(a, q, method="lower"))
        assert_same_bits(got, ordered[(np.asarray(q) * (n - 1)).astype(np.int64)], f"{kind} {len(q)} quantiles")
