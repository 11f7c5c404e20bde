"""searchsorted of so few values that every lane has one, at the edges of its range and of its table, against numpy."""
from __future__ import annotations

import numpy as np
import pytest

import cupynumeric_amd as num

pytestmark = pytest.mark.gpu


def _sorted(dtype, n, rng):
    kind = np.dtype(dtype).kind
    if kind == "f":
        a = (rng.standard_normal(n) * 100).astype(dtype)
        a[: n // 50], a[n // 50 : n // 40] = np.nan, -0.0
        a[n // 40 : n // 30] = np.inf
    elif kind == "b":
        a = rng.integers(0, 2, n).astype(dtype)
    else:
        info = np.iinfo(dtype)
        a = rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)
        a[: n // 50], a[n // 50 : n // 40] = info.max, info.min
    return np.sort(a, kind="stable")


def _check(a, v):
    wide = (lambda x: x.astype(np.float32)) if a.dtype == np.float16 else (lambda x: x)
    for side in ("left", "right"):
        got = np.asarray(num.searchsorted(num.array(a), num.array(v), side=side))
        assert np.array_equal(got, np.searchsorted(wide(a), wide(v), side)), (a.dtype, a.size, v.size, side)


@pytest.mark.parametrize("dtype", [np.bool_, np.int8, np.uint16, np.int32, np.uint64, np.float16, np.float32, np.float64])
def test_types(dtype):
    rng = np.random.default_rng(np.dtype(dtype).num)
    for n, m in ((8191, 2048), (8192, 2047), (8192, 2048), (8193, 2049), (100_003, 5000)):
        a = _sorted(dtype, n, rng)
        v = a[rng.integers(0, n, m)]
        v[: m // 4] = _sorted(dtype, m, rng)[rng.integers(0, m, m // 4)]  # values that are not in the array as well
        _check(a, v)


@pytest.mark.parametrize("n", [2048 * 5 - 1, 2048 * 5, 2048 * 5 + 1, 1_000_003])
@pytest.mark.parametrize("m", [(1 << 19) - 1, 1 << 19, (1 << 19) + 1])
def test_edges_of_the_range(n, m):
    rng = np.random.default_rng(n + m)
    a = _sorted(np.float32, n, rng)
    _check(a, a[rng.integers(0, n, m)])
    a = np.arange(n, dtype=np.int64) * 2
    _check(a, rng.integers(-3, 2 * n + 3, m))


def test_a_long_array():
    """Around the line from which values are grouped by the parts of the array, and the one from which they are sorted first."""
    n = (1 << 28) + 5
    rng = np.random.default_rng(1)
    a = np.arange(n, dtype=np.int32)
    for m in (1 << 16, 1 << 18, (1 << 18) + 1, 1 << 19, (1 << 19) + 1):
        _check(a, rng.integers(-5, n + 5, m).astype(np.int32))
    a = a[: 1 << 23]
    for m in (1 << 18, (1 << 18) + 1):
        _check(a, rng.integers(-5, a.size + 5, m).astype(np.int32))


@pytest.mark.parametrize("n, m", [(16384, 3 << 19), (16385, 11 << 16), (1 << 19, 11 << 16)])
@pytest.mark.parametrize("dtype", [np.float32, np.int64])
def test_the_line_moves_with_the_array(n, m, dtype):
    """As many values as have a lane each, and one more; a result is asked for in the order of the values."""
    rng = np.random.default_rng(n)
    a = np.arange(n).astype(dtype) * 3
    for k in (m, m + 1):
        _check(a, rng.integers(-3, 3 * n + 3, k).astype(dtype))
