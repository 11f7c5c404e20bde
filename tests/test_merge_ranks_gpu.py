"""Requests of few keys whose sorted pieces are merged by rank in one launch (csrc/merge_rows.h), against the
oracle, bit for bit: lengths at the ends of pieces, chunks and of the path itself, ties across pieces, rows whose
pieces do not overlap or lie inside one another (windows of no key and of whole pieces), special values."""
from __future__ import annotations

import numpy as np
import pytest
from conftest import assert_same_bits, make_input
from test_sort_gpu import abi_sort, lib, torch_cuda  # noqa: F401 (fixtures)

from oracle import sort_oracle as oracle

pytestmark = pytest.mark.gpu


def _check(lib, torch, x, what):
    want_v = oracle.local_sort(x, argsort=False, threads=8)
    want_i = oracle.local_sort(x, argsort=True, threads=8)
    v, _ = abi_sort(lib, torch, x, want_values=True)
    assert_same_bits(v, want_v, f"{what}: values")
    _, i = abi_sort(lib, torch, x, want_values=False, want_indices=True, offset=3)
    assert_same_bits(i, want_i + 3, f"{what}: positions")
    v, i = abi_sort(lib, torch, x, want_values=True, want_indices=True, in_place=True)
    assert_same_bits(v, want_v, f"{what}: in place")
    assert_same_bits(i, want_i, f"{what}: in place, positions")


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32, np.uint64])
@pytest.mark.parametrize("n", [8193, 12289, 16385, 40000, 40001, 80001, 100000, 131071, 212992, 262144])
def test_lengths(lib, torch_cuda, dtype, n):
    _check(lib, torch_cuda, make_input(dtype, (1, n), seed=n), f"{np.dtype(dtype)} {n}")


@pytest.mark.parametrize("dtype", [np.float64, np.int32])
def test_rows_and_arrangements(lib, torch_cuda, dtype):
    n = 30_000
    rng = np.random.default_rng(3)
    rows = np.stack([
        np.arange(n), np.arange(n)[::-1], np.full(n, 4), rng.integers(0, 3, n),
        # one piece spread thinly over what the others hold densely, and the reverse
        np.where(np.arange(n) < 4000, rng.integers(0, 1 << 30, n), rng.integers(5000, 6000, n)),
        np.where(np.arange(n) < 4000, rng.integers(5000, 6000, n), rng.integers(0, 1 << 30, n)),
        np.arange(n) // 300,
    ]).astype(dtype)
    _check(lib, torch_cuda, rows, f"{np.dtype(dtype)} arrangements")
    _check(lib, torch_cuda, make_input(dtype, (3, 70_001), seed=9), f"{np.dtype(dtype)} three rows")


def test_level_by_level_still_agrees(lib, torch_cuda):
    """The other way of merging at lengths that the default no longer sends there."""
    prev = lib.cpn_set_merge_rows(8)
    try:
        _check(lib, torch_cuda, make_input(np.float64, (2, 60_001), seed=5), "level by level")
        _check(lib, torch_cuda, make_input(np.float32, (1, 33_000), seed=6), "level by level")
    finally:
        lib.cpn_set_merge_rows(prev)


def _unlike(kind, n, rng):
    x = rng.random(n)
    if kind == "one piece wide":
        x[8192:] = 0.5 + 1e-3 * x[8192:]
    elif kind == "halves":
        x[n // 2 :] = 0.5 + 1e-3 * x[n // 2 :]
    elif kind == "ties":  # whole pieces of one value between two neighbouring keys of another
        x[8192:] = 0.5
        x[4000:4200] = 0.5
    return x


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("kind", ["one piece wide", "halves", "ties"])
@pytest.mark.parametrize("n", [24_577, 40_001, 100_003, 212_991])
def test_unlike_pieces(lib, torch_cuda, dtype, kind, n):
    """Windows too wide for LDS are searched in memory: some of the pieces, nearly all, the short last one."""
    x = _unlike(kind, n, np.random.default_rng(n)).astype(dtype)
    _check(lib, torch_cuda, x.reshape(1, -1), f"{np.dtype(dtype)} {n} {kind}")


def test_unlike_pieces_take_no_multiple_of_the_time(torch_cuda):
    """A workgroup whose windows span the row once copied all of it: 5.4 times what evenly mixed keys take; now the same."""
    import cupynumeric_amd as num

    torch = torch_cuda
    n = 262_144

    def best(x):
        a = num.array(x)
        times = []
        for _ in range(20):
            start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            start.record()
            for _ in range(5):
                num.sort(a)
            end.record()
            end.synchronize()
            times.append(start.elapsed_time(end))
        return min(times)

    rng = np.random.default_rng(0)
    even = best(rng.random(n).astype(np.float32))
    for kind in ("one piece wide", "halves"):
        assert best(_unlike(kind, n, rng).astype(np.float32)) < 2.2 * even, kind


def _merged_by_rank(lib, torch, x, argsort):
    import ctypes

    lib.cpn_profile_enable(1)
    try:
        abi_sort(lib, torch, x, want_values=not argsort, want_indices=argsort)
    finally:
        lib.cpn_profile_enable(0)
    labels, ms = ctypes.create_string_buffer(64 * 64), (ctypes.c_float * 64)()
    count = lib.cpn_profile_collect(labels, 64, ms, 64)
    return any(labels.raw[64 * i : 64 * i + 11] == b"merge_ranks" for i in range(count))


@pytest.mark.parametrize("dtype,argsort,first,last", [
    (np.float32, False, 12_289, 262_144), (np.int32, True, 12_289, 262_144),
    (np.float64, False, 10_241, 212_992), (np.float64, True, 9217, 262_144),
    (np.int64, False, 10_241, 163_840), (np.uint64, True, 9217, 212_992)])
def test_the_lines_of_the_path(lib, torch_cuda, dtype, argsort, first, last):
    """Rows outside them are sorted sooner the other way (int64 with positions, 262 144: 94 us against 110)."""
    for n, by_rank in ((first - 1, False), (first, True), (last, True), (last + 1, False)):
        assert _merged_by_rank(lib, torch_cuda, make_input(dtype, (1, n), seed=n), argsort) == by_rank, n
