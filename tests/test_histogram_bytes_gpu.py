"""The histogram sweep of 8-byte keys counts bytes that a wave agrees on at once (hist_accumulate_batch of
csrc/onesweep.h), against the oracle, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
from conftest import assert_same_bits
from test_sort_gpu import abi_sort, lib, torch_cuda  # noqa: F401 (fixtures)

from oracle import sort_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def global_passes(lib):
    """(Rows of many of these lengths are merged from sorted pieces by default.)"""
    prev = lib.cpn_set_merge_rows(0)
    yield
    lib.cpn_set_merge_rows(prev)


def _check(lib, torch, x, what):
    want_v = oracle.local_sort(x, argsort=False, threads=8)
    want_i = oracle.local_sort(x, argsort=True, threads=8)
    v, _ = abi_sort(lib, torch, x, want_values=True)
    assert_same_bits(v, want_v, f"{what}: values")
    _, i = abi_sort(lib, torch, x, want_values=False, want_indices=True, offset=5)
    assert_same_bits(i, want_i + 5, f"{what}: positions")
    v, i = abi_sort(lib, torch, x, want_values=True, want_indices=True, in_place=True)
    assert_same_bits(v, want_v, f"{what}: in place")
    assert_same_bits(i, want_i, f"{what}: in place, positions")


@pytest.mark.parametrize("dtype", [np.int64, np.uint64, np.float64])
def test_bytes_that_a_wave_agrees_on(lib, torch_cuda, dtype):
    """Bytes that are constant, constant over long stretches, or differ for one key; a misaligned, ragged end."""
    n = 150_003
    rng = np.random.default_rng(1)
    x = rng.integers(0, 1_000_000, n).astype(np.uint64)
    x += (np.arange(n, dtype=np.uint64) // np.uint64(1024)) << np.uint64(40)
    x[77_777] |= np.uint64(1) << np.uint64(62)
    x[n - 1] |= np.uint64(3) << np.uint64(33)
    x = x.view(dtype)
    if np.dtype(dtype).kind == "f":
        x[5::1000] = np.nan
        x[6::1000] = -0.0
    _check(lib, torch_cuda, np.stack([x, x[::-1]]), f"{np.dtype(dtype)}")
