"""Scatter passes in small tiles (small_sweep_items of csrc/sort_driver.h), their look-back, and the launch that finishes a
sort in which no pass ran, against the oracle, bit for bit."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
from conftest import assert_same_bits, make_input
from test_sort_gpu import abi_sort, lib, torch_cuda  # noqa: F401 (fixtures)

from cupynumeric_amd import _lib
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


# ends of the tiles (4096, 8192 and 16384 keys), of the look-back's windows (16 tiles) and of the ranges of either shape
@pytest.mark.parametrize("dtype,n", [(d, n) for d in (np.float32, np.uint32, np.float64, np.int64)
                                     for n in (4096 * 16, 4096 * 17 + 1, 4096 * 33 - 1, 300_007)]
                         + [(d, n) for d in (np.float32, np.int32) for n in (3 << 18, (3 << 18) + 1, 5 << 19, (5 << 19) + 1)]
                         + [(d, n) for d in (np.float64, np.uint64) for n in (1 << 20, (1 << 20) + 1, 1 << 21, (1 << 21) + 1)])
def test_lengths(lib, torch_cuda, dtype, n):
    _check(lib, torch_cuda, make_input(dtype, (1, n), seed=n % 1000), f"{np.dtype(dtype)} {n}")


@pytest.mark.parametrize("dtype", [np.float32, np.int64])
def test_rows(lib, torch_cuda, dtype):
    """Several rows keep the large tiles."""
    _check(lib, torch_cuda, make_input(dtype, (5, 70_001), seed=3), f"{np.dtype(dtype)} five rows")


@pytest.mark.parametrize("dtype", [np.uint8, np.float16, np.float32, np.int64, np.complex64])
@pytest.mark.parametrize("shape", [(1, 200_001), (2, 100_001)])
def test_all_keys_equal(lib, torch_cuda, dtype, shape):
    _check(lib, torch_cuda, np.full(shape, 7, dtype), f"{np.dtype(dtype)} {shape}")


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_one_byte_varies(lib, torch_cuda, dtype):
    """One pass; in place its result is copied back."""
    x = np.random.default_rng(0).integers(0, 200, (1, 200_003)).astype(dtype)
    _check(lib, torch_cuda, x, f"{np.dtype(dtype)}")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_the_smaller_workspace_is_still_taken(lib, torch_cuda, dtype):
    """A workspace that holds the descriptors of large tiles only gets those."""
    torch = torch_cuda
    n = 262_147
    x = np.random.default_rng(0).standard_normal(n).astype(dtype)
    code = _lib.DTYPE_CODES[x.dtype]
    tb = lib.cpn_local_sort_temp_bytes(code, n, n, 1, 0, 0)
    tiles = lambda size: -(-n // size)  # noqa: E731
    small = tb - x.itemsize * 1024 * (tiles(4096) - tiles(16384))
    a = torch.from_numpy(x).cuda()
    out = torch.empty_like(a)
    ws = torch.empty(small, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.cpn_local_sort(code, a.data_ptr(), out.data_ptr(), None, n, n, 0, 1, ws.data_ptr(), small, stream) == 0
    assert lib.cpn_local_sort_check(ws.data_ptr(), stream) == 0
    assert_same_bits(out.cpu().numpy(), np.sort(x), "values")
    assert lib.cpn_local_sort(code, a.data_ptr(), out.data_ptr(), None, n, n, 0, 1, ws.data_ptr(), small - 256, stream) != 0
