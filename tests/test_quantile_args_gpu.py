"""cpn_quantile_sorted_args: positions and weights in host memory, against the call that reads them from the device."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
from conftest import assert_same_bits
from test_sort_gpu import lib, torch_cuda  # noqa: F401 (fixtures)

import cupynumeric_amd as num
from cupynumeric_amd import _lib, _stats
from oracle import sort_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.bool_, np.int8, np.uint16, np.int32, np.uint64, np.float16, np.float32, np.float64])
@pytest.mark.parametrize("interpolate", [0, 1])
def test_same_as_from_the_device(lib, torch_cuda, dtype, interpolate):
    torch, rng = torch_cuda, np.random.default_rng(3)
    outer, n, inner = 3, 101, 5
    x = np.sort((rng.standard_normal((outer, n, inner)) * 50).astype(dtype), axis=1)
    d = torch.from_numpy(x.view(np.uint8)).cuda()
    code, stream = _lib.DTYPE_CODES[x.dtype], ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    for num_q in (1, 2, 15, 16):
        left = rng.integers(0, n, num_q)
        right, gamma = np.minimum(left + 1, n - 1), rng.random(num_q)
        size = num_q * outer * inner * (8 if interpolate else x.itemsize)
        outs = [torch.full((size,), 0x5A, dtype=torch.uint8, device="cuda") for _ in range(2)]
        on_device = [torch.from_numpy(a).cuda() for a in (left, right, gamma)]
        args = (code, d.data_ptr(), outer, n, inner, num_q)
        assert lib.cpn_quantile_sorted(*args, *(a.data_ptr() for a in on_device), interpolate, outs[0].data_ptr(), stream) == 0
        assert lib.cpn_quantile_sorted_args(*args, *(a.ctypes.data for a in (left, right, gamma)), interpolate, outs[1].data_ptr(),
                                            stream) == 0
        assert torch.equal(*outs)
    call = lib.cpn_quantile_sorted_args
    left = np.zeros(17, np.int64)
    rest = (left.ctypes.data, left.ctypes.data, np.zeros(17).ctypes.data, 1, outs[0].data_ptr(), stream)
    assert call(code, d.data_ptr(), outer, n, inner, 17, *rest) == _lib.CPN_ERR_UNSUPPORTED
    assert call(code, d.data_ptr(), outer, 0, inner, 1, *rest) == _lib.CPN_ERR_SHAPE
    assert call(code, d.data_ptr(), outer, n, inner, 0, *rest) == 0 and call(code, d.data_ptr(), 0, n, inner, 1, *rest) == 0
    assert call(code, None, outer, n, inner, 1, *rest) == _lib.CPN_ERR_NULL and call(99, None, outer, n, inner, 1, *rest) == _lib.CPN_ERR_DTYPE
    left[0] = n
    assert call(code, d.data_ptr(), outer, n, inner, 1, *rest) == _lib.CPN_ERR_SHAPE
    left[0] = -1
    assert call(code, d.data_ptr(), outer, n, inner, 1, *rest) == _lib.CPN_ERR_SHAPE


@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int64])
def test_lengths_around_the_line_of_the_selection(dtype):
    rng = np.random.default_rng(4)
    for n in (_stats.SELECT_MIN_SIZE, 4 * _stats.SELECT_MIN_SIZE):
        for m in (n - 1, n):
            x = (rng.standard_normal(m) * 1000).astype(dtype)
            if np.dtype(dtype).kind == "f":
                x[rng.integers(0, m, 20)] = -0.0
            for q in ([50.0], [5.0, 25.0, 50.0, 75.0, 95.0], list(np.linspace(0, 100, 17))):
                assert_same_bits(np.asarray(num.percentile(num.array(x), q)), oracle.percentile(x, q), f"{m} {q}")


@pytest.mark.parametrize("dtype, two, three, nine", [(np.float32, 1, 2, 2), (np.int32, 1, 1, 2), (np.float64, 2, 2, 2), (np.int64, 2, 2, 2)])
def test_which_vectors_are_selected_from(dtype, two, three, nine):
    """By the launches, at the lines of two, three and nine quantiles, and one element before."""
    lib = _lib.load()
    rng = np.random.default_rng(5)
    for q, times in (([25.0, 75.0], two), ([25.0, 50.0, 75.0], three), (list(np.linspace(10, 90, 9)), nine)):
        line = times * _stats.SELECT_MIN_SIZE
        for n in (line - 1, line):
            x = (rng.standard_normal(n) * 1e6).astype(dtype)
            a = num.array(x)
            lib.cpn_profile_enable(1)
            try:
                _lib.profile_collect()
                got = np.asarray(num.percentile(a, q))
                labels = {label for label, _ in _lib.profile_collect()}
            finally:
                lib.cpn_profile_enable(0)
            assert_same_bits(got, oracle.percentile(x, q), f"{np.dtype(dtype)} {n} {q}")
            assert any(label.startswith("select") for label in labels) == (n == line), (n, q, labels)
