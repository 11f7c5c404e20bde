"""The window search of searchsorted: sorted values in tiles, the array read tile by tile into LDS."""
import ctypes

import numpy as np
import pytest

from cupynumeric_amd import _lib

pytestmark = pytest.mark.gpu


def _search(table, values, left, shift=0):
    import torch

    lib = _lib.load()
    code = _lib.DTYPE_CODES[table.dtype]
    memory = torch.empty(table.nbytes + shift * table.itemsize, dtype=torch.uint8, device="cuda")
    d_a = memory[shift * table.itemsize :]  # off a 16-byte boundary by `shift` elements
    d_a.copy_(torch.from_numpy(table.view(np.uint8)))
    d_v = torch.from_numpy(values.view(np.uint8)).cuda()
    out = torch.full((values.size,), -1, dtype=torch.int64, device="cuda")
    tb = lib.cpn_searchsorted_temp_bytes(code, table.size, values.size)
    assert tb > 0
    temp = torch.empty(tb, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = lib.cpn_searchsorted(
        code, d_a.data_ptr(), table.size, d_v.data_ptr(), values.size, int(left), out.data_ptr(), temp.data_ptr(), tb, stream
    )
    assert rc == 0 and lib.cpn_local_sort_check(temp.data_ptr(), stream) == 0
    return out.cpu().numpy()


@pytest.mark.parametrize("dtype", [np.uint8, np.float16, np.int32, np.float32, np.float64])
@pytest.mark.parametrize("spread", ["even", "clustered", "outside", "equal"])
def test_searchsorted_window_tiles(dtype, spread):
    """Values dense in an array of 64 MiB and more: windows that fit, windows that do not (values
    clustered, so that one tile spans most of the array), empty windows, a ragged last tile."""
    rng = np.random.default_rng(np.dtype(dtype).num)
    n = (64 << 20) // np.dtype(dtype).itemsize + 77
    if np.dtype(dtype).kind == "f":
        a = rng.standard_normal(n).astype(np.float32).astype(dtype)
        a[:1000] = np.nan
        a[1000:2000] = -0.0
    else:
        info = np.iinfo(dtype)
        a = rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)
    a = np.sort(a.astype(np.float32), kind="stable").astype(dtype) if dtype == np.float16 else np.sort(a, kind="stable")
    for m in (n // 60 + 3, n // 12 + 1):
        if spread == "even":
            v = a[rng.integers(0, n, m)]
        elif spread == "clustered":
            v = a[np.concatenate([rng.integers(0, n // 1000, m - 9), rng.integers(0, n, 9)])]
        elif spread == "outside":
            v = np.where(rng.random(m) < 0.5, a[0], a[-1]).astype(dtype)
        else:
            v = np.full(m, a[n // 2])
        for left, shift in ((True, 0), (False, 1)):
            if dtype == np.float16:
                want = np.searchsorted(a.astype(np.float32), v.astype(np.float32), "left" if left else "right")
            else:
                want = np.searchsorted(a, v, "left" if left else "right")
            assert np.array_equal(_search(a, v, left, shift), want), (m, left)


def _labels(call):
    """The kernels that a call launches, and its result."""
    import torch

    lib = _lib.load()
    torch.cuda.synchronize()
    lib.cpn_profile_enable(1)
    _lib.profile_collect()
    try:
        result = call()
        torch.cuda.synchronize()
        return {label for label, _ in _lib.profile_collect()}, result
    finally:
        lib.cpn_profile_enable(0)


@pytest.mark.parametrize("dtype", [np.uint8, np.float16, np.int32, np.float32, np.float64])
@pytest.mark.parametrize("windows", [True, False])
def test_searchsorted_route_at_the_least_values_per_tile(dtype, windows):
    """128 values per tile are the fewest that go by windows: 250 bytes of the array per value do, 262 do not."""
    rng = np.random.default_rng(3)
    n = (64 << 20) // np.dtype(dtype).itemsize + 77
    m = (64 << 20) // (250 if windows else 262)
    runs = {1: 200, 2: 3000}.get(np.dtype(dtype).itemsize, n // 3)  # different elements, half of the numbers between them missing
    step = -(-n // runs)
    a = np.arange(n) // step * 2 % (1 << 24)
    v = rng.integers(0, 2 * runs, m)
    if dtype == np.uint8:
        a, v = a // 2, v // 2
    a, v = np.sort(a).astype(dtype), (v % (1 << 24)).astype(dtype)
    wide = np.float32 if dtype == np.float16 else dtype
    for left in (True, False):
        want = np.searchsorted(a.astype(wide), v.astype(wide), "left" if left else "right")
        for shift in (0, 1):
            labels, got = _labels(lambda: _search(a, v, left, shift))
            assert ("window_bounds" in labels) == windows
            assert np.array_equal(got, want), (left, shift)


@pytest.mark.parametrize("n", [1 << 26, (1 << 26) + 1])
def test_searchsorted_route_of_wide_keys(n):
    """8-byte keys of more than 512 MiB take windows only from 256 values per tile on."""
    a = np.arange(n, dtype=np.float64)
    v = np.random.default_rng(5).integers(0, n, n // 25).astype(np.float64)  # 200 bytes of the array per value
    labels, got = _labels(lambda: _search(a, v, False))
    assert ("window_bounds" in labels) == (n == 1 << 26)
    assert np.array_equal(got, v.astype(np.int64) + 1)


@pytest.mark.parametrize("dtype", [np.uint8, np.int32])
def test_searchsorted_windows_of_an_array_that_is_not_sorted(dtype):
    """Bounds that fall from one tile to the next: the answers mean nothing, but they are positions."""
    rng = np.random.default_rng(9)
    n = (64 << 20) // np.dtype(dtype).itemsize
    info = np.iinfo(dtype)
    a = rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)
    v = rng.integers(info.min, info.max, n // 20, dtype=dtype, endpoint=True)
    for table in (a, np.sort(a)[::-1].copy()):
        got = _search(table, v, True)
        assert got.min() >= 0 and got.max() <= n
