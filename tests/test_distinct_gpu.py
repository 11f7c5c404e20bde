"""unique of integer arrays with few values for their length (csrc/distinct.hip), against the oracle's route through a sort:
the limits of its three ways, frequent values, the key that stands for an empty slot, estimates that are wrong."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
from test_sort_gpu import lib, torch_cuda  # noqa: F401 (fixtures)

import cupynumeric_amd as num
from cupynumeric_amd import _lib

pytestmark = pytest.mark.gpu

TILE = 14336
SHORTEST = {4: 1 << 23, 8: 1 << 22}
EMPTY = 0x9E3779B97F4A7C15  # (4-byte keys: the lower half)


def _array(dtype, n, values, seed, power=1):
    """`n` elements; every one of `values` occurs, the others are random, skewed to the first ones with a power above 1."""
    rng = np.random.default_rng(seed)
    which = (rng.random(n) ** power * len(values)).astype(np.int64)
    which[rng.permutation(n)[: len(values)]] = np.arange(len(values))
    return values[which].astype(dtype)


def _check(x):
    got = np.asarray(num.unique(num.array(x)))
    assert got.dtype == x.dtype and np.array_equal(got, np.unique(x))


def _mode(lib, torch, x):
    """Mode, failure, count and values of the attempt."""
    code = _lib.DTYPE_CODES[x.dtype]
    at = ctypes.c_uint64()
    need = lib.cpn_distinct_temp_bytes(code, x.size, ctypes.byref(at))
    temp = torch.full((need,), 0xA5, dtype=torch.uint8, device="cuda")
    d = torch.from_numpy(x.view(np.uint8).copy()).cuda()
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.cpn_distinct_plan(code, d.data_ptr(), x.size, temp.data_ptr(), need, stream) == 0
    mode = int(temp[:4].view(torch.int32).item())
    if mode == 0:
        return 0, 0, None
    assert lib.cpn_distinct(code, d.data_ptr(), x.size, mode, temp.data_ptr(), need, stream) == 0
    _, failed, count = temp[:12].view(torch.int32).tolist()
    found = temp[at.value : at.value + count * x.itemsize].cpu().numpy().view(x.dtype) if failed == 0 else None
    assert np.array_equal(d.cpu().numpy(), x.view(np.uint8))
    return mode, failed, found


@pytest.mark.parametrize("dtype", [np.int32, np.uint32, np.int64, np.uint64])
@pytest.mark.parametrize("count,power,mode", [(1, 1, 1), (2, 1, 1), (2500, 1, 1), (2500, 8, 1), (9000, 1, 2), (300_000, 1, 2),
                                              (300_000, 6, 2)])
def test_ways(lib, torch_cuda, dtype, count, power, mode):
    key = np.dtype(dtype).itemsize
    rng = np.random.default_rng(count)
    info = np.iinfo(dtype)
    values = np.unique(np.concatenate([rng.integers(info.min, info.max, 2 * count + 8, dtype=dtype, endpoint=True),
                                       np.array([EMPTY], np.uint64).view(np.uint32 if key == 4 else np.uint64)[:1].view(dtype),
                                       np.array([info.min, info.max], dtype)]))
    marker = np.array([EMPTY], np.uint64).view(np.uint32 if key == 4 else np.uint64)[:1].view(dtype)[0]
    others = rng.permutation(values[values != marker])
    for keys in (others[:count], np.append(others[: count - 1], marker) if count > 1 else np.array([marker], dtype)):
        n = SHORTEST[key] + 3 * TILE + 5
        x = _array(dtype, n, keys, count, power)
        got, failed, found = _mode(lib, torch_cuda, x)
        assert (got, failed) == (mode, 0)
        assert np.array_equal(np.sort(found), np.sort(keys))
        _check(x)


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_lengths(dtype):
    """Around the shortest length, and a last tile that is full, of one key, or missing one."""
    first = SHORTEST[np.dtype(dtype).itemsize]
    tiles = -(-first // TILE) * TILE
    for n in (first - 1, first, first + 1, tiles - 1, tiles, tiles + 1):
        for count in (100, 50_000):
            _check(_array(dtype, n, np.arange(count) * 997 - 5000, n, 1))


@pytest.mark.parametrize("dtype", [np.int32, np.int64])
def test_wrong_estimates(lib, torch_cuda, dtype):
    """A sample of a few values before many that are seen once: the tables fill up and the array is sorted."""
    key = np.dtype(dtype).itemsize
    n = SHORTEST[key]
    rng = np.random.default_rng(1)
    x = rng.integers(0, 100, n).astype(dtype)
    x[rng.permutation(n)[:20_000]] = (np.arange(20_000) * 2 + 100_000).astype(dtype)
    mode, failed, _ = _mode(lib, torch_cuda, x)
    assert (mode, failed) == (1, 1)
    _check(x)
    if key == 8:  # very unlike frequencies
        x = _array(dtype, 1 << 23, np.arange(1 << 22) * 3 - 77, 2, power=6)
        mode, failed, _ = _mode(lib, torch_cuda, x)
        assert (mode, failed) == (2, 1)
        _check(x)
    # one value, and a second that the sample has not seen
    x = np.full(n, 7, dtype)
    x[12345] = -7
    _check(x)
    _check(np.full(n, 7, dtype))


def test_unaligned_input_and_wrong_mode(lib, torch_cuda):
    """16-byte reads start behind an unaligned head; a mode that the sample did not give ends the attempt."""
    torch = torch_cuda
    n = SHORTEST[4] + 9
    x = _array(np.int32, n + 1, np.arange(777) * 3, 5)
    d = torch.from_numpy(x).cuda()
    at = ctypes.c_uint64()
    code = _lib.DTYPE_CODES[np.dtype(np.int32)]
    need = lib.cpn_distinct_temp_bytes(code, n, ctypes.byref(at))
    temp = torch.empty(need, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    args = (code, d.data_ptr() + 4, n)
    assert lib.cpn_distinct_plan(*args, temp.data_ptr(), need, stream) == 0
    assert lib.cpn_distinct(*args, 1, temp.data_ptr(), need, stream) == 0
    mode, failed, count = temp[:12].view(torch.int32).tolist()
    assert (mode, failed) == (1, 0)
    found = temp[at.value : at.value + 4 * count].view(torch.int32).cpu().numpy()
    assert np.array_equal(np.sort(found), np.unique(x[1:]))
    assert lib.cpn_distinct(*args, 2, temp.data_ptr(), need, stream) == 0
    assert temp[4:8].view(torch.int32).item() == 1


@pytest.mark.parametrize("dtype", [np.int32, np.uint32, np.float32, np.int64, np.float64])
@pytest.mark.parametrize("n", [6145, 8193, 100_000, 1 << 20, (1 << 20) + 1, 1 << 21, (1 << 21) + 1])
@pytest.mark.parametrize("count", [5, 3000, 1 << 40])
def test_sorted_by_a_split(dtype, n, count):
    """Arrays whose sort is split by sampled keys, and their neighbours; NaNs and zeros of both signs among floats."""
    rng = np.random.default_rng(n + count % 97)
    x = rng.integers(-(1 << 30), 1 << 30, min(count, n))[rng.integers(0, min(count, n), n)]
    x = (np.abs(x) if np.dtype(dtype).kind == "u" else x).astype(dtype)
    if np.dtype(dtype).kind == "f":
        x[rng.integers(0, n, 50)] = np.nan
        x[rng.integers(0, n, 50)] = -0.0
        x[rng.integers(0, n, 50)] = 0.0
    got = np.asarray(num.unique(num.array(x)))
    assert got.dtype == x.dtype and np.array_equal(got, np.unique(x), equal_nan=x.dtype.kind == "f")


def test_codes_of_the_entry_points(lib, torch_cuda):
    torch = torch_cuda
    code, n = _lib.DTYPE_CODES[np.dtype(np.int64)], 1 << 22
    need = lib.cpn_distinct_temp_bytes(code, n, None)
    d = torch.zeros(n, dtype=torch.int64, device="cuda")
    temp = torch.empty(need, dtype=torch.uint8, device="cuda")
    for call in (lambda *a: lib.cpn_distinct_plan(*a, None), lambda c, v, m, t, b: lib.cpn_distinct(c, v, m, 1, t, b, None)):
        assert call(99, d.data_ptr(), n, temp.data_ptr(), need) == _lib.CPN_ERR_DTYPE
        assert call(code, d.data_ptr(), n - 1, temp.data_ptr(), need) == _lib.CPN_ERR_UNSUPPORTED
        assert call(code, None, n, temp.data_ptr(), need) == _lib.CPN_ERR_NULL
        assert call(code, d.data_ptr(), n, temp.data_ptr(), need - 1) == _lib.CPN_ERR_TEMP
        assert call(code, d.data_ptr(), n, temp.data_ptr() + 8, need) == _lib.CPN_ERR_TEMP
        assert call(code, d.data_ptr() + 4, n, temp.data_ptr(), need) == _lib.CPN_ERR_ALIGN
    assert lib.cpn_distinct(code, d.data_ptr(), n, 3, temp.data_ptr(), need, None) == _lib.CPN_ERR_UNSUPPORTED
    small = lib.cpn_unique_sorted_temp_bytes(code, 5000)
    count = torch.zeros(1, dtype=torch.int64, device="cuda")
    call = lib.cpn_unique_sorted
    assert call(99, d.data_ptr(), d.data_ptr(), 5000, count.data_ptr(), temp.data_ptr(), small, None) == _lib.CPN_ERR_DTYPE
    assert call(code, d.data_ptr(), None, 5000, count.data_ptr(), temp.data_ptr(), small, None) == _lib.CPN_ERR_NULL
    assert call(code, d.data_ptr(), d.data_ptr(), 0, count.data_ptr(), temp.data_ptr(), small, None) == _lib.CPN_ERR_UNSUPPORTED
    assert call(code, d.data_ptr(), d.data_ptr(), 5000, count.data_ptr(), temp.data_ptr(), small - 1, None) == _lib.CPN_ERR_TEMP
    assert call(code, d.data_ptr(), d.data_ptr(), 5000, count.data_ptr() + 4, temp.data_ptr(), small, None) == _lib.CPN_ERR_ALIGN


@pytest.mark.parametrize("mode", ["lazy", "eager", "off"])
def test_status_of_the_sort_of_the_values(torch_cuda, monkeypatch, mode):
    """2^20 and more values of 4 bytes are sorted by passes, which can fail on the device: `unique` has looked when it returns."""
    from cupynumeric_amd import _thunk
    from cupynumeric_amd.runtime import runtime

    x = _array(np.int32, 1 << 23, np.arange(1_500_000, dtype=np.int32) * 1000, 3)
    a = num.array(x)
    monkeypatch.setattr(runtime, "check_mode", mode)
    assert np.array_equal(np.asarray(num.unique(a)), np.unique(x))
    if mode != "lazy":
        return
    num.unique(a)
    assert runtime._status_used == 0
    sort = _thunk.sort_task

    def failing(*args):
        sort(*args)
        runtime.defer_flag(torch_cuda.ones(1, dtype=torch_cuda.int32, device="cuda"), "sort")

    monkeypatch.setattr(_thunk, "sort_task", failing)
    with pytest.raises(RuntimeError, match="failed on the device"):
        num.unique(a)


@pytest.mark.parametrize("dtype, n, values, tried", [
    (np.int64, 1 << 25, 1 << 24, False),  # 5.2 million different ones: more than the tables hold
    (np.int64, 1 << 23, 1 << 22, True),  # 1.4 million
    (np.int32, 1 << 24, 1 << 23, True),  # 2.7 million
    (np.uint64, (1 << 24) + 9, 1 << 17, True),
])
def test_values_whose_frequencies_fall_with_their_rank(lib, torch_cuda, dtype, n, values, tried):
    """Chao's estimate of them is far too low (47 000 of the first); what the second one does not believe is not tried."""
    x = (float(values) ** np.random.default_rng(values).random(n)).astype(dtype) * dtype(97)
    if tried:
        mode, failed, found = _mode(lib, torch_cuda, x)
        assert (mode, failed) == (2, 0) and np.array_equal(np.sort(found), np.unique(x))
    a = num.array(x)
    num.unique(a)
    lib.cpn_profile_enable(1)
    try:
        _lib.profile_collect()
        got = np.asarray(num.unique(a))
        labels = [label for label, _ in _lib.profile_collect()]
    finally:
        lib.cpn_profile_enable(0)
    assert np.array_equal(got, np.unique(x))
    assert "collect_plan" in labels and ("collect_class" in labels) == tried, labels


@pytest.mark.parametrize("dtype", [np.int32, np.uint64])
@pytest.mark.parametrize("power, tried", [(1.5, False), (2.0, True)])
def test_frequencies_that_fall_as_a_power_of_the_rank(lib, torch_cuda, dtype, power, tried):
    """As word counts do.  Of the power of 1.5 there are 69 000 different ones and the estimate says under 3000: it is not tried, and where it is,
    the table in memory fills up.  Of the power of 2 there are 5000, which it holds."""
    x = np.minimum((1 - np.random.default_rng(5).random(1 << 23)) ** (-1 / (power - 1)), 2e9).astype(dtype)
    mode, failed, found = _mode(lib, torch_cuda, x)
    assert (mode, failed) == (1, 0 if tried else 1)
    assert not tried or np.array_equal(np.sort(found), np.unique(x))
    a = num.array(x)
    num.unique(a)
    lib.cpn_profile_enable(1)
    try:
        _lib.profile_collect()
        got = np.asarray(num.unique(a))
        labels = [label for label, _ in _lib.profile_collect()]
    finally:
        lib.cpn_profile_enable(0)
    assert np.array_equal(got, np.unique(x))
    assert "collect_plan" in labels and ("collect_few" in labels) == tried, labels


@pytest.mark.parametrize("n", [3 << 20, (3 << 20) + 1])
@pytest.mark.parametrize("count", [300, 1 << 40])
def test_the_longest_integers_that_are_split(n, count):
    rng = np.random.default_rng(n)
    _check(rng.integers(-(1 << 40), 1 << 40, min(count, n))[rng.integers(0, min(count, n), n)])
