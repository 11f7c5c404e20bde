"""searchsorted of many values by the parts of the array (csrc/grouped_search.hip), against numpy: lengths at which the parts
and their windows change, values that crowd a part or a tile, batches, and what the entry point refuses."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
from test_sort_gpu import lib, torch_cuda  # noqa: F401 (fixtures)

from cupynumeric_amd import _lib

pytestmark = pytest.mark.gpu

TILE, PARTS, WINDOW = 16384, 2048, 32768  # values; parts; bytes of a window
LEAST = 8 << 20  # bytes


def _search(lib, torch, d_a, a, v, left):
    code = _lib.DTYPE_CODES[a.dtype]
    need = lib.cpn_searchsorted_grouped_temp_bytes(code, d_a.data_ptr(), a.size, v.size)
    assert need != 0
    d_v = torch.from_numpy(v.view(np.uint8)).cuda()
    out = torch.full((v.size + 1,), -1, dtype=torch.int64, device="cuda")
    temp = torch.full((need,), 0xA5, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = lib.cpn_searchsorted_grouped(code, d_a.data_ptr(), a.size, d_v.data_ptr(), v.size, int(left), out.data_ptr(),
                                      temp.data_ptr(), need, stream)
    assert rc == 0, _lib.status_string(rc)
    got = out.cpu().numpy()
    assert got[-1] == -1 and np.array_equal(d_v.cpu().numpy(), v.view(np.uint8))
    return got[:-1]


def _table(dtype, n, rng):
    if np.dtype(dtype).kind == "f":
        a = rng.standard_normal(n).astype(dtype)
        a[:500], a[500:1000], a[1000:1500] = np.nan, -0.0, np.inf
        a[1500:2000] = -np.inf
    else:
        info = np.iinfo(dtype)
        a = rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)
        a[:500], a[500:900] = info.max, info.min
        a[900:5000] = 7  # a run over a window's end
    return np.sort(a, kind="stable")


def _check(lib, torch, a, values):
    d_a = torch.from_numpy(a.view(np.uint8)).cuda()
    for what, v in values:
        for left in (True, False):
            got = _search(lib, torch, d_a, a, v, left)
            assert np.array_equal(got, np.searchsorted(a, v, "left" if left else "right")), (a.dtype, a.size, what, v.size, left)


@pytest.mark.parametrize("dtype", [np.int32, np.uint32, np.float32, np.int64, np.uint64, np.float64])
def test_spreads(lib, torch_cuda, dtype):
    rng = np.random.default_rng(np.dtype(dtype).num)
    n = LEAST // np.dtype(dtype).itemsize + 77
    a = _table(dtype, n, rng)
    m = (1 << 16) + 3 * TILE + 5
    hot = a[n // 3 : n // 3 + 200]
    _check(lib, torch_cuda, a, [
        ("even", a[rng.integers(0, n, m)]),
        ("between", (a[rng.integers(0, n, m)] * dtype(0.999)).astype(dtype) if np.dtype(dtype).kind == "f" else a[rng.integers(0, n, m)] ^ dtype(1)),
        ("clustered", np.where(rng.random(m) < 0.9, hot[rng.integers(0, hot.size, m)], a[rng.integers(0, n, m)])),
        ("equal", np.full(m, a[n // 2])),
        ("ends", np.where(rng.random(m) < 0.5, a[0], a[-1]).astype(dtype)),
        ("largest key", np.full(m, np.nan if np.dtype(dtype).kind == "f" else np.iinfo(dtype).max, dtype)),
        ("ascending", np.sort(a[rng.integers(0, n, m)])),
    ])


@pytest.mark.parametrize("dtype", [np.float32, np.int64])
@pytest.mark.parametrize("shift", [-1, 0, 1, 3])
def test_lengths(lib, torch_cuda, dtype, shift):
    """One window per part and more, a last part or window of few elements; a last tile that is full, of one value, or missing one."""
    key = np.dtype(dtype).itemsize
    per = WINDOW // key
    rng = np.random.default_rng(shift + 5)
    for n in (LEAST // key + per + shift + 1, PARTS * per + shift, 2 * PARTS * per + shift, 3 * PARTS * per // 2 + per + shift):
        a = _table(dtype, n, rng)
        _check(lib, torch_cuda, a, [("even", a[rng.integers(0, n, (1 << 17) + shift + 1)])])


def test_pieces_and_batches(lib, torch_cuda):
    """More values of one part than a piece takes, and more values than a batch has (2^24)."""
    torch, n = torch_cuda, LEAST // 4
    a = np.arange(n, dtype=np.int32) * 3
    rng = np.random.default_rng(3)
    few = rng.integers(0, 3 * 8192, 300_000).astype(np.int32)
    _check(lib, torch, a, [("one part", few), ("one element", np.full(300_000, 299, np.int32))])
    v = torch.randint(0, 3 * n, ((1 << 24) + TILE + 1,), dtype=torch.int32, device="cuda").cpu().numpy()
    d_a = torch.from_numpy(a.view(np.uint8)).cuda()
    assert np.array_equal(_search(lib, torch, d_a, a, v, True), (v.astype(np.int64) + 2) // 3)


def test_not_sorted(lib, torch_cuda):
    """An array that is not sorted: some answer in its range for each value."""
    rng = np.random.default_rng(8)
    a = rng.integers(-1000, 1000, LEAST // 4 + 5, dtype=np.int32)
    d_a = torch_cuda.from_numpy(a.view(np.uint8)).cuda()
    got = _search(lib, torch_cuda, d_a, a, rng.integers(-1100, 1100, 100_000, dtype=np.int32), True)
    assert got.min() >= 0 and got.max() <= a.size


def test_requests_and_codes(lib, torch_cuda):
    torch, size = torch_cuda, lib.cpn_searchsorted_grouped_temp_bytes
    f4, f8, f2, c8 = (_lib.DTYPE_CODES[np.dtype(t)] for t in (np.float32, np.float64, np.float16, np.complex64))
    n, m = LEAST // 4, 1 << 16
    a = torch.zeros(n + 4, dtype=torch.float32, device="cuda")
    v = torch.zeros(m, dtype=torch.float32, device="cuda")
    out = torch.zeros(m, dtype=torch.int64, device="cuda")
    p = a.data_ptr()
    assert size(f4, p, n, m) != 0 and size(f8, p, n // 2, m) != 0
    assert size(f4, p, n - 1, m) == 0 and size(f4, p, n, m - 1) == 0 and size(f4, p + 4, n, m) == 0
    assert size(f2, p, 2 * n, m) == 0 and size(c8, p, n, m) == 0 and size(99, p, n, m) == 0
    assert size(f4, p, 1 << 28, 1 << 21) != 0 and size(f4, p, 1 << 28, (1 << 21) - 1) == 0  # past 512 MiB: 512 bytes per value
    assert size(f8, p, 1 << 27, 1 << 20) != 0 and size(f8, p, 1 << 27, (1 << 20) - 1) == 0
    assert size(f4, p, 1 << 30, 1 << 24) != 0 and size(f4, p, (1 << 30) + 4096, 1 << 24) == 0  # 64 windows per part
    assert size(f8, p, 1 << 29, 1 << 24) != 0 and size(f8, p, (1 << 29) + 4096, 1 << 24) == 0
    need = size(f4, p, n, m)
    temp = torch.zeros(need + 256, dtype=torch.uint8, device="cuda")
    call = lib.cpn_searchsorted_grouped
    t = temp.data_ptr()
    assert call(99, p, n, v.data_ptr(), m, 1, out.data_ptr(), t, need, None) == _lib.CPN_ERR_DTYPE
    assert call(f4, p, n - 1, v.data_ptr(), m, 1, out.data_ptr(), t, need, None) == _lib.CPN_ERR_UNSUPPORTED
    assert call(f4, None, n, v.data_ptr(), m, 1, out.data_ptr(), t, need, None) == _lib.CPN_ERR_NULL
    assert call(f4, p, n, v.data_ptr() + 2, m, 1, out.data_ptr(), t, need, None) == _lib.CPN_ERR_ALIGN
    assert call(f4, p, n, v.data_ptr(), m, 1, out.data_ptr() + 4, t, need, None) == _lib.CPN_ERR_ALIGN
    assert call(f4, p, n, v.data_ptr(), m, 1, out.data_ptr(), t, need - 1, None) == _lib.CPN_ERR_TEMP
    assert call(f4, p, n, v.data_ptr(), m, 1, out.data_ptr(), t + 8, need, None) == _lib.CPN_ERR_TEMP


def test_captured(lib, torch_cuda):
    """Every replay counts its pieces anew: other values, spread otherwise, into the same graph."""
    torch, rng = torch_cuda, np.random.default_rng(6)
    n, m = LEAST // 4 + 9, 100_000
    a = np.sort(rng.standard_normal(n).astype(np.float32))
    code = _lib.DTYPE_CODES[a.dtype]
    d_a = torch.from_numpy(a).cuda()
    buf = torch.zeros(m, dtype=torch.float32, device="cuda")
    out = torch.full((m,), -1, dtype=torch.int64, device="cuda")
    need = lib.cpn_searchsorted_grouped_temp_bytes(code, d_a.data_ptr(), n, m)
    temp = torch.full((need,), 0xA5, dtype=torch.uint8, device="cuda")

    def search():
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        return lib.cpn_searchsorted_grouped(code, d_a.data_ptr(), n, buf.data_ptr(), m, 1, out.data_ptr(), temp.data_ptr(), need, stream)

    assert need != 0 and search() == 0
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        assert search() == 0
    for spread in (1.0, 0.001, 100.0, 1.0):
        x = (rng.standard_normal(m) * spread).astype(np.float32)
        buf.copy_(torch.from_numpy(x))
        out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), np.searchsorted(a, x)), spread


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_the_public_call_comes_here(lib, torch_cuda, dtype):
    """The launches of the public call from the line on, and one value below it."""
    import cupynumeric_amd as num
    from cupynumeric_amd._thunk import GROUPED_MIN_VALUES

    rng = np.random.default_rng(9)
    a = np.sort(rng.standard_normal(LEAST // np.dtype(dtype).itemsize + 5).astype(dtype))
    d_a = num.array(a)
    for m, grouped in ((GROUPED_MIN_VALUES, True), (GROUPED_MIN_VALUES - 1, False)):
        v = rng.standard_normal(m).astype(dtype)
        d_v = num.array(v)
        lib.cpn_profile_enable(1)
        try:
            _lib.profile_collect()
            got = np.asarray(num.searchsorted(d_a, d_v))
            labels = {label for label, _ in _lib.profile_collect()}
        finally:
            lib.cpn_profile_enable(0)
        assert np.array_equal(got, np.searchsorted(a, v))
        assert ({"find_group", "find_search"} <= labels) == grouped, labels
