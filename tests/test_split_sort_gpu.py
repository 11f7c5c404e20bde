"""Single rows that are split by sampled keys and sorted part by part (csrc/split_sort.h), against the oracle, bit for bit:
lengths at which the plan changes, keys that crowd the sample's bins or a bucket's, buckets that do not fit in LDS."""
from __future__ import annotations

import ctypes
import threading

import numpy as np
import pytest
from conftest import assert_same_bits, make_input
from test_sort_gpu import lib, torch_cuda  # noqa: F401 (fixtures)

import cupynumeric_amd as num
from cupynumeric_amd import _lib
from oracle import sort_oracle as oracle

pytestmark = pytest.mark.gpu


def _split_sort(lib, torch, x, want_values, want_indices, in_place=False, offset=0):
    code, n = _lib.DTYPE_CODES[x.dtype], x.size
    tb = lib.cpn_local_sort_split_temp_bytes(code, n, n, int(want_indices))
    assert tb != 0, (x.dtype, n)
    d_in = torch.from_numpy(x.view(np.uint8).copy()).cuda()
    d_val = d_in if in_place else (torch.zeros_like(d_in) if want_values else None)
    d_idx = torch.full((n,), -7, dtype=torch.int64, device="cuda") if want_indices else None
    temp = torch.full((tb,), 0xFF, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    rc = lib.cpn_local_sort_ex(code, d_in.data_ptr(), d_val.data_ptr() if d_val is not None else None,
                               d_idx.data_ptr() if want_indices else None, n, n, offset, 1, _lib.CPN_SORT_SPLIT, temp.data_ptr(),
                               tb, stream)
    assert rc == 0, _lib.status_string(rc)
    assert lib.cpn_local_sort_check(temp.data_ptr(), stream) == 0
    if not in_place:
        assert np.array_equal(d_in.cpu().numpy(), x.view(np.uint8))
    return (d_val.cpu().numpy().view(x.dtype) if d_val is not None else None,
            d_idx.cpu().numpy() if want_indices else None)


def _check(lib, torch, x, what):
    want_v = oracle.local_sort(x.reshape(1, -1), argsort=False, threads=8)[0]
    want_i = oracle.local_sort(x.reshape(1, -1), argsort=True, threads=8)[0]
    v, _ = _split_sort(lib, torch, x, True, False)
    assert_same_bits(v, want_v, f"{what}: values")
    _, i = _split_sort(lib, torch, x, False, True, offset=3)
    assert_same_bits(i, want_i + 3, f"{what}: positions")
    v, i = _split_sort(lib, torch, x, True, True, in_place=True)
    assert_same_bits(v, want_v, f"{what}: in place")
    assert_same_bits(i, want_i, f"{what}: in place, positions")


# shortest and longest row, and where the number of buckets, of sampled keys and of tiles changes
EDGES = [8193, 65536, 65537, 131072, 131073, 262144, 262145, 524288, 524289, (1 << 20) - 1, 1 << 20]


@pytest.mark.parametrize("dtype", [np.float32, np.int32, np.uint32, np.float64, np.int64, np.uint64])
@pytest.mark.parametrize("n", EDGES)
def test_lengths(lib, torch_cuda, dtype, n):
    _check(lib, torch_cuda, make_input(dtype, (n,), seed=n % 1000), f"{np.dtype(dtype)} {n}")


# 8-byte keys only; from 2^20 the sample is sorted ahead (ends of the numbers of buckets, of sampled keys and of tiles)
@pytest.mark.parametrize("dtype", [np.float64, np.int64, np.uint64])
@pytest.mark.parametrize("n", [6145, 8192, (1 << 20) + 1, 1024 * 1365, 1024 * 1365 + 1, 1 << 21, (1 << 21) + 1, 256 * 14336, 256 * 14336 + 1,
                               1 << 22, (1 << 22) + 1, 4096 * 2048 + 1, 4096 * 2560])
def test_lengths_of_wide_keys(lib, torch_cuda, dtype, n):
    _check(lib, torch_cuda, make_input(dtype, (n,), seed=n), f"{np.dtype(dtype)} {n}")


def _kind(kind, dtype, n):
    rng = np.random.default_rng(n)
    if kind == "equal":
        x = np.full(n, 7)
    elif kind == "two values":
        x = rng.integers(0, 2, n) * 1000
    elif kind == "hundred values":
        x = rng.integers(0, 1 << 62, 100)[rng.integers(0, 100, n)] if np.dtype(dtype).itemsize == 8 else rng.integers(0, 100, n) * 20_000_000
    elif kind == "ascending":
        x = np.arange(n)
    elif kind == "descending":
        x = n - np.arange(n)
    elif kind == "runs":  # neighbours are alike
        x = np.repeat(rng.integers(0, 1 << 30, n // 50 + 1), 50)[:n]
    elif kind == "magnitudes":  # crowds the bins of the sample
        x = np.exp(rng.standard_normal(n) * 4) * (1 if np.dtype(dtype).kind == "f" else 100)
    elif kind == "cluster":  # half of the keys in a range that one bin of the sample covers
        x = np.where(rng.random(n) < 0.5, rng.integers(0, 1 << 30, n), 1000 + rng.integers(0, 50, n))
    elif kind == "far":  # finite values whose span overflows, infinities, NaNs
        x = rng.standard_normal(n)
        if np.dtype(dtype).kind == "f":
            big = np.finfo(dtype).max
            x[rng.integers(0, n, 50)] = big
            x[rng.integers(0, n, 50)] = -big
            x[rng.integers(0, n, 50)] = np.inf
            x[rng.integers(0, n, 50)] = -np.inf
            x[rng.integers(0, n, n // 20)] = np.nan
            x[rng.integers(0, n, n // 20)] = -0.0
            x[rng.integers(0, n, n // 20)] = 0.0
        else:
            x = rng.integers(np.iinfo(dtype).min, np.iinfo(dtype).max, n, dtype=dtype, endpoint=True)
    if np.dtype(dtype).kind != "f" and x.dtype.kind == "f":
        x = np.minimum(x, 2.0e9)
    return x.astype(dtype)


@pytest.mark.parametrize("dtype", [np.float32, np.int32, np.float64, np.uint64])
@pytest.mark.parametrize("kind", ["equal", "two values", "hundred values", "ascending", "descending", "runs", "magnitudes",
                                  "cluster", "far"])
@pytest.mark.parametrize("n", [9001, 100_003, 200_001, 700_001, 2_500_001])
def test_kinds_of_keys(lib, torch_cuda, dtype, kind, n):
    if n > 1 << 20 and np.dtype(dtype).itemsize == 4:
        pytest.skip("4-byte keys are split up to 2^20")
    _check(lib, torch_cuda, _kind(kind, dtype, n), f"{np.dtype(dtype)} {n} {kind}")


def _sample_places(n, samples):
    """split_sample_place of csrc/split_sort.h."""
    i = np.arange(samples, dtype=np.uint64)
    lo, hi = i * n // samples, (i + 1) * n // samples
    h = i.astype(np.uint32)
    for shift, factor in ((16, 0x7FEB352D), (15, 0x846CA68B)):
        h = (h ^ (h >> np.uint32(shift))) * np.uint32(factor)
    h ^= h >> np.uint32(16)
    return (lo + (h.astype(np.uint64) * (hi - lo) >> np.uint64(32))).astype(np.int64)


@pytest.mark.parametrize("dtype", [np.float32, np.int32, np.float64, np.uint64])
@pytest.mark.parametrize("n,samples", [(20_000, 1024), (150_001, 2048), (300_007, 4096), (1_100_001, 16384)])
@pytest.mark.parametrize("share", ["all", "some"])
def test_buckets_beyond_lds(lib, torch_cuda, dtype, n, samples, share):
    """A row made so that its sample says nothing: the sampled keys are the largest.  All others share a bucket, or, where
    an eighth of the sample is left as it is, buckets of several times the room."""
    if n > 1 << 20 and np.dtype(dtype).itemsize == 4:
        pytest.skip("4-byte keys are split up to 2^20")
    rng = np.random.default_rng(n)
    x = rng.integers(0, 1 << 30, n).astype(dtype)
    places = _sample_places(n, samples)
    assert places.size == np.unique(places).size and places.max() < n
    if share == "some":
        places = places[rng.random(samples) < 0.98]
    x[places] = (1 << 30) + rng.integers(0, 1 << 20, places.size).astype(dtype)
    if np.dtype(dtype).kind == "f":
        x[rng.integers(0, n, 100)] = np.nan
        x[rng.integers(0, n, 100)] = -0.0
        x[rng.integers(0, n, 100)] = 0.0
    _check(lib, torch_cuda, x, f"{np.dtype(dtype)} {n} {share}")


def test_the_public_calls_take_it(lib, torch_cuda):
    """Rows in its range, through sort, argsort and an in-place sort: two or three launches and no status to look at; rows
    outside it, and several rows, go where they went."""
    from cupynumeric_amd.runtime import runtime

    def labels(call):
        lib.cpn_profile_enable(1)
        try:
            call()
        finally:
            lib.cpn_profile_enable(0)
        return [k for k, _ in _lib.profile_collect()]

    rng = np.random.default_rng(0)
    for n, launches in ((100_000, ["split_tiles", "split_buckets"]), (600_000, ["split_gather", "split_tiles", "split_buckets"])):
        x = rng.standard_normal(n)
        a = num.array(x)
        runtime.flush_status()
        got = []
        assert labels(lambda: got.append(num.argsort(a))) == launches
        assert np.array_equal(np.asarray(got[0]), np.argsort(x, kind="stable"))
        assert labels(lambda: got.append(num.sort(a))) == launches and runtime._status_used == 0
        assert np.array_equal(np.asarray(got[1]), np.sort(x))
        assert labels(lambda: a.sort()) == launches
        assert np.array_equal(np.asarray(a), np.sort(x))
    x = rng.integers(0, 1 << 40, (1 << 20) + 1)
    got = []
    assert labels(lambda: got.append(num.argsort(num.array(x))))[-3:] == ["split_table", "split_tiles", "split_buckets"]
    assert runtime._status_used == 0 and np.array_equal(np.asarray(got[0]), np.argsort(x, kind="stable"))
    for x in (rng.standard_normal(4000), rng.standard_normal((2, 30_000)), rng.standard_normal((1 << 20) + 1).astype(np.float32),
              rng.standard_normal(4096 * 2560 + 1)):
        assert "split_tiles" not in labels(lambda: num.sort(num.array(x)))


@pytest.mark.parametrize("n", [150_000, 1_300_000])
def test_captured_and_replayed(lib, torch_cuda, n):
    """The launches in a graph, replayed on other keys with eager work between the replays."""
    torch = torch_cuda
    code = _lib.DTYPE_CODES[np.dtype(np.float64)]
    tb = lib.cpn_local_sort_split_temp_bytes(code, n, n, 1)
    x = torch.empty(n, dtype=torch.float64, device="cuda")
    v, i = torch.empty_like(x), torch.empty(n, dtype=torch.int64, device="cuda")
    temp = torch.empty(tb, dtype=torch.uint8, device="cuda")

    def call():
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert lib.cpn_local_sort_ex(code, x.data_ptr(), v.data_ptr(), i.data_ptr(), n, n, 0, 1, _lib.CPN_SORT_SPLIT,
                                     temp.data_ptr(), tb, stream) == 0

    x.normal_()
    call()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call()
    for seed in range(4):
        g = torch.Generator(device="cuda").manual_seed(seed)
        x.normal_(generator=g)
        if seed == 2:
            x.round_()
        v.zero_()
        i.zero_()
        graph.replay()
        torch.cuda.synchronize()
        host = x.cpu().numpy()
        want = oracle.local_sort(host.reshape(1, -1), argsort=True, threads=8)[0]
        assert np.array_equal(i.cpu().numpy(), want)
        assert_same_bits(v.cpu().numpy(), host[want], f"replay {seed}")


def test_a_smaller_workspace_sorts_the_other_way(lib, torch_cuda):
    """The option with the workspace of cpn_local_sort_temp_bytes."""
    torch = torch_cuda
    n = 400_000
    code = _lib.DTYPE_CODES[np.dtype(np.int32)]
    tb = lib.cpn_local_sort_temp_bytes(code, n, n, 0, 1, 0)
    assert tb < lib.cpn_local_sort_split_temp_bytes(code, n, n, 1)
    x = torch.randint(-(1 << 31), (1 << 31) - 1, (n,), dtype=torch.int32, device="cuda")
    i = torch.empty(n, dtype=torch.int64, device="cuda")
    temp = torch.empty(tb, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.cpn_local_sort_ex(code, x.data_ptr(), None, i.data_ptr(), n, n, 0, 1, _lib.CPN_SORT_SPLIT, temp.data_ptr(), tb,
                                 stream) == 0
    assert lib.cpn_local_sort_check(temp.data_ptr(), stream) == 0
    assert np.array_equal(i.cpu().numpy(), np.argsort(x.cpu().numpy(), kind="stable"))


@pytest.mark.parametrize("dtype", [np.uint32, np.float32, np.int64, np.float64])
@pytest.mark.parametrize("n", [9001, 100_000, 1 << 20, 2_100_000])
@pytest.mark.parametrize("low_bits", ["differ", "shared"])
def test_few_values_that_only_lower_bits_tell_apart(lib, torch_cuda, dtype, n, low_bits):
    """A bucket of a few values, each too often for a bin: its leading 16 varying bits are not enough, then 40 are not; or
    the low bits are the same in all keys and take no pass."""
    key = np.dtype(dtype).itemsize
    if lib.cpn_local_sort_split_temp_bytes(_lib.DTYPE_CODES[np.dtype(dtype)], n, n, 1) == 0:
        pytest.skip("not a row that is split")
    rng = np.random.default_rng(n)
    clusters = max(1, n // 200)
    apart = np.array([0, 1, 1 << 12, 1 << 25] if key == 8 else [0, 1, 2, 5], np.uint64)
    if low_bits == "shared":
        apart = apart << np.uint64(20 if key == 8 else 3)
    top, least = (62, 46) if key == 8 else (30, 6)
    step = max((1 << top) // clusters >> least << least, 1 << least)
    keys = (rng.integers(0, clusters, n).astype(np.uint64) * np.uint64(step)) + apart[rng.integers(0, 4, n)]
    x = keys.astype(np.uint64 if key == 8 else np.uint32).view(dtype)
    _check(lib, torch_cuda, x, f"{np.dtype(dtype)} {n} {low_bits}")


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_whole_numbers_held_as_floats(lib, torch_cuda, dtype):
    for n, values in ((100_000, 500), (300_000, 3000), (1 << 20, 20_000)):
        x = np.random.default_rng(values).integers(-values, values, n).astype(dtype)
        _check(lib, torch_cuda, x, f"{np.dtype(dtype)} {n} {values}")


def test_streams_and_threads_at_once(torch_cuda):
    """Rows of every kind of plan, sorted by eight threads on streams of their own, whose workspaces come from one allocator."""
    torch = torch_cuda
    rng = np.random.default_rng(12)
    rows = [rng.standard_normal(9000).astype(np.float32), rng.standard_normal(100_000), rng.integers(0, 1 << 30, 600_000).astype(np.int32),
            rng.integers(0, 1 << 40, 1_100_000), rng.standard_normal(2_300_000), rng.integers(0, 300, 2_300_000),
            np.full(2_200_000, 5), rng.integers(0, 1 << 62, 5_000_000)]
    want = [(np.sort(x), np.argsort(x, kind="stable")) for x in rows]
    arrays = [num.array(x) for x in rows]
    for a in arrays:
        num.sort(a)  # (uploads it)
    torch.cuda.synchronize()
    wrong = []

    def work(i):
        stream = torch.cuda.Stream()
        with torch.cuda.stream(stream):
            for turn in range(6):
                k = (i + turn) % len(rows)
                got = [num.sort(arrays[k]), num.argsort(arrays[k])]  # both in flight before either is read
                for g, w in zip(got, want[k]):
                    if not np.array_equal(np.asarray(g), w):
                        wrong.append((i, k))

    threads = [threading.Thread(target=work, args=(i,)) for i in range(len(rows))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong, wrong
