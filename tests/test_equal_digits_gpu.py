"""Sorts of 8-byte keys by equalised digits (csrc/equal_digits.h) against the oracle, bit for bit.

The threshold is lowered so that rows of a few hundred thousand keys take the path.  The inputs are those where it
can go wrong: digits from a sample that misses the ends of the range, buckets of one value (kept), of many keys
(larger tile), of a value and a few neighbours of it (the byte passes take over, before or after the passes on
equalised digits), NaNs and zeros of both signs, and lengths at the ends of tiles and stretches.
"""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
from conftest import assert_same_bits
from test_sort_gpu import abi_sort, lib, torch_cuda  # noqa: F401 (fixtures)

from oracle import sort_oracle as oracle

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def lowered_threshold(lib):
    """(Rows of this length are merged from sorted pieces by default.)"""
    prev, merged = lib.cpn_set_equal_digit_threshold(1 << 18), lib.cpn_set_merge_rows(0)
    yield
    lib.cpn_set_equal_digit_threshold(prev)
    lib.cpn_set_merge_rows(merged)


def _keys(kind, dtype, n, rng):
    dt = np.dtype(dtype)
    if dt.kind == "f":
        x = rng.standard_normal(n)
        u = rng.random(n)
        if kind == "spread":
            return rng.random(n)
        if kind == "bits":  # every magnitude, NaNs of many payloads
            return rng.integers(0, 1 << 63, n, dtype=np.int64).view(np.float64) * np.where(u < 0.5, -1.0, 1.0)
        if kind == "specials":
            x[u < 0.02] = np.nan
            x[(u >= 0.02) & (u < 0.03)] = 0.0
            x[(u >= 0.03) & (u < 0.04)] = -0.0
            x[(u >= 0.04) & (u < 0.05)] = np.inf
            x[(u >= 0.05) & (u < 0.06)] = -np.inf
        elif kind == "crowd":  # a quarter is one value, and two neighbours of it are too few for the sample
            x[u < 0.25] = 50.0
            x[n // 3], x[n // 2] = np.nextafter(50.0, 51.0), np.nextafter(50.0, 49.0)
        elif kind == "repeated":
            x = rng.standard_normal(n // 40)[rng.integers(0, n // 40, n)]
        return x
    info = np.iinfo(dtype)
    x = rng.integers(info.min, info.max, n, dtype=dtype, endpoint=True)
    if kind == "specials":  # the smallest and largest key, often
        x[rng.random(n) < 0.02] = info.min
        x[rng.random(n) < 0.02] = info.max
    elif kind == "crowd":
        mid = dt.type(info.max // 3)
        x[rng.random(n) < 0.25] = mid
        x[n // 3], x[n // 2] = mid + dt.type(1), mid - dt.type(1)
    elif kind == "repeated":
        x = x[: n // 40][rng.integers(0, n // 40, n)]
    elif kind == "bits":  # few bytes vary: the byte passes keep it
        x = (x.view(np.uint64) >> np.uint64(33)).astype(dtype)
    return x


@pytest.mark.parametrize("dtype", [np.float64, np.int64, np.uint64])
@pytest.mark.parametrize("kind", ["spread", "bits", "normal", "specials", "crowd", "repeated"])
def test_kinds_of_keys(lib, torch_cuda, dtype, kind):
    if kind == "normal" and np.dtype(dtype).kind != "f":
        pytest.skip("float keys only")
    rng = np.random.default_rng(len(kind) + np.dtype(dtype).num)
    n = 700_001
    x = _keys(kind, dtype, n, rng).astype(dtype, copy=False)
    want_v = oracle.local_sort(x, argsort=False, threads=8)
    want_i = oracle.local_sort(x, argsort=True, threads=8)
    v, _ = abi_sort(lib, torch_cuda, x, want_values=True, want_indices=False)
    assert_same_bits(v, want_v, "values")
    _, i = abi_sort(lib, torch_cuda, x, want_values=False, want_indices=True, offset=7)
    assert_same_bits(i, want_i + 7, "positions")
    v, i = abi_sort(lib, torch_cuda, x, want_values=True, want_indices=True)
    assert_same_bits(v, want_v, "both: values")
    assert_same_bits(i, want_i, "both: positions")
    v, i = abi_sort(lib, torch_cuda, x, want_values=True, want_indices=True, in_place=True)
    assert_same_bits(v, want_v, "in place")
    assert_same_bits(i, want_i, "in place: positions")
    v, _ = abi_sort(lib, torch_cuda, x, want_values=True, in_place=True)
    assert_same_bits(v, want_v, "in place, values only")


@pytest.mark.parametrize("n", [(1 << 18), (1 << 18) + 1, 16384 * 17 - 1, 16384 * 17, 2304 * 120, 2304 * 120 + 1, 3072 * 100 - 1])
def test_lengths(lib, torch_cuda, n):
    """The shortest row that is sampled, ends of the scatter tiles (16384) and of the LDS sort's stretches (2304)."""
    rng = np.random.default_rng(n)
    x = rng.standard_normal(n)
    _, i = abi_sort(lib, torch_cuda, x, want_values=False, want_indices=True)
    assert_same_bits(i, oracle.local_sort(x, argsort=True, threads=8), "positions")
    v, _ = abi_sort(lib, torch_cuda, x, want_values=True)
    assert_same_bits(v, oracle.local_sort(x, argsort=False, threads=8), "values")


def test_the_smaller_workspace_is_still_taken(lib, torch_cuda):
    """A caller that asked for the workspace while the path was out of use gets the byte passes."""
    torch = torch_cuda
    n = 300_000
    x = np.random.default_rng(0).standard_normal(n)
    lib.cpn_set_equal_digit_threshold(1 << 40)
    small = lib.cpn_local_sort_temp_bytes(11, n, n, 1, 0, 0)
    lib.cpn_set_equal_digit_threshold(1 << 18)
    assert small < lib.cpn_local_sort_temp_bytes(11, n, n, 1, 0, 0)
    a = torch.from_numpy(x).cuda()
    out = torch.empty_like(a)
    ws = torch.empty(small, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.cpn_local_sort(11, a.data_ptr(), out.data_ptr(), None, n, n, 0, 1, ws.data_ptr(), small, stream) == 0
    assert lib.cpn_local_sort_check(ws.data_ptr(), stream) == 0
    assert_same_bits(out.cpu().numpy(), np.sort(x), "values")


def _sort(lib, torch, x, want_values, want_indices, in_place=False, offset=0):
    """cpn_local_sort on device buffers; returns values, positions and what became of the plan (mode, failed, ...)."""
    code, n = 11 if x.dtype == np.float64 else (4 if x.dtype == np.int64 else 8), x.size
    a = torch.from_numpy(x.view(np.int64).copy()).cuda()
    v = a if in_place else (torch.empty_like(a) if want_values else None)
    i = torch.empty(n, dtype=torch.int64, device="cuda") if want_indices else None
    shape = (n, n, int(want_values), int(want_indices), int(in_place))
    need = lib.cpn_local_sort_temp_bytes(code, *shape)
    ws = torch.full((need,), 0xFF, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.cpn_local_sort(code, a.data_ptr(), v.data_ptr() if want_values else None, i.data_ptr() if want_indices else None,
                              n, n, offset, 1, ws.data_ptr(), need, stream) == 0
    status = lib.cpn_local_sort_check(ws.data_ptr(), stream)
    plan = (ctypes.c_uint32 * 5)()
    assert lib.cpn_equal_digit_plan(code, *shape, ws.data_ptr(), need, plan, stream) == 0
    return status, (v.cpu().numpy().view(x.dtype) if want_values else None), (i.cpu().numpy() if want_indices else None), tuple(plan)


REQUESTS = [(True, False, False), (False, True, False), (True, True, False), (True, False, True), (True, True, True)]


def _check(lib, torch, x, mode, failed, what):
    want_v, want_i = oracle.local_sort(x, argsort=False, threads=8), oracle.local_sort(x, argsort=True, threads=8)
    for want_values, want_indices, in_place in REQUESTS:
        status, v, i, plan = _sort(lib, torch, x, want_values, want_indices, in_place)
        assert status == 0 and plan[:2] == (mode, failed), (what, want_values, want_indices, in_place, plan)
        if want_values:
            assert_same_bits(v, want_v, f"{what}: values")
        if want_indices:
            assert_same_bits(i, want_i, f"{what}: positions")


# (uint64 "bits": few bytes vary; the others that keep the byte passes: a value that occurs often has keys in its cell that
# do not, any integer in those of the smallest and the largest; float rows that span zero have cells of two octaves)
@pytest.mark.parametrize("dtype,kind,mode,failed", [
    (np.float64, "spread", 1, 0), (np.float64, "normal", 0, 0), (np.float64, "repeated", 0, 0), (np.float64, "specials", 0, 0),
    (np.int64, "spread", 1, 0), (np.uint64, "specials", 0, 0), (np.int64, "crowd", 0, 0), (np.uint64, "bits", 0, 0)])
def test_the_path_that_is_taken(lib, torch_cuda, dtype, kind, mode, failed):
    x = _keys(kind, dtype, 700_001, np.random.default_rng(7)).astype(dtype, copy=False)
    _check(lib, torch_cuda, x, mode, failed, kind)


def _far_value(x, value, rng):
    """A quarter of the keys is a value far from the others, with two neighbours that the sample misses."""
    n = x.size
    x[rng.random(n) < 0.25] = value
    x[n // 3], x[n // 2] = value + 1, value - 1
    return x


@pytest.mark.parametrize("dtype", [np.int64, np.uint64, np.float64])
@pytest.mark.parametrize("top", [40, 48, 56])
def test_late_failure_with_constant_bytes(lib, torch_cuda, dtype, top):
    """Six, seven and eight bytes vary: an odd number of byte passes takes a copying one more when they go on."""
    rng = np.random.default_rng(top)
    x = _far_value(rng.integers(0, 1 << (top - 4), 400_003), 15 << (top - 4), rng).astype(np.int64).view(dtype)
    _check(lib, torch_cuda, x, 1, 1, f"{np.dtype(dtype)} {top}")


@pytest.fixture
def both_thresholds_lowered(lib):
    prev = lib.cpn_set_virtual_digit_threshold(1 << 18)
    yield
    lib.cpn_set_virtual_digit_threshold(prev)


@pytest.mark.parametrize("dtype", [np.int64, np.float64])
def test_few_values_keep_the_pass_on_their_ranks(lib, torch_cuda, both_thresholds_lowered, dtype):
    rng = np.random.default_rng(1)
    values = rng.standard_normal(200).view(np.int64).astype(np.int64).view(dtype)
    _check(lib, torch_cuda, values[rng.integers(0, 200, 300_001)], 0, 0, "few values")


@pytest.mark.parametrize("dtype,bytes_that_vary", [(np.int64, 6), (np.int64, 8), (np.float64, 6), (np.uint64, 8)])
def test_late_failure_goes_on_with_grouped_digits(lib, torch_cuda, both_thresholds_lowered, dtype, bytes_that_vary):
    """Few values in every byte: three groups of two bytes (an odd number of passes) and four."""
    rng = np.random.default_rng(bytes_that_vary)
    n, x = 500_009, np.zeros(500_009, np.int64)
    for b in range(bytes_that_vary):
        x |= (rng.integers(0, 8, n) * 9) << (8 * b)
    x = _far_value(x, 0x7B << (8 * (bytes_that_vary - 1)), rng)
    _check(lib, torch_cuda, x.view(dtype), 1, 1, f"{bytes_that_vary} bytes")


def test_evenly_spread_keys_with_both_kinds_of_digits_in_force(lib, torch_cuda, both_thresholds_lowered):
    _check(lib, torch_cuda, np.random.default_rng(3).random(600_011), 1, 0, "evenly spread")


@pytest.mark.parametrize("dtype", [np.int64, np.float64])
def test_passes_that_give_up(lib, torch_cuda, dtype):
    """Every wait for an earlier tile ends at the first unanswered poll: an error is reported, or the result is right."""
    x = _keys("spread", dtype, 700_001, np.random.default_rng(5)).astype(dtype, copy=False)
    want = oracle.local_sort(x, argsort=False, threads=8)
    prev = lib.cpn_set_lookback_spin_limit(1)
    try:
        for _ in range(5):
            status, v, _, plan = _sort(lib, torch_cuda, x, True, False)
            assert status in (0, -7) and plan[:2] == (1, 0)
            if status == 0:
                assert_same_bits(v, want, "values")
    finally:
        lib.cpn_set_lookback_spin_limit(prev)
    assert _sort(lib, torch_cuda, x, True, False)[0] == 0


def _long_row(torch, kind, log2):
    n, gen = 1 << log2, torch.Generator(device="cuda").manual_seed(log2)
    if kind == "uniform":
        return torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
    x = torch.randn(n, generator=gen, device="cuda", dtype=torch.float64)
    if kind == "logistic":
        u = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64)
        return torch.log(u / (1 - u))
    if kind == "wide":
        return 3 * x
    if kind == "repeated":  # every value two hundred times
        x = x.abs()
        return x[: n // 200][torch.randint(0, n // 200, (n,), generator=gen, device="cuda")]
    if kind.endswith("groups"):  # neighbouring numbers in far groups of n / count keys
        count = int(kind.split()[0])
        return (torch.randint(0, count, (n,), generator=gen, device="cuda") << 32) + torch.randint(0, 1 << 16, (n,), generator=gen, device="cuda")
    return x


# (The shortest rows that are tried by default.)
@pytest.mark.parametrize("kind,log2,mode", [("uniform", 25, 1), ("normal", 25, 0), ("uniform", 26, 1), ("normal", 26, 0), ("repeated", 25, 0),
                                            ("repeated", 26, 0), ("5000 groups", 26, 0), ("20000 groups", 26, 0), ("logistic", 26, 0), ("wide", 26, 0)])
def test_long_rows_that_do_not_fit_keep_the_byte_passes(lib, torch_cuda, kind, log2, mode):
    """The plan declines them; none is sorted twice (2^26 normal keys: 2.5 ms, and 4.1 when that was seen too late)."""
    torch = torch_cuda
    lib.cpn_set_equal_digit_threshold(-1)
    a = _long_row(torch, kind, log2)
    n, code = a.numel(), 11 if a.dtype == torch.float64 else 4
    v = torch.empty_like(a)
    need = lib.cpn_local_sort_temp_bytes(code, n, n, 1, 0, 0)
    ws = torch.empty(need, dtype=torch.uint8, device="cuda")
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    assert lib.cpn_local_sort(code, a.data_ptr(), v.data_ptr(), None, n, n, 0, 1, ws.data_ptr(), need, stream) == 0
    assert lib.cpn_local_sort_check(ws.data_ptr(), stream) == 0
    plan = (ctypes.c_uint32 * 5)()
    assert lib.cpn_equal_digit_plan(code, n, n, 1, 0, 0, ws.data_ptr(), need, plan, stream) == 0
    assert tuple(plan[:2]) == (mode, 0), tuple(plan)
    assert torch.equal(v, torch.sort(a).values)


def _repeated(n, repeats, share, rng):
    """A share of the keys are values that occur `repeats` times each, the others are all different."""
    x = rng.random(n)
    count = int(n * share)
    if count:
        x[:count] = np.repeat(rng.random(count // repeats + 1), repeats)[:count]
        rng.shuffle(x)
    return x


# bins for a thread (up to 8 keys), for a wave (64), for the workgroup (512), and of more
@pytest.mark.parametrize("repeats,share", [(8, 1.0), (9, 1.0), (24, 1.0), (40, 0.5), (64, 0.5), (65, 0.5), (200, 0.3), (511, 0.3), (512, 0.3), (513, 0.3), (700, 0.2)])
def test_repeated_values(lib, torch_cuda, repeats, share):
    x = _repeated(700_001, repeats, share, np.random.default_rng(repeats))
    _check(lib, torch_cuda, x, 1, 0, f"{repeats} times each")
    if repeats <= 40:  # (bins of more than a wave are left to the general sort when there are several)
        plan = _sort(lib, torch_cuda, x, True, True)[3]
        assert plan[4] == 0, plan  # no piece went to the general sort


def test_crowded_bins_of_different_keys(lib, torch_cuda):
    """Clusters of neighbouring numbers narrower than a bin: 25 to 500 keys each, in no order."""
    rng = np.random.default_rng(11)
    x = rng.integers(0, 1 << 62, 600_007)
    at = 0
    for size in (25, 64, 100, 300, 500):
        for centre in rng.integers(0, 1 << 62, 60):
            x[at : at + size] = centre + rng.integers(0, 200, size)
            at += size
    rng.shuffle(x)
    _check(lib, torch_cuda, x, 1, 0, "clusters")
    _check(lib, torch_cuda, (x - (1 << 61)).view(np.uint64), 1, 0, "clusters, unsigned")


def test_rows_of_narrow_clusters_keep_the_byte_passes(lib, torch_cuda):
    """300 000 groups of a hundred neighbouring numbers each, all of a group in one bin of the LDS sort: 4 to 8 times the
    byte passes' time when every piece had its bins put in order one by one."""
    test_long_rows_that_do_not_fit_keep_the_byte_passes(lib, torch_cuda, "300000 groups", 25, 0)


@pytest.mark.parametrize("n", [(1 << 18), (1 << 18) + 1, 16384 * 17 - 1, 16384 * 17, 2304 * 120, 2304 * 120 + 1, 3072 * 100 - 1])
def test_lengths_of_evenly_spread_rows(lib, torch_cuda, n):
    """As test_lengths, with keys that take the path."""
    rng = np.random.default_rng(n)
    _check(lib, torch_cuda, rng.random(n), 1, 0, f"{n}")
    _check(lib, torch_cuda, rng.integers(-(1 << 63), (1 << 63) - 1, n), 1, 0, f"{n} int64")


def test_special_values_among_huge_keys(lib, torch_cuda):
    """Keys so large that the cells reach the infinity and the NaNs above them: pieces that hold a NaN go the general way."""
    rng = np.random.default_rng(2)
    x = 10.0 ** rng.uniform(280, 308, 500_003)
    x[rng.random(x.size) < 0.0005] = np.nan
    x[rng.random(x.size) < 0.0005] = np.inf
    x.view(np.uint64)[::50_021] = 0x7FF8_0000_0000_1234  # a payload
    _check(lib, torch_cuda, x, 1, 0, "huge keys")
    assert _sort(lib, torch_cuda, x, True, True)[3][4] > 0
