"""Single rows of 8-byte keys of which few bytes vary: sorted by the passes over those bytes, ahead of the split by sampled keys
(csrc/split_plan.h, csrc/sort_driver.h: sort_narrow).  Against the oracle, and which of the two ways the row went."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
from conftest import assert_same_bits
from test_sort_gpu import lib, torch_cuda  # noqa: F401 (fixtures)

from cupynumeric_amd import _lib
from oracle import sort_oracle as oracle

pytestmark = pytest.mark.gpu

LONGEST = 4096 * 2560
SHORT = 1 << 21  # rows up to here try two passes, of floats none; longer ones three, of floats two


class _Row:
    def __init__(self, lib, torch, x, values, indices, in_place=False):
        self.lib, self.torch, self.n, self.dtype, self.in_place = lib, torch, x.size, x.dtype, in_place
        self.code = _lib.DTYPE_CODES[x.dtype]
        self.need = lib.cpn_local_sort_split_temp_bytes(self.code, x.size, x.size, int(indices))
        assert self.need != 0
        self.d_in = torch.from_numpy(x.view(np.int64).copy()).cuda()
        self.d_val = self.d_in if in_place else (torch.zeros_like(self.d_in) if values else None)
        self.d_idx = torch.full((x.size,), -7, dtype=torch.int64, device="cuda") if indices else None
        self.temp = torch.full((self.need,), 0xFF, dtype=torch.uint8, device="cuda")

    def issue(self):
        stream = ctypes.c_void_p(self.torch.cuda.current_stream().cuda_stream)
        rc = self.lib.cpn_local_sort_ex(self.code, self.d_in.data_ptr(), self.d_val.data_ptr() if self.d_val is not None else None,
                                        self.d_idx.data_ptr() if self.d_idx is not None else None, self.n, self.n, 5, 1,
                                        _lib.CPN_SORT_SPLIT, self.temp.data_ptr(), self.need, stream)
        assert rc == 0, _lib.status_string(rc)

    def check(self, x, what):
        """True: sorted by passes."""
        self.torch.cuda.synchronize()
        status, _, narrow = self.temp[:12].view(self.torch.int32).tolist()
        assert status == 0 and narrow in (0, 1, 2), what  # (2: equal keys)
        order = oracle.local_sort(x.reshape(1, -1), argsort=True, threads=8)[0]
        if self.d_val is not None:
            assert_same_bits(self.d_val.cpu().numpy().view(x.dtype), x[order], f"{what}: values")
        if self.d_idx is not None:
            assert np.array_equal(self.d_idx.cpu().numpy(), order + 5), f"{what}: positions"
        return narrow != 0


def _both(lib, torch, x, what):
    ways = set()
    for values, indices, in_place in ((True, False, False), (False, True, False), (True, False, True), (True, True, True), (True, True, False)):
        row = _Row(lib, torch, x, values, indices, in_place)
        row.issue()
        ways.add(row.check(x, f"{what} {values} {indices} {in_place}"))
    assert len(ways) == 1
    return ways.pop()


# kind -> least number of varying bytes of int64 keys, None: more than the passes take
KINDS = {"equal": 0, "zeros": 0, "labels": 1, "two bytes": 2, "second byte": 2, "three bytes": 3, "five": None, "negative": None}


def _whole(kind, n):
    rng = np.random.default_rng(n)
    return {
        "equal": lambda: np.full(n, -123456789012345), "zeros": lambda: np.zeros(n), "labels": lambda: rng.integers(0, 200, n),
        "two bytes": lambda: rng.integers(0, 20_000, n), "second byte": lambda: (1 << 50) + 256 * rng.integers(0, 100, n),
        "three bytes": lambda: rng.integers(0, 300_000, n), "five": lambda: rng.integers(0, 1 << 34, n),
        "negative": lambda: rng.integers(-3, 3, n),
    }[kind]()


@pytest.mark.parametrize("dtype", [np.int64, np.uint64])
@pytest.mark.parametrize("n", [(1 << 20) + 1, SHORT, SHORT + 1, 3_000_017])
@pytest.mark.parametrize("kind", list(KINDS))
def test_whole_numbers(lib, torch_cuda, dtype, n, kind):
    vary = KINDS[kind]
    x = _whole(kind, n).astype(np.int64).view(dtype)
    assert _both(lib, torch_cuda, x, f"{np.dtype(dtype)} {n} {kind}") == (vary is not None and vary <= (2 if n <= SHORT else 3))


@pytest.mark.parametrize("n", [SHORT, SHORT + 1, 3_000_017])
@pytest.mark.parametrize("kind", ["equal", "NaN", "zeros of either sign", "flags", "eighths", "NaN among flags", "thousands"])
def test_floats(lib, torch_cuda, n, kind):
    rng = np.random.default_rng(n)
    x = {
        "equal": lambda: np.full(n, -3.7), "NaN": lambda: np.full(n, np.nan),
        "zeros of either sign": lambda: np.where(rng.random(n) < 0.5, 0.0, -0.0),
        "flags": lambda: rng.integers(0, 2, n).astype(np.float64), "eighths": lambda: rng.integers(8, 16, n) / 8.0,
        "NaN among flags": lambda: np.where(rng.random(n) < 0.1, np.nan, rng.integers(0, 2, n).astype(np.float64)),
        "thousands": lambda: rng.integers(0, 5000, n).astype(np.float64),
    }[kind]()
    # (the image of a NaN has all bits set)
    assert _both(lib, torch_cuda, x, f"{n} {kind}") == (n > SHORT and kind not in ("NaN among flags", "thousands"))


def test_the_longest_row(lib, torch_cuda):
    assert _both(lib, torch_cuda, _whole("three bytes", LONGEST), "longest")


@pytest.mark.parametrize("where", [1, 2_000_001, 2_999_999])
def test_a_key_that_the_sample_misses(lib, torch_cuda, where):
    """The count says so, and the row is split after all."""
    x = _whole("labels", 3_000_000)
    x[where] = 1 << 40
    assert not _both(lib, torch_cuda, x, f"{where}")


def test_passes_that_give_up(lib, torch_cuda):
    """With one poll per wait some tile gives up (if none does the row is sorted by passes): the split sorts, also in place."""
    prev = lib.cpn_set_lookback_spin_limit(1)
    by_passes = []
    try:
        for n in (1_500_000, 2_500_000, LONGEST):
            x = _whole("two bytes", n)
            for values, indices, in_place in ((True, False, False), (False, True, False), (True, True, True)):
                row = _Row(lib, torch_cuda, x, values, indices, in_place)
                row.issue()
                by_passes.append(row.check(x, f"{n} {values} {indices} {in_place}"))
    finally:
        lib.cpn_set_lookback_spin_limit(prev)
    if all(by_passes):
        pytest.skip("every poll was answered at once")


def test_captured(lib, torch_cuda):
    """One graph, replayed on keys that go either way, with eager work between."""
    torch, n = torch_cuda, 2_200_000
    first = _whole("labels", n)
    row = _Row(lib, torch, first, True, True)
    row.issue()
    assert row.check(first, "eager")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        row.issue()
    for kind in ("two bytes", "five", "equal", "five", "labels"):
        x = _whole(kind, n).astype(np.int64)
        row.d_in.copy_(torch.from_numpy(x))
        row.d_val.zero_()
        row.d_idx.fill_(-7)
        graph.replay()
        assert row.check(x, kind) == (kind != "five")
