"""Host side of the split by sampled keys (csrc/split_plan.h): which requests have a workspace for it, and how large."""
from __future__ import annotations

import pytest

from cupynumeric_amd import _lib

F16, F32, F64, I64, C64 = 9, 10, 11, 4, 12


@pytest.fixture(scope="module")
def lib():
    return _lib.load()


def test_requests_in_range(lib):
    size = lib.cpn_local_sort_split_temp_bytes
    for code, kb in ((F32, 4), (F64, 8), (I64, 8)):
        for idx in (0, 1):
            first = 6145 if kb == 8 else 8193
            assert size(code, first - 1, first - 1, idx) == 0 and size(code, first, first, idx) != 0
            for n in (8193, 100_000, 1 << 18, (1 << 18) + 1, 1 << 20):
                need = size(code, n, n, idx)
                # the keys, two words and a place per key, and a table of at most a word per key and bucket's tile
                assert n * (kb + 8 + 2 * idx) <= need <= n * (kb + 8 + 2 * idx) + (1 << 20), (code, n, idx)
                assert need % 256 == 0
            last = 4096 * 2560 if kb == 8 else 1 << 20
            assert size(code, last, last, idx) != 0 and size(code, last + 1, last + 1, idx) == 0
            if kb == 8:  # and the sample's own sort
                for n in ((1 << 20) + 1, last):
                    assert n * (kb + 8 + 2 * idx) < size(code, n, n, idx) < n * (kb + 8 + 2 * idx) + 40 * (1 << 20), (code, n, idx)
    for code in (F16, C64):
        assert size(code, 100_000, 100_000, 0) == 0
    assert size(F32, 200_000, 100_000, 0) == 0 and size(F32, 0, 0, 0) == 0 and size(99, 100_000, 100_000, 0) == 0
    assert size(F32, 100_000, 99_999, 0) == 0


def test_switches(lib):
    size = lib.cpn_local_sort_split_temp_bytes
    for setter, value in ((lib.cpn_set_merge_rows, 0), (lib.cpn_set_merge_rows, 8), (lib.cpn_set_lds_row_limit, 0)):
        prev = setter(value)
        try:
            assert size(F64, 100_000, 100_000, 1) == 0
        finally:
            setter(prev)
        assert size(F64, 100_000, 100_000, 1) != 0


def test_the_option_keeps_the_checks(lib):
    """A missing, small or misaligned workspace is refused as without the option."""
    n = 100_000
    need = lib.cpn_local_sort_split_temp_bytes(F32, n, n, 0)
    least = 2048
    for temp, tb in ((None, need), (264, need), (256, least)):
        assert lib.cpn_local_sort_ex(F32, 4096, 8192, None, n, n, 0, 1, _lib.CPN_SORT_SPLIT, temp, tb, None) == _lib.CPN_ERR_TEMP
    assert lib.cpn_local_sort_ex(F32, 4098, 8192, None, n, n, 0, 1, _lib.CPN_SORT_SPLIT, 256, need, None) == _lib.CPN_ERR_ALIGN
    assert lib.cpn_local_sort_ex(F32, None, 8192, None, n, n, 0, 1, _lib.CPN_SORT_SPLIT, 256, need, None) == _lib.CPN_ERR_NULL
    assert lib.cpn_local_sort_ex(F32, 4096, 8192, None, n, n, 0, 1, 0x80 | _lib.CPN_SORT_SPLIT, 256, need, None) == _lib.CPN_ERR_UNSUPPORTED
