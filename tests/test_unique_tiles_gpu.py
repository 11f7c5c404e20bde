"""Sizes at the edges of the tiles of unique's compaction."""
import numpy as np
import pytest

import cupynumeric_amd as num

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.int8, np.float16, np.uint32, np.float64, np.complex128])
@pytest.mark.parametrize("n", [1, 2, 63, 65, 4095, 4096, 4097, 8193, 69_633])
@pytest.mark.parametrize("distinct", ["one", "few", "all"])
def test_unique_tile_edges(dtype, n, distinct):
    """Tiles of 4096 elements without a head, with a few and with heads only."""
    rng = np.random.default_rng(n)
    count = {"one": 1, "few": min(n, 7), "all": n}[distinct]
    x = rng.permutation(np.arange(n) % count).astype(np.int64)
    x = x % 128 if dtype == np.int8 else x % 2048 if dtype == np.float16 else x
    got = np.asarray(num.unique(num.array(x.astype(dtype))))
    assert np.array_equal(got, np.unique(x).astype(dtype))


def test_unique_scan_over_several_rounds():
    """More tiles than one round of the scan of their counts holds (16384), the last one short."""
    n = 4096 * 16385 + 5
    x = np.arange(n, dtype=np.uint32) // 3
    got = np.asarray(num.unique(num.array(x[::-1].copy())))
    assert np.array_equal(got, np.arange((n + 2) // 3, dtype=np.uint32))
