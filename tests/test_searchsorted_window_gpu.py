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
