"""Which sorts deal their tiles per XCD (csrc/onesweep.h, claim_tile): one of a device's at a time.  Two that do may wait for each
other's workgroups until their bounded waits run out."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
from test_sort_gpu import lib, torch_cuda  # noqa: F401 (fixtures)

from cupynumeric_amd import _lib

pytestmark = pytest.mark.gpu


class _Sort:
    """An argsort (a plain sort for 8-byte keys) of one row, with its workspace."""

    def __init__(self, lib, torch, x, options=0):
        self.lib, self.torch, self.x, self.options = lib, torch, x, options
        self.code, self.argsort = _lib.DTYPE_CODES[x.dtype], x.dtype.itemsize == 4
        self.d_in = torch.from_numpy(x).cuda()
        self.out = torch.zeros(x.size, dtype=torch.int64, device="cuda")
        self.need = lib.cpn_local_sort_temp_bytes(self.code, x.size, x.size, int(not self.argsort), int(self.argsort), 0)
        self.temp = torch.full((self.need,), 0xA5, dtype=torch.uint8, device="cuda")

    def issue(self, stream):
        n, out = self.x.size, self.out.data_ptr()
        rc = self.lib.cpn_local_sort_ex(self.code, self.d_in.data_ptr(), None if self.argsort else out, out if self.argsort else None, n, n,
                                        0, 1, self.options, self.temp.data_ptr(), self.need, ctypes.c_void_p(stream.cuda_stream))
        assert rc == 0, _lib.status_string(rc)

    def check(self):
        """After a wait: right, and whether it dealt per XCD."""
        status, per_xcd = self.temp[:8].view(self.torch.int32).tolist()
        got = self.out.cpu().numpy()
        want = np.argsort(self.x, kind="stable") if self.argsort else np.sort(self.x)
        assert status == 0 and np.array_equal(got.view(want.dtype), want)
        return per_xcd == 1


def _keys(dtype, n, seed):
    return np.random.default_rng(seed).integers(0, 1 << (62 if np.dtype(dtype).itemsize == 8 else 31), n).astype(dtype)


# byte passes; byte passes of a row that may use virtual digits; equalised digits
@pytest.mark.parametrize("dtype, n", [(np.int32, 3_000_000), (np.int64, 3_000_000), (np.int64, 1 << 25)])
def test_while_another_has_the_order(lib, torch_cuda, dtype, n):
    torch = torch_cuda
    stream = torch.cuda.current_stream()
    sort = _Sort(lib, torch, _keys(dtype, n, 1))
    for hold in (0, 1, 0):
        assert lib.cpn_hold_tile_order(hold, ctypes.c_void_p(stream.cuda_stream)) == 0
        sort.out.fill_(-1)
        sort.issue(stream)
        torch.cuda.synchronize()
        assert sort.check() == (hold == 0)


def test_who_does_without(lib, torch_cuda):
    """Small tiles, and a request for the one counter; neither keeps the order from the next sort."""
    torch = torch_cuda
    stream = torch.cuda.current_stream()
    for x, options in ((_keys(np.int32, 1_500_000, 2), 0), (_keys(np.int32, 3_000_000, 3), _lib.CPN_SORT_SINGLE_TICKET)):
        sort = _Sort(lib, torch, x, options)
        sort.issue(stream)
        torch.cuda.synchronize()
        assert not sort.check()
    sort = _Sort(lib, torch, _keys(np.int32, 3_000_000, 4))
    for _ in range(2):
        sort.issue(stream)
        torch.cuda.synchronize()
        assert sort.check()


def test_streams_and_replays(lib, torch_cuda):
    """Sorts on several streams are right and leave the order free; a captured one takes it anew at each replay."""
    torch = torch_cuda
    streams = [torch.cuda.Stream() for _ in range(3)]
    sorts = [(_Sort(lib, torch, _keys(np.int32, 2_700_000 + 99 * i, i)), streams[i % 3]) for i in range(6)]
    torch.cuda.synchronize()
    for sort, stream in sorts:
        sort.issue(stream)
    torch.cuda.synchronize()
    for sort, _ in sorts:
        sort.check()
    sort = sorts[0][0]
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        sort.issue(torch.cuda.current_stream())
    stream = torch.cuda.current_stream()
    for hold in (0, 1, 0, 0):
        assert lib.cpn_hold_tile_order(hold, ctypes.c_void_p(stream.cuda_stream)) == 0
        sort.out.fill_(-1)
        graph.replay()
        torch.cuda.synchronize()
        assert sort.check() == (hold == 0)
