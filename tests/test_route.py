"""cpn_local_sort_route: the workspace size and the two bits beside it, for every request the same as the calls it stands for;
sorts that share one status word, on several streams and threads and in a captured graph."""
from __future__ import annotations

import threading

import numpy as np
import pytest

import cupynumeric_amd as num
from cupynumeric_amd import _lib
from cupynumeric_amd.runtime import STATUS_LINE_BYTES, runtime


def test_answers():
    lib = _lib.load()
    alone = 0
    for dtype, code in _lib.DTYPE_CODES.items():
        for n in (1, 7, 128, 1000, 4096, 6144, 6145, 16384, 20_000, 57_345, 100_000, 1 << 20):
            for rows in (1, 3):
                for values, indices, in_place in ((1, 0, 0), (0, 1, 0), (1, 0, 1)):
                    got = lib.cpn_local_sort_route(code, rows * n, n, values, indices, in_place)
                    need = lib.cpn_local_sort_temp_bytes(code, rows * n, n, values, indices, in_place)
                    fail = lib.cpn_local_sort_may_fail(code, rows * n, n, indices, need)
                    bits = _lib.CPN_ROUTE_MAY_FAIL | _lib.CPN_ROUTE_STATUS_ONLY
                    assert got & ~bits == need and bool(got & _lib.CPN_ROUTE_MAY_FAIL) == bool(fail), (dtype, n, rows)
                    only = bool(got & _lib.CPN_ROUTE_STATUS_ONLY)
                    assert only == (need == STATUS_LINE_BYTES and not fail), (dtype, n, rows)
                    alone += only
    assert alone > 100
    assert lib.cpn_local_sort_route(99, 10, 10, 1, 0, 0) == 0 and lib.cpn_local_sort_route(4, 10, 3, 1, 0, 0) == 0


class _Recorder:
    """Stands for torch: what is allocated, and when its stream is waited for."""

    uint8 = int32 = device = None

    def __init__(self, capturing=False):
        self.events, self.capturing, self.cuda = [], capturing, self

    def is_current_stream_capturing(self):
        return self.capturing

    def current_stream(self):
        return self

    def synchronize(self):
        self.events.append("wait")

    def zeros(self, *args, **kwargs):
        self.events.append("allocate")
        return self

    def data_ptr(self):
        self.events.append("publish")
        return 4096

    def __getitem__(self, where):
        return self

    def copy_(self, word):
        self.events.append("write")


def _runtime_on(torch):
    r = type(runtime)()
    r._torch, r._device_seen, r._current_device, r._devices = torch, True, lambda: 0, {0: "device"}
    return r


def test_line_is_published_after_its_stream_was_waited_for():
    """The line is memory that the allocator may have had from work still queued on the allocating stream: no other stream may
    write to it before that has run."""
    torch = _Recorder()
    r = _runtime_on(torch)
    assert r.status_line() == 4096 and torch.events == ["allocate", "wait", "publish"]
    assert r.status_line() == 4096 and torch.events == ["allocate", "wait", "publish"]  # once
    torch = _Recorder(capturing=True)
    assert _runtime_on(torch).status_line() is None and torch.events == []


def test_deferred_words_lie_where_no_earlier_work_writes():
    """The same for the words that sorts on any stream leave there."""
    torch = _Recorder()
    r = _runtime_on(torch)
    r.defer_flag(torch, "sort")
    r.defer_flag(torch, "sort")
    assert torch.events == ["allocate", "wait", "write", "write"]


@pytest.mark.gpu
def test_streams_and_threads_share_a_status_word():
    import torch

    x = np.random.default_rng(1).standard_normal((8, 40, 500)).astype(np.float32)
    want = np.sort(x, axis=-1)
    wrong = []

    def work(i):
        with torch.cuda.stream(torch.cuda.Stream()):
            for _ in range(20):
                got = np.asarray(num.sort(num.array(x[i])))
                if not np.array_equal(got, want[i]):
                    wrong.append(i)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not wrong
    lines = {a for a in runtime._status_lines.values()}
    assert len(lines) == 1 and all(int(m[:4].view(torch.int32).item()) == 0 for m in runtime._status_memory)


@pytest.mark.gpu
def test_captured():
    import torch

    from cupynumeric_amd._thunk import DeviceArray

    rng = np.random.default_rng(2)
    buf = torch.zeros(1000, dtype=torch.float64, device="cuda")
    a = num.ndarray((1000,), np.float64, thunk=DeviceArray.from_device(buf, (1000,), np.float64))
    num.sort(a)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = num.sort(a)
    for _ in range(4):
        x = rng.standard_normal(1000)
        buf.copy_(torch.from_numpy(x))
        graph.replay()
        torch.cuda.synchronize()
        assert np.array_equal(out._thunk.base.device().view(torch.float64).cpu().numpy(), np.sort(x))
        assert np.array_equal(np.asarray(num.sort(num.array(x[:300]))), np.sort(x[:300]))
