"""Device-array thunk: the slice of the reference's `DeferredArray` that the sort path uses
(`cupynumeric/_thunk/deferred.py`: `sort` :5453-5474, `copy` :394-398, `swapaxes` :2341-2351,
`reshape` :2136-2316), over a dense row-major device buffer instead of a Legate store.
"""
from __future__ import annotations

import ctypes
from typing import TYPE_CHECKING, Any

import numpy as np

from . import _lib
from ._sort import sort_deferred, sort_task
from .runtime import runtime

if TYPE_CHECKING:
    import torch

# Where in its workspace `cpn_unique` may put the count: beside the status word, in a line that nothing else uses.
UNIQUE_COUNT_OFFSET = 64
# From so many values on they are grouped by the parts of the array (`cpn_searchsorted_grouped`), where that is done.  us per call,
# grouped / each value by itself, values spread as the array / half of them in a thousandth of it:
#   float32   in 2^21     262 144  44 / 25  51 / 19   393 216  48 / 34  53 / 27   524 288  51 / 44  54 / 35   786 432  60 / 65  57 / 50
#             in 4*10^6   262 144  38 / 33  50 / 23   393 216  39 / 44  52 / 31   524 288  40 / 55  53 / 40   786 432  43 / 79  59 / 58
#             in 3*10^7   262 144  78 / 51  94 / 31   393 216  79 / 77  95 / 42   524 288  80 / 95 101 / 54   786 432  82 / 126 105 / 79
#   float64   in 2^20     262 144  50 / 25  54 / 20   393 216  53 / 34  56 / 28   524 288  58 / 44  58 / 36   786 432  65 / 61  60 / 49
#             in 4*10^6   262 144  49 / 38  59 / 25   393 216  50 / 51  61 / 33   524 288  51 / 64  63 / 43   786 432  52 / 92  68 / 62
#             in 3*10^7   262 144 116 / 55 129 / 33   393 216 119 / 80 132 / 44   524 288 119 / 100 136 / 57  786 432 123 / 146 142 / 82
GROUPED_MIN_VALUES = (1 << 19) + 1
# Up to so many of 4 and 8 bytes are not sorted first in a long array where they are not grouped; sorted / each by itself:
#   float32   in 2^28     524 288 165 / 149 130 / 87   786 432 253 / 188 215 / 145   2^20 270 / 229 232 / 157   3*2^19 322 / 348 286 / 225
#   float64   in 2^27     524 288 243 / 152 210 / 94   786 432 353 / 193 317 / 153   2^20 377 / 232 340 / 164   3*2^19 433 / 346 397 / 225
UNSORTED_MAX_VALUES = 1 << 20
# Longest array of integers that `unique` splits by sampled keys (`cpn_local_sort_split_temp_bytes`).  Arrays that it is asked
# of repeat their values, and 8-byte ones mostly leave upper bytes constant, whose passes the sort of `cpn_unique` skips.
# us per call that way / split, int64 below 10^9 of as many values, of a quarter as many, of 1000, and of full range:
#   2^20 + 1  130 / 116  129 / 117   97 / 102  194 / 118        2^21       149 / 126  148 / 133  106 / 110  229 / 123
#   3*10^6    161 / 152  160 / 161  115 / 119  251 / 152        2^22 - 1   175 / 177  172 / 185  121 / 126  271 / 173
#   2^22      206 / 211  162 / 164   (hashed)  299 / 204        2^23       297 / 306  293 / 318   (hashed)  469 / 296
UNIQUE_SPLIT_INTEGERS = 3 << 20

# dtypes the reference supports (`cupynumeric/_utils/array.py:28-43`)
SUPPORTED_DTYPES = tuple(_lib.DTYPE_CODES.keys())


def check_dtype(dtype: Any) -> np.dtype:
    """Same error text as `to_core_type` (`cupynumeric/_utils/array.py:64-68`)."""
    try:
        dt = np.dtype(dtype)
    except TypeError:
        raise TypeError(f"cuPyNumeric does not support dtype={dtype}")
    if dt not in _lib.DTYPE_CODES:
        raise TypeError(f"cuPyNumeric does not support dtype={dt}")
    return dt


class Storage:
    """A dense device buffer.  Host data handed in at creation is uploaded on first device use,
    so that building an array does not need a GPU (Legate attaches host data lazily as well)."""

    def __init__(self, nbytes: int, host: np.ndarray | None = None) -> None:
        self.nbytes = int(nbytes)
        self._host = host
        self._dev: "torch.Tensor | None" = None

    def device(self) -> "torch.Tensor":
        if self._dev is None:
            if self._host is not None:
                self._dev = runtime.upload(self._host)
                self._host = None
            else:
                self._dev = runtime.empty_bytes(self.nbytes)
        return self._dev

    def ptr(self) -> int:
        return int(self.device().data_ptr())

    def to_numpy(self, shape: tuple[int, ...], dtype: np.dtype) -> np.ndarray:
        if 0 in shape:
            return np.empty(shape, dtype=dtype)  # nothing to fetch; works without a device
        if self._dev is None and self._host is not None:
            return np.array(self._host, dtype=dtype).reshape(shape)
        return runtime.download(self.device(), shape, dtype)


class DeviceArray:
    """Shape + dtype + `base` storage.  `base` can be re-bound, as the reference's sort helpers
    do with `output.base = result.base` (`cupynumeric/_thunk/_sort.py:47,73,76`)."""

    def __init__(self, shape: tuple[int, ...], dtype: Any, base: Storage | None = None) -> None:
        self.shape = tuple(map(int, shape))
        self.dtype = check_dtype(dtype)
        self.base = base if base is not None else Storage(self.size * self.dtype.itemsize)

    @classmethod
    def from_numpy(cls, arr: np.ndarray) -> "DeviceArray":
        dt = check_dtype(arr.dtype)
        host = np.array(arr, dtype=dt, order="C", copy=True)
        return cls(host.shape, dt, Storage(host.nbytes, host=host))

    @classmethod
    def from_device(cls, buf: "torch.Tensor", shape: tuple[int, ...], dtype: Any) -> "DeviceArray":
        """An array over device memory that already holds its dense row-major data: `buf` is a
        contiguous torch tensor on the GPU (any element type) of exactly the array's bytes.  The
        memory is shared, not copied."""
        dt = check_dtype(dtype)
        raw = buf.reshape(-1).view(runtime.torch.uint8)
        out = cls(shape, dt, Storage(raw.numel()))
        if raw.numel() != out.size * dt.itemsize or not raw.is_cuda:
            raise ValueError("from_device: the buffer must be device memory of exactly shape x dtype bytes")
        out.base._dev = raw
        return out

    @property
    def ndim(self) -> int:
        return len(self.shape)

    @property
    def size(self) -> int:
        n = 1
        for s in self.shape:
            n *= s
        return n

    def __numpy_array__(self) -> np.ndarray:
        return self.base.to_numpy(self.shape, self.dtype)

    # -- data movement the sort path needs ------------------------------------------------
    def reshape(self, newshape: tuple[int, ...], order: str = "C") -> "DeviceArray":
        """C-order reshape.  Buffers are always dense row-major, so the storage is shared."""
        if order != "C":
            raise NotImplementedError("only C-order reshape is used by the sort path")
        out = DeviceArray(newshape, self.dtype, self.base)
        if out.size != self.size:
            raise ValueError("cannot reshape array: sizes differ")
        return out

    def copy(self) -> "DeviceArray":
        """Dense copy with storage of its own (`DeferredArray.copy(deep=True)`, `cupynumeric/_thunk/deferred.py:394-398`);
        host data that has not been uploaded yet is copied on the host."""
        if self.base._dev is None and self.base._host is not None:
            return DeviceArray.from_numpy(np.asarray(self.base._host).reshape(self.shape))
        sub = Storage(self.size * self.dtype.itemsize)
        if self.size:
            sub._dev = self.base.device()[: sub.nbytes].clone()
        return DeviceArray(self.shape, self.dtype, sub)

    def slice_first_axis(self, i: int, count: int, shape: tuple[int, ...]) -> "DeviceArray":
        """`self[i]` as an array of `shape` (`count` elements) over the same memory: rows of a
        dense row-major buffer are themselves dense."""
        nbytes = count * self.dtype.itemsize
        sub = Storage(nbytes)
        if self.base._dev is None and self.base._host is not None:
            host = np.asarray(self.base._host).reshape(self.shape)
            sub._host = np.ascontiguousarray(host[i])
        else:
            sub._dev = self.base.device()[i * nbytes : (i + 1) * nbytes] if nbytes else runtime.empty_bytes(0)
        return DeviceArray(shape, self.dtype, sub)

    def swapaxes_copy(self, axis1: int, axis2: int) -> "DeviceArray":
        """Dense copy with two axes exchanged: the reference's `swapaxes` view followed by
        `copy(deep=True)` (`cupynumeric/_thunk/_sort.py:59-65`) in one kernel."""
        shape = list(self.shape)
        shape[axis1], shape[axis2] = shape[axis2], shape[axis1]
        out = DeviceArray(tuple(shape), self.dtype)
        if self.size == 0:
            return out
        lib = _lib.load()
        c_shape = (ctypes.c_int64 * max(self.ndim, 1))(*self.shape)
        status = lib.cpn_swapaxes_copy(
            self.dtype.itemsize,
            self.base.ptr(),
            out.base.ptr(),
            c_shape,
            self.ndim,
            axis1,
            axis2,
            runtime.stream_handle(),
        )
        _lib.check(status, "cpn_swapaxes_copy")
        return out

    def take_along_last_axis(self, indices: "DeviceArray", check: str = "now") -> "DeviceArray":
        """`take_along_axis(self, indices, axis=-1)` for arrays whose leading dimensions agree
        (`cupynumeric/_module/indexing.py:648-760`; the TAKE task's no-broadcast case).

        `check`: what happens to the kernel's out-of-bounds flag.  "now": read back before returning
        (one stream synchronisation; the public `take_along_axis` raises IndexError from the call, as
        the reference does); "deferred": reported with the next host read (`runtime.flush_status`), so
        that the stream keeps running; "trusted": no flag at all, for indices that this package
        produced itself (the argsorts inside `lexsort`)."""
        if indices.dtype != np.dtype(np.int64):
            raise TypeError("`indices` must be an int64 array")
        if self.ndim != indices.ndim or self.ndim == 0:
            raise ValueError("`indices` and `a` must have the same number of dimensions")
        lead_a, lead_i = self.shape[:-1], indices.shape[:-1]
        if any(m != n and m != 1 and n != 1 for m, n in zip(lead_a, lead_i)):
            raise IndexError(
                "shape mismatch: indexing arrays could not be broadcast together with shapes "
                f"{self.shape} {indices.shape} (every dimension but the axis must agree or be 1)"
            )
        lead_out = tuple(max(m, n) if min(m, n) != 0 else 0 for m, n in zip(lead_a, lead_i))
        out = DeviceArray(lead_out + indices.shape[-1:], self.dtype)
        if out.size == 0:
            return out
        if self.shape[-1] == 0:
            raise IndexError("index out of bounds: cannot take from an empty axis")
        lib = _lib.load()
        if runtime.check_mode == "off":
            check = "trusted"
        elif runtime.check_mode == "eager" and check == "deferred":
            check = "now"
        flag = runtime.zero_flag() if check != "trusted" else None
        flag_ptr = flag.data_ptr() if flag is not None else None
        stream = ctypes.c_void_p(runtime.stream_handle())
        if lead_a == lead_i:
            status = lib.cpn_take_along_last_axis(
                self.dtype.itemsize, self.base.ptr(), indices.base.ptr(), out.base.ptr(), out.size // indices.shape[-1],
                self.shape[-1], indices.shape[-1], flag_ptr, stream,
            )
        else:
            # rows per step of each leading dimension on either side: the dense stride, 0 where broadcast
            def row_strides(lead: tuple[int, ...]) -> list[int]:
                strides, run = [0] * len(lead), 1
                for d in range(len(lead) - 1, -1, -1):
                    strides[d] = run if lead[d] != 1 else 0
                    run *= lead[d]
                return strides

            n = len(lead_out)
            u64 = ctypes.c_uint64 * max(n, 1)
            status = lib.cpn_take_along_last_axis_broadcast(
                self.dtype.itemsize, self.base.ptr(), indices.base.ptr(), out.base.ptr(), n, u64(*lead_out),
                u64(*row_strides(lead_a)), u64(*row_strides(lead_i)), self.shape[-1], indices.shape[-1], flag_ptr, stream,
            )
        _lib.check(status, "cpn_take_along_last_axis")
        if check == "deferred":
            runtime.defer_flag(flag, "index")
        elif check == "now":
            runtime.flush_status()  # (errors of earlier work first: the read below synchronises anyway)
            if int(flag.item()) != 0:
                raise IndexError("index out of bounds in take_along_axis")
        return out

    # -- the sort entry point ---------------------------------------------------------------
    def sort(
        self,
        rhs: "DeviceArray",
        argsort: bool = False,
        axis: int | None = -1,
        kind: str = "quicksort",
        order: str | list[str] | None = None,
    ) -> None:
        """`DeferredArray.sort` (`cupynumeric/_thunk/deferred.py:5453-5474`): `self` receives the
        result of sorting `rhs`."""
        # (messages and exception types are the reference's: callers and its tests match on them)
        if order is not None:
            raise NotImplementedError(
                "cuPyNumeric does not support sorting with 'order' as "
                "ndarray only supports numeric values"
            )
        if axis is not None and not -rhs.ndim <= axis < rhs.ndim:
            raise ValueError("invalid axis")
        # only "stable" sets the flag (any other kind, "mergesort" included, does not); every kernel
        # here is stable whatever the flag says
        sort_deferred(self, rhs, argsort, axis, stable=(kind == "stable"))

    def partition(
        self,
        rhs: "DeviceArray",
        kth: Any,
        argpartition: bool = False,
        axis: int | None = -1,
        kind: str = "introselect",
        order: str | list[str] | None = None,
    ) -> None:
        """`DeferredArray.partition` (`cupynumeric/_thunk/deferred.py:5476-5494`): falls back to an
        (unstable-flagged) sort, which satisfies the partition property for every `kth`."""
        if order is not None:
            raise NotImplementedError(
                "cuPyNumeric does not support partitioning with 'order' as "
                "ndarray only supports numeric values"
            )
        if axis is not None and not -rhs.ndim <= axis < rhs.ndim:
            raise ValueError("invalid axis")
        sort_deferred(self, rhs, argpartition, axis, False)  # a sorted row is partitioned at every kth

    def astype(self, dtype: Any) -> "DeviceArray":
        """Dense copy converted to `dtype` (`DeferredArray.convert`, `cupynumeric/_thunk/deferred.py:1899-1937`,
        a UNARY_OP convert task in the reference)."""
        dt = check_dtype(dtype)
        out = DeviceArray(self.shape, dt)
        if self.size == 0:
            return out
        lib = _lib.load()
        status = lib.cpn_astype(
            _lib.DTYPE_CODES[self.dtype],
            self.base.ptr(),
            _lib.DTYPE_CODES[dt],
            out.base.ptr(),
            self.size,
            ctypes.c_void_p(runtime.stream_handle()),
        )
        _lib.check(status, "cpn_astype")
        return out

    def searchsorted(self, rhs: "DeviceArray", v: "DeviceArray", side: str = "left") -> None:
        """`DeferredArray.searchsorted` (`cupynumeric/_thunk/deferred.py:5425-5451`): `self` (int64,
        shape of `v`) receives the insertion points of `v` into the sorted 1-D `rhs`.  Any
        `side` other than "left" means "right", as in the reference (`is_left = side == "left"`)."""
        is_left = side == "left"
        if v.size == 0:
            return
        if rhs.dtype != v.dtype or self.dtype != np.dtype(np.int64):
            raise TypeError("searchsorted: arrays must share one dtype and the result must be int64")
        lib = _lib.load()
        code = _lib.DTYPE_CODES[rhs.dtype]
        stream = ctypes.c_void_p(runtime.stream_handle())
        if v.size >= GROUPED_MIN_VALUES:
            args = (code, rhs.base.ptr() if rhs.size else None, rhs.size)
            temp_bytes = lib.cpn_searchsorted_grouped_temp_bytes(*args, v.size)
            if temp_bytes != 0:  # (cannot fail on the device: no status to look at)
                temp = runtime.empty_bytes(temp_bytes)
                status = lib.cpn_searchsorted_grouped(
                    *args, v.base.ptr(), v.size, int(is_left), self.base.ptr(), temp.data_ptr(), temp_bytes, stream
                )
                _lib.check(status, "cpn_searchsorted")
                return
        if v.size <= UNSORTED_MAX_VALUES and rhs.dtype.itemsize >= 4 and rhs.dtype.kind != "c":
            temp_bytes = 0
        else:
            temp_bytes = lib.cpn_searchsorted_temp_bytes(code, rhs.size, v.size)
        temp = runtime.empty_bytes(temp_bytes) if temp_bytes else None
        status = lib.cpn_searchsorted(
            code,
            rhs.base.ptr() if rhs.size else None,
            rhs.size,
            v.base.ptr(),
            v.size,
            int(is_left),
            self.base.ptr(),
            temp.data_ptr() if temp is not None else None,
            temp_bytes,
            stream,
        )
        _lib.check(status, "cpn_searchsorted")
        if temp is not None and runtime.check_mode == "lazy":
            runtime.defer_status(temp)  # (the values were sorted first: that sort's status word)
        elif temp is not None and runtime.check_mode == "eager":
            _lib.check(lib.cpn_local_sort_check(temp.data_ptr(), stream), "cpn_searchsorted")

    def unique(self) -> "DeviceArray":
        """`DeferredArray.unique` (`cupynumeric/_thunk/deferred.py:5375-5395`): sorted distinct
        values of the flattened array.  The result size is only known on the device (an unbound
        store in the reference) and read back before the call returns."""
        if self.size == 0:
            return DeviceArray((0,), self.dtype)
        lib = _lib.load()
        code = _lib.DTYPE_CODES[self.dtype]
        stream = ctypes.c_void_p(runtime.stream_handle())
        list_offset = ctypes.c_uint64()
        few_bytes = lib.cpn_distinct_temp_bytes(code, self.size, ctypes.byref(list_offset))
        split = self.dtype.kind == "f" or self.size <= UNIQUE_SPLIT_INTEGERS
        split = split and lib.cpn_local_sort_split_temp_bytes(code, self.size, self.size, 0) != 0
        temp_bytes = (lib.cpn_unique_sorted_temp_bytes if split else lib.cpn_unique_temp_bytes)(code, self.size)
        if temp_bytes == 0:
            raise NotImplementedError(f"cpn_unique: no workspace layout for dtype={self.dtype}, size={self.size}")
        out = DeviceArray((self.size,), self.dtype)
        temp = runtime.empty_bytes(max(temp_bytes + 8, few_bytes))
        if few_bytes != 0:
            few = self._unique_by_hash(lib, code, temp, list_offset.value, stream)
            if few is not None:
                return few
        if split:  # the sort that cannot fail on the device, then what follows it
            ordered = DeviceArray((self.size,), self.dtype)
            sort_task(ordered, DeviceArray((self.size,), self.dtype, self.base), False, True)
            at = temp_bytes
            status = lib.cpn_unique_sorted(
                code, ordered.base.ptr(), out.base.ptr(), self.size, temp.data_ptr() + at, temp.data_ptr(), temp_bytes, stream
            )
        else:
            at = UNIQUE_COUNT_OFFSET
            status = lib.cpn_unique(
                code, self.base.ptr(), out.base.ptr(), self.size, temp.data_ptr() + at, temp.data_ptr(), temp_bytes, stream
            )
        _lib.check(status, "cpn_unique")
        if runtime.check_mode != "off":
            runtime.flush_status()  # errors of earlier work first
        # one copy brings the count, and the status word where there is one
        head = temp[0 if not split else at : at + 8].cpu().numpy()
        if not split and runtime.check_mode != "off" and head[:4].view(np.uint32)[0] != 0:
            _lib.check(_lib.CPN_ERR_DEVICE, "cpn_unique")
        n_unique = int(head[-8:].view(np.int64)[0])
        return DeviceArray((n_unique,), self.dtype, out.base)

    def _unique_by_hash(self, lib: Any, code: int, temp: Any, list_offset: int, stream: Any) -> "DeviceArray | None":
        """`unique` of an integer array with few values for its length: they are collected unsorted
        (`cpn_distinct`), then sorted.  None: not such an array."""
        if runtime.check_mode != "off":
            runtime.flush_status()  # errors of earlier work first
        args = (code, self.base.ptr(), self.size)
        _lib.check(lib.cpn_distinct_plan(*args, temp.data_ptr(), temp.numel(), stream), "cpn_distinct_plan")
        head = temp[:24].view(runtime.torch.int32)
        mode, _, _, _, _, doubt = head.tolist()  # (waits, so that an array that is sorted after all waits for no more than this)
        if mode == 0 or doubt != 0:
            return None
        _lib.check(lib.cpn_distinct(*args, mode, temp.data_ptr(), temp.numel(), stream), "cpn_distinct")
        _, failed, count, *_ = head.tolist()
        if failed != 0:
            return None
        found = DeviceArray.from_device(temp[list_offset : list_offset + count * self.dtype.itemsize], (count,), self.dtype)
        out = DeviceArray((count,), self.dtype)
        sort_task(out, found, False, True)
        if runtime.check_mode != "off":
            runtime.flush_status()  # (more values than a row split takes: a sort that can fail)
        return out

    def to_complex(self, dtype: Any) -> "DeviceArray":
        """Real -> complex cast (`astype` in `sort_complex`, `cupynumeric/_module/ssc_sorting.py:150-159`)."""
        dt = check_dtype(dtype)
        out = DeviceArray(self.shape, dt)
        if self.size == 0:
            return out
        lib = _lib.load()
        status = lib.cpn_real_to_complex(
            _lib.DTYPE_CODES[self.dtype],
            self.base.ptr(),
            _lib.DTYPE_CODES[dt],
            out.base.ptr(),
            self.size,
            runtime.stream_handle(),
        )
        _lib.check(status, "cpn_real_to_complex")
        return out
