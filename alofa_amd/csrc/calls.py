"""The C entries by way of ctypes, where the binding (host/binding) can be neither found nor built (no C++ compiler, or no Python headers). The
answers are the binding's: ``call`` the entry's own, and the checks the sizes that a launch needs, or None, which leaves the operands to the checks
in Python. Some 12 us a product instead of 3."""
from __future__ import annotations

import ctypes
import threading

import torch

_entry = ctypes.CFUNCTYPE(ctypes.c_int)
_entries: dict = {}      # address -> the entry (no parameter types: every argument below brings its own)


def call(address, *args) -> int:
    entry = _entries.get(address)
    if entry is None:
        if not address:
            raise ValueError("call: no such entry")
        entry = _entries[address] = _entry(address)
    passed = []
    for a in args:
        if isinstance(a, float):
            passed.append(ctypes.c_float(a))
        elif isinstance(a, int):
            if not -(1 << 63) <= a < 1 << 63:
                raise OverflowError("call: the number does not fit 64 bits")
            passed.append(ctypes.c_int64(a))
        elif a is None or isinstance(a, torch.Tensor):
            passed.append(ctypes.c_void_p(None if a is None else a.data_ptr()))
        else:
            raise TypeError(f"call: a {type(a).__name__} is no tensor, number or None")
    return entry(*passed)


class _Noting(threading.local):
    calls = None


_noting = _Noting()


def note(address, *args) -> int:
    rc = call(address, *args)
    if _noting.calls is not None and rc == 0:
        _noting.calls.append((address, [a.data_ptr() if isinstance(a, torch.Tensor) else a for a in args]))
    return rc


def tape() -> None:
    _noting.calls = []


def taped(*ranges):
    calls, _noting.calls = _noting.calls, None
    if calls is None:
        raise RuntimeError("taped: no tape is being written")
    inside = lambda x: next(((r, x - at) for r, (at, size) in enumerate(ranges) if 0 <= x - at < size), None) if isinstance(x, int) else None      # noqa: E731
    return len(ranges), [(address, args, {k: inside(x) for k, x in enumerate(args) if inside(x) is not None}) for address, args in calls]


def play(tape, at) -> int:
    ranges, calls = tape
    if len(at) != ranges:
        raise ValueError("play: another count of ranges than the tape's")
    for address, args, places in calls:
        rc = call(address, *[at[places[k][0]] + places[k][1] if k in places else x for k, x in enumerate(args)])
        if rc != 0:
            return rc
    return 0


def _leading(t) -> int:
    """The leading dimension of a matrix on the GPU with contiguous rows; -1 for anything else."""
    if not isinstance(t, torch.Tensor) or not t.is_cuda or t.dim() != 2 or (t.stride(1) != 1 and t.shape[1] > 1):
        return -1
    return t.stride(0) if t.shape[0] > 1 else max(t.stride(0), t.shape[1])


def product(out, a, w, w2, bias):
    lds = ldo, lda, ldw = _leading(out), _leading(a), _leading(w)
    if min(lds) < 0 or a.dtype is not torch.bfloat16 or w.dtype is not torch.bfloat16 or out.dtype not in (torch.float32, torch.bfloat16):
        return None
    (M, K), N = a.shape, w.shape[0]
    if w.shape[1] != K or tuple(out.shape) != (M, N) or K % 8 or lda % 8 or ldw % 8 or a.data_ptr() % 16 or w.data_ptr() % 16:
        return None
    if w2 is not None and (out.dtype is not torch.bfloat16 or _leading(w2) != ldw or w2.dtype is not torch.bfloat16 or tuple(w2.shape) != (N, K) or w2.data_ptr() % 16):
        return None
    if bias is not None and not (isinstance(bias, torch.Tensor) and bias.is_cuda and bias.dtype is torch.float32 and bias.dim() == 1 and bias.is_contiguous() and bias.shape[0] == N):
        return None
    return M, N, K, ldo, lda, ldw, int(out.dtype is torch.bfloat16)


def _left_to_python(*operands):
    return None


norm = caches = turn = attention = _left_to_python
