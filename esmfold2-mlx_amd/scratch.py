"""One device-memory scratch buffer per GPU, shared by every module of this package.

The kernels' scratch (the triangle update's a, b and x planes, the 8-bit linear's
split-K partials) is live only during one call, so a trunk of many updates, or an
ESMC of many linears, needs one buffer sized for its largest call rather than one
per module (a 6B fold's 68 updates at L=512 would otherwise hold 68 x 201 MB).

Rules:
  * ``get`` returns a 256-byte aligned view of the device's buffer with at least the
    requested bytes, growing the buffer when a call needs more. Every stream that has used
    the buffer is recorded on it (``Tensor.record_stream``), so when a grown buffer replaces
    it the caching allocator keeps the old memory until the work queued on each of those
    streams is done.
  * Calls on one device are ordered through the buffer: a user holds ``guard(device)`` from its
    ``get`` until the launches that touch the bytes are queued, so two threads never interleave
    theirs (a native call runs without the interpreter lock). When ``get`` is called on a stream
    other than the buffer's last user, that stream first waits for the work already queued on
    the last user (``wait_stream``), so two streams never run their scratch users at once.
    Under HIP-graph capture no wait is recorded (the caller orders the capture).
  * Each ``get`` starts a new generation: a view handed out earlier (``Q8Linear.partials``)
    is valid only until the next ``get`` on that device, which ``check_generation`` tells (the
    consumer holds the guard from that check until it is queued).
  * A HIP graph that captured calls keeps the buffers they used alive: ``current`` gives
    the buffer to hold next to the graph.
"""

from __future__ import annotations

import contextlib
import threading
from dataclasses import dataclass

import torch

ALIGN = 256
_lock = threading.Lock()


@dataclass
class _Slot:
    buf: torch.Tensor
    stream: torch.cuda.Stream          # the last stream that called get()
    generation: int = 0


_slots: dict[int, _Slot] = {}
_guards: dict[int, threading.RLock] = {}
_UNGUARDED = contextlib.nullcontext()


def _index(device) -> int:
    d = device if type(device) is torch.device else (
        torch.device(device) if device is not None else torch.device("cuda", torch.cuda.current_device()))
    if d.type != "cuda":
        raise ValueError(f"scratch lives in device memory, got {d}")
    return torch.cuda.current_device() if d.index is None else d.index


def guard(device=None, nbytes: int = 1):
    """The lock that a user of the device's scratch holds from its ``get`` until its launches are queued (for a
    call that turns out to need none, ``nbytes`` 0, one that nobody waits for)."""
    if not nbytes:
        return _UNGUARDED
    idx = _index(device)
    g = _guards.get(idx)
    return _guards.setdefault(idx, threading.RLock()) if g is None else g


def _claim(nbytes: int, device):
    """(the device's buffer, grown if need be, the current stream on it)."""
    idx = _index(device)
    need = max(int(nbytes), 1) + ALIGN
    stream = torch.cuda.current_stream(idx)
    with _lock:
        slot = _slots.get(idx)
        moved = slot is not None and slot.stream != stream
        capturing = moved and torch.cuda.is_current_stream_capturing()
        if moved and not capturing:
            stream.wait_stream(slot.stream)  # the previous user's queued work first
        if slot is None or slot.buf.numel() < need:
            # grow geometrically so a slowly rising size does not reallocate every call; the
            # old buffer is freed here, and record_stream has told the allocator who used it
            size = need if slot is None else max(need, slot.buf.numel() + slot.buf.numel() // 4)
            buf = torch.empty(size, dtype=torch.uint8, device=torch.device("cuda", idx))
            slot = _slots[idx] = _Slot(buf, stream, 0 if slot is None else slot.generation)
        elif moved:
            if not capturing:
                slot.buf.record_stream(stream)
            slot.stream = stream
        slot.generation += 1
        return slot.buf, stream


def get(nbytes: int, device=None) -> torch.Tensor:
    """A uint8 view of ``nbytes`` (>= 1) at a 256-byte aligned address of the device's scratch, for a caller
    that holds ``guard(device)`` until the launches that use it are queued."""
    buf, _ = _claim(nbytes, device)
    off = (-buf.data_ptr()) % ALIGN
    return buf[off:off + max(int(nbytes), 1)]


def take(nbytes: int, device=None):
    """``get`` for one launch: (buffer, 256-byte aligned address in it, raw stream). The caller holds the
    buffer and ``guard(device)`` until its launches are queued."""
    buf, stream = _claim(nbytes, device)
    return buf, (buf.data_ptr() + ALIGN - 1) // ALIGN * ALIGN, stream.cuda_stream


def generation(device=None) -> int:
    """How many times the device's scratch has been handed out (0 before the first ``get``)."""
    with _lock:
        slot = _slots.get(_index(device))
        return 0 if slot is None else slot.generation


def check_generation(gen: int, device=None, what: str = "a scratch view") -> None:
    """Raise if the scratch was handed out again since ``gen``: a view from then is overwritten."""
    now = generation(device)
    if now != gen:
        raise RuntimeError(f"{what} is stale: the device scratch was reused ({now - gen} later call(s)) "
                           "before it was consumed")


def current(device=None) -> torch.Tensor | None:
    """The device's scratch buffer now (None before the first ``get``)."""
    with _lock:
        slot = _slots.get(_index(device))
        return None if slot is None else slot.buf


def reserved(device=None) -> int:
    """Bytes held by the device's scratch buffer."""
    b = current(device)
    return 0 if b is None else b.numel()


def release(device=None) -> None:
    """Drop the device's scratch buffer (the next call allocates a new one)."""
    with _lock:
        _slots.pop(_index(device), None)
