"""Workspaces of the split-K kernels: one per shape for MLA decode and the fused gate_up + silu
kernels (`ScratchCache`), one for all shapes for paged decode (`SharedScratch`).

Each of those kernels keeps arrival counters at the end of its workspace: every launch
bumps them and the last arrival returns them to zero, so a buffer is zero-filled once and
then reused. Two launches that overlap on one buffer would interfere (a counter reset by
one launch can erase another's increment), so a buffer belongs to one stream: the cache
key holds the launch stream beside the device and the shape. During torch.cuda.graph capture
the current stream is the capture stream, so graphs captured on one capture stream share
buffers and must be replayed one after another on a single stream; graphs that replay
concurrently need distinct capture streams.

With `EMBERSERVE_CHECK_INDICES=1` the caller verifies after each launch that the counter
region is back at zero (`verify_counters`). A non-zero counter (an aborted launch, or an
overlap the rule above forbids) would otherwise leave some rows unmerged on every later
call; the check re-zeroes the region with a fill kernel (never a memset, so it is safe
inside a captured graph) and raises.
"""

from __future__ import annotations

import threading
from ctypes import byref, c_uint64
from typing import Callable, NamedTuple

import torch
from torch import Tensor

from . import _lib


def _stream_key(device: torch.device) -> int:
    idx = device.index if device.index is not None else torch.cuda.current_device()
    return torch._C._cuda_getCurrentRawStream(idx)


class _Verified:
    what: str

    def verify_counters(self, buf: Tensor, start_bytes: int, end_bytes: int) -> None:
        """Raises RuntimeError (after re-zeroing them) when the counters in
        [start_bytes, end_bytes) of `buf` are not all zero. Synchronises."""
        region = buf.view(torch.int32)[start_bytes // 4:end_bytes // 4]
        if bool(region.any()):
            region.zero_()
            raise RuntimeError(f"{self.what}: split-K arrival counters were left non-zero (an aborted "
                               "launch, or two overlapping launches on one workspace); re-zeroed")


class ScratchCache(_Verified):
    """Zero-filled workspaces keyed by (shape key, device, current stream)."""

    def __init__(self, what: str, min_bytes: int = 256) -> None:
        self.what = what
        self.min_bytes = min_bytes
        self._bufs: dict[tuple, Tensor] = {}

    def get(self, key: tuple, nbytes: Callable[[], int], device: torch.device) -> Tensor:
        full = (*key, str(device), _stream_key(device))
        buf = self._bufs.get(full)
        if buf is None:
            n = int(nbytes())
            if n < 0:
                raise ValueError(f"{self.what}: no workspace for {key}")
            buf = torch.zeros(max(n, self.min_bytes) // 4, dtype=torch.float32, device=device)
            self._bufs[full] = buf
        return buf

    def __len__(self) -> int:
        return len(self._bufs)


class _Buffer(NamedTuple):
    tensor: Tensor
    partial: int    # bytes at the front that partials may use
    counters: int   # bytes at the end that counters may use, zero between launches
    capture: int    # the graph capture that recorded the counters' zero fill, 0: filled eagerly


class SharedScratch(_Verified):
    """One workspace per (thread, device, current stream) for calls of every shape, for an entry
    point that keeps its partials at the workspace's start and its counters at the end
    (ember_paged_decode_shared). Per thread, because a call may be two launches (the fp32 kernel and
    its merge), between which another thread's on the same stream would overwrite its partials. The
    split count varies with the batch, so that a workspace for each shape, kept for good, came to
    1.3 GB over batches of 1 to 256 (32q/8kv x 128, 8192-key tables), against 40 MB here. The
    partials' part at least doubles when it grows. An outgrown buffer is kept, because a captured
    graph may hold its address: all of a stream's together are at most four times its largest
    call's need.

    A call captured where no eager call has left a large enough workspace gets one that belongs to
    that capture: its memory is the graph's own, and the zero fill of its counters is recorded in
    the graph, which therefore replays correctly whichever graphs ran before it."""

    MIN_PARTIAL = 1 << 20
    MIN_COUNTERS = 1 << 14

    def __init__(self, what: str) -> None:
        self.what = what
        self._bufs: dict[tuple, _Buffer] = {}
        self._captured: dict[tuple, _Buffer] = {}
        self._outgrown: list[Tensor] = []
        self._lock = threading.Lock()

    def get(self, partial: int, counters: int, device: torch.device) -> Tensor:
        """A workspace for `partial` bytes of partials and `counters` bytes of counters."""
        key = (threading.get_ident(), device.index, _stream_key(device))
        buf = self._bufs.get(key)
        if buf is None or partial > buf.partial or counters > buf.counters:
            buf = self._grow(key, partial, counters, device)
        return buf.tensor

    def _grow(self, key: tuple, partial: int, counters: int, device: torch.device) -> _Buffer:
        capture = _capture_id(device)
        bufs = self._captured if capture else self._bufs
        with self._lock:
            old = bufs.get(key)
            if old is not None and old.capture == capture:
                if partial <= old.partial and counters <= old.counters:
                    return old
                partial = max(partial, 2 * old.partial if partial > old.partial else old.partial)
                counters = max(counters, 2 * old.counters if counters > old.counters else old.counters)
            partial = round_up(max(partial, self.MIN_PARTIAL), 256)
            counters = round_up(max(counters, self.MIN_COUNTERS), 256)
            tensor = torch.empty((partial + counters) // 4, dtype=torch.float32, device=device)
            tensor[partial // 4:].zero_()
            if old is not None and not capture:
                self._outgrown.append(old.tensor)
            bufs[key] = buf = _Buffer(tensor, partial, counters, capture)
            return buf

    def nbytes(self) -> int:
        """Bytes held, those of captures apart (they are the graphs' memory)."""
        return 4 * (sum(b.tensor.numel() for b in self._bufs.values()) + sum(t.numel() for t in self._outgrown))


def _capture_id(device: torch.device) -> int:
    """The id of the capture that the current stream takes part in, 0 outside one."""
    if device.type != "cuda" or not torch.cuda.is_current_stream_capturing():
        return 0
    got = c_uint64(0)
    _lib.check(_lib.load().ember_stream_capture_id(_stream_key(device), byref(got)), "ember_stream_capture_id")
    return got.value


def round_up(n: int, m: int) -> int:
    return (n + m - 1) // m * m
