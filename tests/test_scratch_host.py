"""Host-side checks of the split-K workspaces (no GPU): one buffer per (shape, device, stream), one
for all shapes of paged decode, counters verified and re-zeroed when left non-zero, and the MLA decode error word
mapped to exceptions."""

from __future__ import annotations

import threading

import pytest
import torch

from emberserve_amd import _lib, _scratch, mla_decode, paged_decode


def test_two_streams_get_different_workspaces(monkeypatch):
    cache = _scratch.ScratchCache("t")
    stream = {"id": 1}
    monkeypatch.setattr(_scratch, "_stream_key", lambda device: stream["id"])
    dev = torch.device("cpu")
    a = cache.get((2, 4), lambda: 1024, dev)
    assert cache.get((2, 4), lambda: 1024, dev) is a  # same stream, same shape: reused
    stream["id"] = 2
    b = cache.get((2, 4), lambda: 1024, dev)
    assert b is not a and b.data_ptr() != a.data_ptr()
    assert len(cache) == 2
    assert not bool(a.any()) and not bool(b.any())  # zero-filled


def test_workspace_size_floor_and_invalid(monkeypatch):
    monkeypatch.setattr(_scratch, "_stream_key", lambda device: 0)
    cache = _scratch.ScratchCache("t", min_bytes=256)
    assert cache.get((1,), lambda: 16, torch.device("cpu")).numel() * 4 == 256
    with pytest.raises(ValueError):
        cache.get((2,), lambda: -1, torch.device("cpu"))


def test_verify_counters_rezeroes_and_raises():
    cache = _scratch.ScratchCache("t")
    buf = torch.zeros(64, dtype=torch.float32)
    cache.verify_counters(buf, 128, 192)  # all zero: passes
    buf.view(torch.int32)[40] = 3  # a counter left at 3 by an aborted launch
    buf[0] = 1.5  # partials outside the region are not counters
    with pytest.raises(RuntimeError, match="non-zero"):
        cache.verify_counters(buf, 128, 192)
    assert int(buf.view(torch.int32)[32:48].abs().sum()) == 0
    assert float(buf[0]) == 1.5
    cache.verify_counters(buf, 128, 192)


def test_mla_decode_error_word_mapping():
    mla_decode.raise_decode_errors(0)
    with pytest.raises(RuntimeError, match="handshake"):
        mla_decode.raise_decode_errors(_lib.ERR_SYNC)
    with pytest.raises(IndexError, match="block id"):
        mla_decode.raise_decode_errors(_lib.ERR_BLOCK_ID)
    with pytest.raises(IndexError, match="context length"):
        mla_decode.raise_decode_errors(_lib.ERR_DECODE_CTX | _lib.ERR_SYNC)


def test_round_up():
    assert _scratch.round_up(0, 16) == 0 and _scratch.round_up(17, 16) == 32 and _scratch.round_up(256, 256) == 256


@pytest.mark.parametrize("heads,kv_heads", [(32, 8), (28, 4)])
def test_paged_decode_workspaces_are_bounded_over_batch_sizes(monkeypatch, heads, kv_heads):
    """Every batch size and table width of a stream shares one workspace: all that is held stays
    under four times the largest call's need (a workspace per shape came to gigabytes)."""
    pd = paged_decode
    monkeypatch.setattr(_scratch, "_stream_key", lambda device: 0)
    monkeypatch.setattr(pd, "num_sms", lambda device: 256)
    monkeypatch.setattr(pd, "_SCRATCH", _scratch.SharedScratch("t"))
    need = _lib.load().ember_paged_decode_workspace_bytes
    q, largest = torch.empty(0), 0
    for width in (8192, 2048, 4096):
        for batch in range(1, 257):
            splits, ws = pd._plan(batch, heads, 128, kv_heads, width, q)
            if splits == 1:
                continue
            assert ws.numel() * 4 >= need(batch, heads, 128, splits)
            largest = max(largest, need(batch, heads, 128, splits))
    assert largest > 16 << 20 and pd._SCRATCH.nbytes() <= 4 * largest


def test_shared_workspace_growth(monkeypatch):
    """A request inside the parts leaves the buffer alone; an outgrown buffer is kept (a captured
    graph may hold its address), the counters start at zero, and threads and streams have buffers
    of their own."""
    stream = {"id": 1}
    monkeypatch.setattr(_scratch, "_stream_key", lambda device: stream["id"])
    s, dev = _scratch.SharedScratch("t"), torch.device("cpu")
    a = s.get(100, 16, dev)
    assert a.numel() * 4 == s.MIN_PARTIAL + s.MIN_COUNTERS and a.data_ptr() % 16 == 0
    assert s.get(s.MIN_PARTIAL, s.MIN_COUNTERS, dev) is a
    assert not bool(a[s.MIN_PARTIAL // 4:].view(torch.int32).any())
    b = s.get(s.MIN_PARTIAL + 1, 16, dev)
    assert b.numel() * 4 == 2 * s.MIN_PARTIAL + s.MIN_COUNTERS and s.get(1, 1, dev) is b
    c = s.get(1, s.MIN_COUNTERS + 1, dev)
    assert c.numel() * 4 == 2 * s.MIN_PARTIAL + 2 * s.MIN_COUNTERS
    assert [t.data_ptr() for t in s._outgrown] == [a.data_ptr(), b.data_ptr()]
    assert s.nbytes() == 4 * (a.numel() + b.numel() + c.numel())
    stream["id"] = 2
    assert s.get(1, 1, dev) is not c
    stream["id"], other = 1, []
    t = threading.Thread(target=lambda: other.append(s.get(1, 1, dev)))
    t.start()
    t.join()
    assert other[0] is not c and s.get(1, 1, dev) is c


def test_shared_workspace_under_capture(monkeypatch):
    """A capture uses the eager workspace where it is large enough, and otherwise one of its own,
    which later captures and eager calls do not get."""
    state = {"capture": 0}
    monkeypatch.setattr(_scratch, "_stream_key", lambda device: 0)
    monkeypatch.setattr(_scratch, "_capture_id", lambda device: state["capture"])
    s, dev = _scratch.SharedScratch("t"), torch.device("cpu")
    state["capture"] = 7
    a = s.get(100, 16, dev)
    assert s.get(200, 16, dev) is a  # the same capture: one zero fill recorded
    state["capture"] = 8
    b = s.get(100, 16, dev)
    assert b is not a
    state["capture"] = 0
    e = s.get(100, 16, dev)
    assert e is not b and s.nbytes() == 4 * e.numel()
    state["capture"] = 9
    assert s.get(100, 16, dev) is e
    assert s.get(s.MIN_PARTIAL + 1, 16, dev) is not e and s.get(100, 16, dev) is e
