"""The native host path (csrc/fast_ops.cpp) answers exactly the ordinary GPU calls: on the CPU
every function declines; on the GPU each is compared bit for bit, with its outputs' shapes and
strides, with the Python wrapper it stands in for, over the forms it accepts, and declines
the others (which the wrappers convert, refuse or run eagerly)."""

from __future__ import annotations

import ctypes
import os
import subprocess
import sys
from pathlib import Path

import pytest
import torch

from emberserve_amd import _lib, build, ops
from emberserve_amd.mla_decode import mla_decode
from emberserve_amd.paged_decode import paged_attention_decode
from emberserve_amd.rope import RotaryEmbedding
from oracle import inputs as gen

fast = _lib.fast


def _same(got, want, what):
    for g, w in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
        if w is None:
            assert g is None, what
            continue
        assert g.shape == w.shape and g.stride() == w.stride() and g.dtype == w.dtype and g.device == w.device, what
        assert not g.requires_grad, what
        assert torch.equal(g.view(torch.uint8) if g.is_contiguous() else g, w.view(torch.uint8) if w.is_contiguous() else w), what


def test_every_function_declines_cpu_tensors():
    _lib.load()
    x, w = torch.randn(3, 8), torch.randn(8)
    q, k = torch.randn(3, 2, 8), torch.randn(3, 1, 8)
    pos, tab = torch.zeros(3, dtype=torch.int64), torch.randn(4, 8)
    cache = torch.zeros(1, 16, 1, 8)
    assert fast.rmsnorm(x, w, 1e-6) is None and fast.add_rmsnorm(x, x, w, 1e-6) is None
    assert fast.silu_and_mul(x) is None and fast.embedding(pos, x) is None
    assert fast.rope(q, k, tab, tab, pos) is None and fast.qk_norm_rope(q, k, w, w, 1e-6, tab, tab, pos) is None
    assert fast.rope_kv_cache(q, k, k, tab, tab, pos, pos, cache, cache, None, None, 1e-6) is None
    assert fast.mla_latent_rope(x, x, q, w, 1e-6, tab, tab, pos) is None
    assert fast.mla_latent_rope_cache(x, x, q, w, 1e-6, tab, tab, pos, pos, cache[..., 0, :], True) is None
    assert fast.paged_decode(q, cache, cache, pos.int()[:, None], pos.int(), 1.0, None) is None
    assert fast.mla_decode(q, q, cache[..., 0, :], pos.int()[:, None], pos.int(), 1.0, None) is None
    assert fast.rmsnorm("x", None, 1e-6) is None and fast.rmsnorm(x) is None  # no tensors, no such arguments


def test_extension_is_imported_by_load():
    """A process may import the package before anything is built: the extension comes with load()."""
    code = ("import sys, emberserve_amd; from emberserve_amd import _lib\n"
            "assert 'emberserve_amd._fast' not in sys.modules and _lib.fast.rmsnorm(1) is None\n"
            "_lib.load(); assert 'rmsnorm' in vars(_lib.fast)")
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300)


def test_the_library_loads_without_the_extension(tmp_path):
    """A tree built without a host compiler: the package warns once and runs the Python wrappers."""
    pkg = tmp_path / "emberserve_amd"
    pkg.mkdir()
    for f in Path(_lib.__file__).parent.iterdir():
        if f.name not in ("_fast.so", "__pycache__"):
            (pkg / f.name).symlink_to(f)
    code = ("import warnings, torch; from emberserve_amd import _lib, ops\n"
            "with warnings.catch_warnings(record=True) as w:\n"
            "    warnings.simplefilter('always'); _lib.load(); _lib.load()\n"
            "assert ['native host path' in str(x.message) for x in w].count(True) == 1, w\n"
            "assert _lib.__file__.startswith(%r) and _lib.fast.rmsnorm(1) is None\n"
            "x = torch.randn(2, 8); assert torch.equal(ops.silu_and_mul(x), ops.silu_and_mul_torch(x))" % str(tmp_path))
    subprocess.run([sys.executable, "-c", code], check=True, timeout=300, cwd=tmp_path,
                   env={**os.environ, "PYTHONPATH": ""})


def test_build_without_a_compiler_leaves_no_extension(tmp_path, monkeypatch):
    monkeypatch.delenv("CXX", raising=False)
    monkeypatch.setattr(build.shutil, "which", lambda name: None)
    monkeypatch.setattr(build, "hipcc", lambda: "/opt/rocm/bin/hipcc")
    monkeypatch.setattr(build, "FAST_PATH", tmp_path / "_fast.so")
    (tmp_path / "_fast.so").write_bytes(b"stale")
    with pytest.warns(RuntimeWarning, match="compiler"):
        build._build_fast()
    assert not (tmp_path / "_fast.so").exists()


gpu = pytest.mark.gpu
DEV = "cuda"


def _rand(*shape, dtype=torch.bfloat16, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed)).to(dtype).to(DEV)


@gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_row_ops_equal_the_python_wrappers(dtype):
    for rows, h in ((1, 896), (5, 33), (3, 4096), (700, 64)):
        wide = _rand(rows, h + 8, dtype=dtype, seed=rows)
        for x in (wide[:, :h], wide[:, :h].contiguous(), wide[:, 1:h + 1], _rand(2, rows, h, dtype=dtype)):
            r = _rand(*x.shape, dtype=dtype, seed=9)
            for w in (_rand(h, dtype=dtype, seed=3), _rand(h, dtype=torch.float32, seed=3)):
                w = torch.nn.Parameter(w)
                _same(fast.rmsnorm(x, w, 1e-6), ops.rmsnorm_hip(x, w, 1e-6), "rmsnorm")
                _same(fast.add_rmsnorm(x, r, w, 1e-6), ops.fused_add_rmsnorm_hip(x, r, w, 1e-6), "add_rmsnorm")
            if h % 2 == 0:
                _same(fast.silu_and_mul(x), ops.silu_and_mul_hip(x), "silu")
    table = _rand(50, 72, dtype=dtype)
    for ids in (torch.tensor([3, 49, 0], device=DEV), torch.tensor([[1, 2], [3, 4]], device=DEV)):
        for t in (table, table[:, :64]):
            _same(fast.embedding(ids, t), ops.embedding_hip(ids, t), "embedding")


@gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("hq,hk,d", [(14, 2, 64), (32, 8, 128), (3, 1, 96)])
def test_head_ops_equal_the_python_wrappers(dtype, hq, hk, d):
    n = 37
    cos, sin = RotaryEmbedding(d, 512, 1e6).full_tables(torch.device("cuda", 0))
    pos = torch.randint(0, 512, (n,), generator=torch.Generator().manual_seed(1)).to(DEV)
    slots = torch.randperm(64, generator=torch.Generator().manual_seed(2))[:n].to(DEV)
    slots[5] = -1  # a padding row
    qw, kw = _rand(d, dtype=dtype, seed=4), _rand(d, dtype=dtype, seed=5)
    qkv = _rand(n, (hq + 2 * hk) * d, dtype=dtype)

    def parts():
        q, k, v = qkv.clone().split([hq * d, hk * d, hk * d], dim=-1)
        return q.view(n, hq, d), k.view(n, hk, d), v.view(n, hk, d)
    for norm in (False, True):
        a, b = parts(), parts()
        if norm:
            got = fast.qk_norm_rope(a[0], a[1], qw, kw, 1e-6, cos, sin, pos)
            want = ops.qk_norm_rope_hip(b[0], b[1], qw, kw, 1e-6, cos, sin, pos)
        else:
            got, want = fast.rope(a[0], a[1], cos, sin, pos), ops.rope_hip(b[0], b[1], cos, sin, pos)
        assert got[0] is a[0] and got[1] is a[1]
        _same(got, want, "rope")
        for padded in (0, 8):
            caches = [torch.zeros(4, 16, hk, d + padded, dtype=dtype, device=DEV)[..., :d] for _ in range(4)]
            a, b = parts(), parts()
            w = (qw, kw) if norm else (None, None)
            got = fast.rope_kv_cache(*a, cos, sin, pos, slots, caches[0], caches[1], *w, 1e-6)
            want = ops.rope_kv_cache_hip(*b, cos, sin, pos, slots, caches[2], caches[3], *w, 1e-6)
            if d == 96:  # heads that the fused kernel refuses: the wrappers run the unfused pair
                assert got is None
                got = ops.rope_kv_cache_hip(*a, cos, sin, pos, slots, caches[0], caches[1], *w, 1e-6)
            assert got[0] is a[0] and got[1] is a[1]
            _same(got, want, "rope_kv_cache")
            assert torch.equal(caches[0], caches[2]) and torch.equal(caches[1], caches[3])


@gpu
@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_mla_ops_equal_the_python_wrappers(dtype):
    n, heads, r, dr = 21, 16, 512, 64
    cos, sin = RotaryEmbedding(dr, 512, 5e4).full_tables(torch.device("cuda", 0))
    pos = torch.randint(0, 512, (n,), generator=torch.Generator().manual_seed(1)).to(DEV)
    slots = torch.randperm(32, generator=torch.Generator().manual_seed(2))[:n].to(DEV)
    w = _rand(r, dtype=dtype, seed=6)
    row = _rand(n, heads * 192 + r + dr, dtype=dtype)

    def parts():
        t = row.clone()
        return (t[:, heads * 192:heads * 192 + r], t[:, heads * 192 + r:],
                t[:, :heads * 192].view(n, heads, 192)[..., 128:])
    a, b = parts(), parts()
    got = fast.mla_latent_rope(*a, w, 1e-6, cos, sin, pos)
    assert got[0] is a[2]
    _same(got, ops.mla_latent_rope_hip(*b, w, 1e-6, cos, sin, pos), "mla_latent_rope")
    for keep in (True, False):
        c1, c2 = (torch.zeros(2, 16, r + dr, dtype=dtype, device=DEV) for _ in range(2))
        a, b = parts(), parts()
        _same(fast.mla_latent_rope_cache(*a, w, 1e-6, cos, sin, pos, slots, c1, keep),
              ops.mla_latent_rope_cache_hip(*b, w, 1e-6, cos, sin, pos, slots, c2, keep), "mla_latent_rope_cache")
        assert torch.equal(c1, c2)


@gpu
def test_decode_equals_the_python_wrapper(monkeypatch):
    """The wrapper runs when `out` is given; both at the default split count."""
    for ctx, hq, hkv, d, dtype in (([5, 700, 33], 32, 8, 128, torch.bfloat16), ([1] * 3, 14, 2, 64, torch.float16),
                                   ([40, 9], 4, 2, 64, torch.float32)):
        q, kc, vc, bt, cl = (t.to(DEV) for t in gen.decode_inputs(ctx, hq, hkv, d, 16, dtype, seed=d))
        want = paged_attention_decode(q, kc, vc, bt, cl, 0.1, out=torch.empty_like(q))
        calls = []
        real = fast.paged_decode
        monkeypatch.setattr(_lib, "fast", type("F", (), {"paged_decode": staticmethod(
            lambda *a: calls.append(real(*a)) or calls[-1])}))
        got = paged_attention_decode(q, kc, vc, bt, cl, 0.1)
        monkeypatch.undo()
        assert calls[0] is got  # the native path answered
        _same(got, want, "paged_decode")
    q, lat, bt, cl = (t.to(DEV) for t in gen.mla_decode_inputs([5, 700, 33], 16, 512, 64, 16, torch.bfloat16, seed=3))
    want = mla_decode(q, lat, bt, cl, 0.07, 512, out=torch.empty(3, 16, 512, dtype=q.dtype, device=DEV))
    real = fast.mla_decode
    for operand, what in ((q, "mla_decode"), ((q[..., :512].contiguous(), q[..., 512:].contiguous()), "pair")):
        calls = []
        monkeypatch.setattr(_lib, "fast", type("F", (), {"mla_decode": staticmethod(
            lambda *a: calls.append(real(*a)) or calls[-1])}))
        got = mla_decode(operand, lat, bt, cl, 0.07, 512)
        monkeypatch.undo()
        assert calls[0] is got
        _same(got, want, what)
    assert _lib.read_errors() == 0


@gpu
def test_other_calls_are_left_to_the_python_wrappers(monkeypatch):
    x, w = _rand(4, 64), _rand(64)
    assert fast.rmsnorm(x, w, 1e-6) is not None
    assert fast.rmsnorm(x.t(), _rand(4), 1e-6) is None              # needs a copy
    assert fast.rmsnorm(x, w.half(), 1e-6) is None                  # a weight to convert
    assert fast.rmsnorm(x, w[:32], 1e-6) is None                    # refused by the wrapper
    assert fast.rmsnorm(x, w.cpu(), 1e-6) is None
    assert fast.rmsnorm(x.long(), w, 1e-6) is None
    assert fast.rmsnorm(x[:0], w, 1e-6) is None
    assert fast.add_rmsnorm(x, x[:2], w, 1e-6) is None
    assert fast.silu_and_mul(x[:, :63]) is None
    assert fast.embedding(torch.tensor([1], dtype=torch.int32, device=DEV), x) is None

    class Sub(torch.Tensor):
        pass
    assert fast.rmsnorm(x.as_subclass(Sub), w, 1e-6) is None
    assert torch.equal(ops.rmsnorm(x.as_subclass(Sub), w, 1e-6).as_subclass(torch.Tensor), ops.rmsnorm_hip(x, w, 1e-6))
    for name, value in (("EMBERSERVE_FUSED_OPS", "0"), ("EMBERSERVE_CHECK_INDICES", "1")):
        monkeypatch.setenv(name, value)
        assert fast.rmsnorm(x, w, 1e-6) is None
        monkeypatch.delenv(name)
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    class Seen(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))
    with Seen():
        assert fast.rmsnorm(x, w, 1e-6) is None
    with TorchFunctionMode():
        assert fast.rmsnorm(x, w, 1e-6) is None
    seen = []
    torch.func.vmap(lambda t: seen.append(fast.rmsnorm(t, w, 1e-6)) or t)(x[None])
    assert seen == [None]
    with pytest.raises(ValueError):
        ops.rmsnorm(x, w[:32], 1e-6)


@gpu
def test_a_failed_launch_is_raised_and_not_run_again(monkeypatch):
    """EMBER_ELAUNCH can come with the kernel enqueued (an earlier, uncleared HIP error), so no
    wrapper may run the call a second time: in place, that would rotate q and k twice. The
    status is forced by stub entry points; nothing is launched."""
    from emberserve_amd import _fast
    lib, st = _lib.load(), 3
    real = {name: ctypes.cast(getattr(lib, name), ctypes.c_void_p).value for name in _lib.SIGNATURES}
    names = ("ember_rope", "ember_rope_kv_cache", "ember_rmsnorm", "ember_paged_decode_shared")
    stubs = [ctypes.CFUNCTYPE(ctypes.c_int, *_lib.SIGNATURES[n])(lambda *a: st) for n in names]
    again = []
    for name in ("rope_hip", "rope_kv_cache_hip", "rmsnorm_hip"):
        monkeypatch.setattr(ops, name, lambda *a, name=name: again.append(name))
    q, k, v = _rand(3, 4, 64), _rand(3, 2, 64, seed=1), _rand(3, 2, 64, seed=2)
    cos, sin = RotaryEmbedding(64, 16, 1e4).full_tables(q.device)
    pos = torch.arange(3, device=DEV)
    caches = [torch.zeros(1, 16, 2, 64, dtype=q.dtype, device=DEV) for _ in range(2)]
    dec = [t.to(DEV) for t in gen.decode_inputs([5, 7], 4, 2, 64, 16, torch.bfloat16, seed=1)]
    calls = {"rope": lambda: ops.rope(q, k, cos, sin, pos),
             "rope_kv_cache": lambda: ops.rope_kv_cache(q, k, v, cos, sin, pos, pos, *caches),
             "rmsnorm": lambda: ops.rmsnorm(q.view(3, -1), _rand(256), 1e-6),
             "paged_decode_shared": lambda: paged_attention_decode(*dec, 0.1)}
    _fast.bind({**real, **{n: ctypes.cast(s, ctypes.c_void_p).value for n, s in zip(names, stubs)}})
    try:
        for what, call in calls.items():
            with pytest.raises(RuntimeError, match=f"ember_{what} failed.*status 3"):
                call()
        st = 1  # refused before any launch: the wrappers' turn
        calls["rope"]()
        assert again == ["rope_hip"]
    finally:
        _fast.bind(real)


@gpu
def test_fast_calls_capture_and_follow_the_current_stream():
    x, w = _rand(64, 256), _rand(256)
    want = ops.rmsnorm_hip(x, w, 1e-6)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        got = fast.rmsnorm(x, w, 1e-6)
    s.synchronize()
    assert torch.equal(got, want)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        y, z = fast.add_rmsnorm(x, x, w, 1e-6)
    for seed in (1, 2, 3):
        x.copy_(_rand(64, 256, seed=seed))
        g.replay()
        _same((y, z), ops.fused_add_rmsnorm_hip(x, x, w, 1e-6), "replay")
