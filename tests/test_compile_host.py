"""torch.compile traces the ops and layers the same way before and after the library is loaded:
the native host path is a C function that Dynamo cannot enter, so compiled code must not meet it."""

from __future__ import annotations

import pytest
import torch

from emberserve_amd import _lib, layers, ops

X, W = torch.randn(3, 8, generator=torch.Generator().manual_seed(1)), torch.ones(8)
Q, K = X.view(3, 2, 4), X.view(3, 2, 4)[:, :1]
POS, TAB = torch.arange(3), torch.randn(4, 4, generator=torch.Generator().manual_seed(2))
NORM = layers.RMSNorm(8, 1e-6)

CALLS = {
    "rmsnorm": lambda: ops.rmsnorm(X, W, 1e-6),
    "fused_add_rmsnorm": lambda: ops.fused_add_rmsnorm(X, X, W, 1e-6),
    "silu_and_mul": lambda: ops.silu_and_mul(X),
    "embedding": lambda: ops.embedding(POS, X),
    "rope": lambda: ops.rope(Q.clone(), K.clone(), TAB, TAB, POS),
    "qk_norm_rope": lambda: ops.qk_norm_rope(Q.clone(), K.clone(), W[:4], W[:4], 1e-6, TAB, TAB, POS),
    "mla_latent_rope": lambda: ops.mla_latent_rope(X, X[:, :4].clone(), Q.clone(), W, 1e-6, TAB, TAB, POS),
    "RMSNorm": lambda: NORM(X),
}


@pytest.mark.parametrize("name", sorted(CALLS))
def test_ops_compile_without_graph_breaks_once_loaded(name):
    _lib.load()
    torch._dynamo.reset()
    got = torch.compile(CALLS[name], backend="eager", fullgraph=True)()
    want = CALLS[name]()
    for g, w in zip(got if isinstance(got, tuple) else (got,), want if isinstance(want, tuple) else (want,)):
        assert torch.equal(g, w)
