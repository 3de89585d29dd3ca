"""The work a serving engine has this framework do, as timed cases: one decoder layer's row
ops (dense and MLA), paged and MLA decode attention, and the gate_up + silu_and_mul of the
dense MLP and of routed experts, each through the package's public entry points.

Shapes are those of the repository's benchmark and tests: Qwen2.5-0.5B / 7B and Qwen3-8B
(dense), Moonlight (MLA and routed experts). Sizes run from one decode token to an
8192-token prefill; context lengths and routing are ragged, as a batch of requests is.
"""

from __future__ import annotations

import math

import torch

from emberserve_amd import gate_up_silu as gus
from emberserve_amd import layers, mla_decode, moe, ops, paged_decode
from emberserve_amd.rope import RotaryEmbedding

DEV = "cuda"
BLOCK = 16          # tokens per paged-cache block
EPS = 1e-6

DENSE = {  # hidden, intermediate, q heads, kv heads, head dim, qk-norm, rope base
    "qwen2.5-0.5b": (896, 4864, 14, 2, 64, False, 1e6),
    "qwen2.5-7b": (3584, 18944, 28, 4, 128, False, 1e6),
    "qwen3-8b": (4096, 12288, 32, 8, 128, True, 1e6),
}
# Moonlight: hidden, heads, nope dim, rope dim, latent rank, rope base; routed experts
MLA_HIDDEN, MLA_HEADS, MLA_NOPE, MLA_ROPE, MLA_RANK, MLA_BASE = 2048, 16, 128, 64, 512, 5e4
MOE_HIDDEN, MOE_INTER, MOE_EXPERTS, MOE_TOPK = 2048, 1408, 64, 6
VOCAB = 151936
MAX_POS = 32768
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def listed():
    return [
        # one decode token through a small model's layer: launches and host latency only
        dict(name="layer_1", kind="layer", model="qwen2.5-0.5b", tokens=1, dtype="fp16"),
        # a mixed step (39 decode rows and a 300-token prompt) of a 7B layer
        dict(name="layer_339", kind="layer", model="qwen2.5-7b", tokens=339, dtype="fp16"),
        # the largest prefill step of a Qwen3-8B layer (qk-norm, 32 + 8 heads)
        dict(name="layer_8192", kind="layer", model="qwen3-8b", tokens=8192, dtype="bf16"),
        # the first MLA layer of an odd-sized prefill step: embedding, norm, latent split
        dict(name="mla_layer_5003", kind="mla_layer", tokens=5003, dtype="bf16"),
        # decode attention, a small model under light load
        dict(name="decode_32", kind="decode", model="qwen2.5-0.5b", batch=32, max_context=2048, dtype="fp16"),
        # decode attention, Qwen3-8B under full load with long, ragged contexts
        dict(name="decode_64", kind="decode", model="qwen3-8b", batch=64, max_context=8192, dtype="bf16"),
        # MLA decode of a medium batch
        dict(name="mla_decode_32", kind="mla_decode", batch=32, max_context=4096, dtype="bf16"),
        # a decode batch through the dense MLP's packed gate_up weight
        dict(name="mlp_16", kind="mlp", model="qwen2.5-7b", tokens=16, keep=True, dtype="bf16"),
        # a chunked-prefill or mixed step of ordinary size, both weight copies held
        dict(name="mlp_200", kind="mlp", model="qwen3-8b", tokens=200, keep=True, dtype="bf16"),
        # the largest prefill step with one copy of the weight (the packed one)
        dict(name="mlp_8192", kind="mlp", model="qwen3-8b", tokens=8192, keep=False, dtype="bf16"),
        # routed experts: a decode batch, and an odd-sized prefill step
        dict(name="moe_24", kind="moe", tokens=24, dtype="bf16"),
        dict(name="moe_4099", kind="moe", tokens=4099, dtype="bf16"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "mla_layer", "decode", "decode", "mla_decode", "mlp", "mlp", "moe", "moe"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    model = rng.choice(sorted(DENSE))
    if kind == "layer":
        return dict(kind=kind, model=model, tokens=_log(rng, 1, 8192), dtype=dtype)
    if kind == "mla_layer":
        return dict(kind=kind, tokens=_log(rng, 1, 8192), dtype=dtype)
    if kind == "decode":
        return dict(kind=kind, model=model, batch=_log(rng, 1, 128), max_context=BLOCK * _log(rng, 8, 512), dtype=dtype)
    if kind == "mla_decode":
        return dict(kind=kind, batch=_log(rng, 1, 256), max_context=BLOCK * _log(rng, 8, 512), dtype=dtype)
    if kind == "mlp":
        hidden, inter = DENSE[model][:2]
        most = min(8192, 8192 * 4096 * 12288 // (hidden * inter))
        return dict(kind=kind, model=model, tokens=_log(rng, 1, most), keep=rng.random() < 0.5, dtype=dtype)
    return dict(kind=kind, tokens=_log(rng, 1, 8192), dtype=dtype)


# ---- inputs ------------------------------------------------------------------------------

class _Rand:
    """Seeded draws on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed))

    def normal(self, shape, dtype, std=1.0, mean=0.0):
        t = torch.empty(shape, dtype=dtype, device=DEV)
        return t.normal_(mean, std, generator=self.g)

    def ints(self, n, lo, hi, dtype=torch.int64):
        return torch.randint(lo, hi, (n,), generator=self.g, device=DEV).to(dtype)

    def perm(self, n):
        return torch.randperm(n, generator=self.g, device=DEV)


def _layer_inputs(c, seed):
    r, dt, t = _Rand(seed), DTYPES[c["dtype"]], c["tokens"]
    hidden, inter, hq, hk, d, norm, base = DENSE[c["model"]]
    slots_n = -(-t // BLOCK) * BLOCK + 4 * BLOCK
    return dict(
        x=r.normal((t, hidden), dt), residual=r.normal((t, hidden), dt), attn=r.normal((t, hidden), dt),
        qkv=r.normal((t, (hq + 2 * hk) * d), dt), gate_up=r.normal((t, 2 * inter), dt, std=2.0),
        w1=r.normal((hidden,), dt, std=0.1, mean=1.0), w2=r.normal((hidden,), dt, std=0.1, mean=1.0),
        qw=r.normal((d,), dt, std=0.1, mean=1.0) if norm else None,
        kw=r.normal((d,), dt, std=0.1, mean=1.0) if norm else None,
        positions=r.ints(t, 0, MAX_POS), slots=r.perm(slots_n)[:t].contiguous(),
        k_cache=torch.zeros(slots_n // BLOCK, BLOCK, hk, d, dtype=dt, device=DEV),
        v_cache=torch.zeros(slots_n // BLOCK, BLOCK, hk, d, dtype=dt, device=DEV),
        rotary=_rotary(d, base))


def _mla_layer_inputs(c, seed):
    r, dt, t = _Rand(seed), DTYPES[c["dtype"]], c["tokens"]
    slots_n = -(-t // BLOCK) * BLOCK + 4 * BLOCK
    width = MLA_HEADS * (MLA_NOPE + MLA_ROPE) + MLA_RANK + MLA_ROPE
    return dict(
        ids=r.ints(t, 0, VOCAB), table=r.normal((VOCAB, MLA_HIDDEN), dt, std=0.02),
        w1=r.normal((MLA_HIDDEN,), dt, std=0.1, mean=1.0), qkv_a=r.normal((t, width), dt),
        w_latent=r.normal((MLA_RANK,), dt, std=0.1, mean=1.0),
        positions=r.ints(t, 0, MAX_POS), slots=r.perm(slots_n)[:t].contiguous(),
        cache=torch.zeros(slots_n // BLOCK, BLOCK, MLA_RANK + MLA_ROPE, dtype=dt, device=DEV),
        rotary=_rotary(MLA_ROPE, MLA_BASE))


def _rotary(d, base):
    rotary = RotaryEmbedding(d, MAX_POS, base)
    rotary.full_tables(torch.device(DEV, torch.cuda.current_device()))
    return rotary


def _contexts(r, batch, max_context):
    """Ragged lengths, uniform in [1, max_context]: of a batch of requests at any point of
    their lives. Block tables over a shuffled pool, padded with block 0."""
    ctx = r.ints(batch, 1, max_context + 1, torch.int32)
    width = max_context // BLOCK
    blocks = batch * width
    tables = r.perm(blocks).view(batch, width).to(torch.int32)
    used = torch.arange(width, device=DEV)[None, :] * BLOCK < ctx[:, None]
    return ctx, torch.where(used, tables, torch.zeros_like(tables)).contiguous(), blocks


def _decode_inputs(c, seed):
    r, dt = _Rand(seed), DTYPES[c["dtype"]]
    _, _, hq, hk, d, _, _ = DENSE[c["model"]]
    ctx, tables, blocks = _contexts(r, c["batch"], c["max_context"])
    return dict(q=r.normal((c["batch"], hq, d), dt), ctx=ctx, tables=tables, scale=d ** -0.5,
                k_cache=r.normal((blocks, BLOCK, hk, d), dt), v_cache=r.normal((blocks, BLOCK, hk, d), dt))


def _mla_decode_inputs(c, seed):
    r, dt = _Rand(seed), DTYPES[c["dtype"]]
    ctx, tables, blocks = _contexts(r, c["batch"], c["max_context"])
    return dict(q_c=r.normal((c["batch"], MLA_HEADS, MLA_RANK), dt, std=0.5),
                q_pe=r.normal((c["batch"], MLA_HEADS, MLA_ROPE), dt), ctx=ctx, tables=tables,
                scale=(MLA_NOPE + MLA_ROPE) ** -0.5, cache=r.normal((blocks, BLOCK, MLA_RANK + MLA_ROPE), dt))


def _mlp_inputs(c, seed):
    r, dt = _Rand(seed), DTYPES[c["dtype"]]
    hidden, inter = DENSE[c["model"]][:2]
    return dict(x=r.normal((c["tokens"], hidden), dt), w=r.normal((2 * inter, hidden), dt, std=1.5 / hidden ** 0.5))


def _moe_inputs(c, seed):
    r, dt = _Rand(seed), DTYPES[c["dtype"]]
    x = r.normal((c["tokens"], MOE_HIDDEN), dt)
    w = r.normal((MOE_EXPERTS, 2 * MOE_INTER, MOE_HIDDEN), dt, std=1.5 / MOE_HIDDEN ** 0.5)
    # a trained router favours some experts: a bias beside each token's own logits
    logits = r.normal((c["tokens"], MOE_EXPERTS), torch.float32) + r.normal((MOE_EXPERTS,), torch.float32, std=0.3)
    return dict(x=x, w=w, ids=torch.topk(logits, MOE_TOPK, dim=-1).indices.contiguous())


_INPUTS = dict(layer=_layer_inputs, mla_layer=_mla_layer_inputs, decode=_decode_inputs,
               mla_decode=_mla_decode_inputs, mlp=_mlp_inputs, moe=_moe_inputs)


def prepare(case, seed):
    s = _INPUTS[case["kind"]](case, seed)
    s["case"] = case
    if case["kind"] == "mlp":  # weights are packed once, when a model is loaded
        s["packed"] = gus.pack_gate_up_weight(s["w"])
        if not case["keep"]:
            s["w"] = None
    elif case["kind"] == "moe":
        s["packed"] = moe.pack_moe_gate_up_weight(s["w"])
    elif case["kind"] == "layer":
        hidden = s["w1"].numel()
        s["norms"] = [_norm(s[k], hidden) for k in ("w1", "w2")]
    elif case["kind"] == "mla_layer":
        s["embed"] = layers.Embedding(VOCAB, MLA_HIDDEN, _weight=s["table"])
        s["embed"].requires_grad_(False)
        s["norm"] = _norm(s["w1"], MLA_HIDDEN)
    return s


def _norm(weight, hidden):
    m = layers.RMSNorm(hidden, EPS)
    m.weight = torch.nn.Parameter(weight, requires_grad=False)
    return m


# ---- one pass ----------------------------------------------------------------------------

def _run_layer(s):
    hq, hk, d = DENSE[s["case"]["model"]][2:5]
    qkv = s["qkv"]
    n = qkv.shape[0]
    normed, residual = s["norms"][0].forward_with_residual(s["x"], s["residual"])
    q, k, v = qkv.split([hq * d, hk * d, hk * d], dim=-1)
    cos, sin = s["rotary"].full_tables(qkv.device)
    q, k = ops.rope_kv_cache(q.view(n, hq, d), k.view(n, hk, d), v.view(n, hk, d), cos, sin, s["positions"],
                             s["slots"], s["k_cache"], s["v_cache"], s["qw"], s["kw"], EPS)
    normed2, residual2 = s["norms"][1].forward_with_residual(s["attn"], residual)
    act = ops.silu_and_mul(s["gate_up"])
    return dict(normed=normed, residual=residual, q=q, k=k, k_cache=s["k_cache"], v_cache=s["v_cache"],
                normed2=normed2, residual2=residual2, act=act)


def _run_mla_layer(s):
    qkv_a = s["qkv_a"]
    n = qkv_a.shape[0]
    hidden = s["embed"](s["ids"])
    normed = s["norm"](hidden)
    q, ckv = qkv_a.split([MLA_HEADS * (MLA_NOPE + MLA_ROPE), MLA_RANK + MLA_ROPE], dim=-1)
    q_pe = q.view(n, MLA_HEADS, MLA_NOPE + MLA_ROPE)[..., MLA_NOPE:]
    c, k_pe = ckv.split([MLA_RANK, MLA_ROPE], dim=-1)
    cos, sin = s["rotary"].full_tables(qkv_a.device)
    q_pe, latent = ops.mla_latent_rope_cache(c, k_pe, q_pe, s["w_latent"], EPS, cos, sin, s["positions"],
                                             s["slots"], s["cache"])
    return dict(hidden=hidden, normed=normed, q_pe=q_pe, latent=latent, cache=s["cache"])


def run(state):
    kind = state["case"]["kind"]
    if kind == "layer":
        return _run_layer(state)
    if kind == "mla_layer":
        return _run_mla_layer(state)
    if kind == "decode":
        return paged_decode.paged_attention_decode(state["q"], state["k_cache"], state["v_cache"], state["tables"],
                                                   state["ctx"], state["scale"])
    if kind == "mla_decode":
        return mla_decode.mla_decode((state["q_c"], state["q_pe"]), state["cache"], state["tables"], state["ctx"],
                                     state["scale"], MLA_RANK)
    if kind == "mlp":
        return gus.gate_up_silu(state["x"], state["w"], packed=state["packed"])
    return moe.fused_moe_gate_up(state["x"], state["ids"], state["w"], packed=state["packed"])


# ---- what a pass cannot do without ---------------------------------------------------------

def work(case):
    e, kind = 2, case["kind"]
    if kind == "layer":
        hidden, inter, hq, hk, d, _, _ = DENSE[case["model"]]
        t = case["tokens"]
        norms = 2 * (4 * t * hidden + hidden) * e
        rope = (2 * t * (hq + hk) * d + t * hk * d + 2 * t * hk * d) * e + 16 * t
        return {"bytes": norms + rope + 3 * t * inter * e, "flops": 0}
    if kind == "mla_layer":
        t, lat = case["tokens"], MLA_RANK + MLA_ROPE
        embed = t * (8 + 2 * MLA_HIDDEN * e)
        norm = 2 * t * MLA_HIDDEN * e
        split = t * (3 * lat + 2 * MLA_HEADS * MLA_ROPE) * e + 16 * t
        return {"bytes": embed + norm + split, "flops": 0}
    if kind in ("decode", "mla_decode"):
        keys = case["batch"] * (case["max_context"] + 1) / 2  # expected
        if kind == "decode":
            _, _, hq, hk, d, _, _ = DENSE[case["model"]]
            return {"bytes": (keys * 2 * hk * d + 2 * case["batch"] * hq * d) * e, "flops": 4 * keys * hq * d}
        lat = MLA_RANK + MLA_ROPE
        return {"bytes": (keys * lat + case["batch"] * MLA_HEADS * (lat + MLA_RANK)) * e,
                "flops": 2 * keys * MLA_HEADS * (lat + MLA_RANK)}
    if kind == "mlp":
        hidden, inter = DENSE[case["model"]][:2]
        t = case["tokens"]
        return {"bytes": (2 * inter * hidden + t * hidden + t * inter) * e, "flops": 4 * t * hidden * inter}
    t = case["tokens"]
    experts = MOE_EXPERTS * (1 - (1 - MOE_TOPK / MOE_EXPERTS) ** t)  # expected
    return {"bytes": (experts * 2 * MOE_INTER * MOE_HIDDEN + t * MOE_HIDDEN + t * MOE_TOPK * MOE_INTER) * e,
            "flops": 4 * t * MOE_TOPK * MOE_HIDDEN * MOE_INTER}


def tolerance(case):
    # four times the largest distance of a pass from its 64-bit value, which is the rounding
    # of results (and of the projections before silu) to the storage type
    bf = case["dtype"] == "bf16"
    if case["kind"] in ("mlp", "moe"):
        return {"rel": 1.5e-2 if bf else 2e-3}
    return {"rel": 1.3e-2 if bf else 1.7e-3}


# ---- the same in 64 bits, in plain torch ---------------------------------------------------

def _rms64(x, w):
    return x / torch.sqrt(x.pow(2).mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, positions, d, base):
    inv = base ** (-torch.arange(0, d, 2, dtype=torch.float64, device=DEV) / d)
    a = positions.double()[:, None, None] * inv
    lo, hi = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def _put64(cache, slots, rows):
    out = torch.zeros(cache.shape, dtype=torch.float64, device=DEV)
    out.view(-1, *rows.shape[1:])[slots] = rows
    return out


def _exact_layer(c, seed):
    s = _layer_inputs(c, seed)
    _, _, hq, hk, d, norm, base = DENSE[c["model"]]
    n = c["tokens"]
    residual = s["x"].double() + s["residual"].double()
    residual2 = residual + s["attn"].double()
    q, k, v = s["qkv"].double().split([hq * d, hk * d, hk * d], -1)
    q, k, v = q.view(n, hq, d), k.view(n, hk, d), v.view(n, hk, d)
    if norm:
        q, k = _rms64(q, s["qw"]), _rms64(k, s["kw"])
    q, k = _rope64(q, s["positions"], d, base), _rope64(k, s["positions"], d, base)
    g, u = s["gate_up"].double().chunk(2, -1)
    return dict(normed=_rms64(residual, s["w1"]), residual=residual, q=q, k=k,
                k_cache=_put64(s["k_cache"], s["slots"], k), v_cache=_put64(s["v_cache"], s["slots"], v),
                normed2=_rms64(residual2, s["w2"]), residual2=residual2, act=g * torch.sigmoid(g) * u)


def _exact_mla_layer(c, seed):
    s = _mla_layer_inputs(c, seed)
    n = c["tokens"]
    hidden = s["table"][s["ids"]].double()
    q, lat, k_pe = s["qkv_a"].double().split([MLA_HEADS * (MLA_NOPE + MLA_ROPE), MLA_RANK, MLA_ROPE], -1)
    q_pe = q.view(n, MLA_HEADS, MLA_NOPE + MLA_ROPE)[..., MLA_NOPE:]
    q_pe = _rope64(q_pe, s["positions"], MLA_ROPE, MLA_BASE)
    k_pe = _rope64(k_pe[:, None], s["positions"], MLA_ROPE, MLA_BASE)[:, 0]
    latent = torch.cat([_rms64(lat, s["w_latent"]), k_pe], -1)
    return dict(hidden=hidden, normed=_rms64(hidden, s["w1"]), q_pe=q_pe, latent=latent,
                cache=_put64(s["cache"], s["slots"], latent))


def _exact_decode(c, seed):
    s = _decode_inputs(c, seed)
    _, _, hq, hk, d, _, _ = DENSE[c["model"]]
    out = torch.empty(c["batch"], hq, d, dtype=torch.float64, device=DEV)
    for b, n in enumerate(s["ctx"].tolist()):
        rows = s["tables"][b, : -(-n // BLOCK)].long()
        k = s["k_cache"][rows].view(-1, hk, d)[:n].double()
        v = s["v_cache"][rows].view(-1, hk, d)[:n].double()
        for h in range(hk):
            qh = s["q"][b, h * (hq // hk): (h + 1) * (hq // hk)].double()
            p = torch.softmax(qh @ k[:, h].t().contiguous() * s["scale"], -1)
            out[b, h * (hq // hk): (h + 1) * (hq // hk)] = p @ v[:, h].contiguous()
    return out


def _exact_mla_decode(c, seed):
    s = _mla_decode_inputs(c, seed)
    out = torch.empty(c["batch"], MLA_HEADS, MLA_RANK, dtype=torch.float64, device=DEV)
    for b, n in enumerate(s["ctx"].tolist()):
        rows = s["cache"][s["tables"][b, : -(-n // BLOCK)].long()].view(-1, MLA_RANK + MLA_ROPE)[:n].double()
        q = torch.cat([s["q_c"][b], s["q_pe"][b]], -1).double()
        out[b] = torch.softmax(q @ rows.t().contiguous() * s["scale"], -1) @ rows[:, :MLA_RANK].contiguous()
    return out


def _act64(x, w):
    g, u = (x @ w.double().t().contiguous()).chunk(2, -1)
    return g * torch.sigmoid(g) * u


def _exact_mlp(c, seed):
    s = _mlp_inputs(c, seed)
    return _act64(s["x"].double(), s["w"])


def _exact_moe(c, seed):
    s = _moe_inputs(c, seed)
    flat = s["ids"].view(-1)
    out = torch.empty(flat.numel(), MOE_INTER, dtype=torch.float64, device=DEV)
    for e in range(MOE_EXPERTS):
        mine = (flat == e).nonzero().view(-1)
        if mine.numel():
            out[mine] = _act64(s["x"][mine // MOE_TOPK].double(), s["w"][e])
    return out


_EXACT = dict(layer=_exact_layer, mla_layer=_exact_mla_layer, decode=_exact_decode,
              mla_decode=_exact_mla_decode, mlp=_exact_mlp, moe=_exact_moe)


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)
