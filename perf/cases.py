"""What this framework is timed on: calls that an encoder engine makes through
``inl_hip``, from one short query to a batch of long documents.

Two kinds of case. Layer calls: packed attention in the forms the engines use
(causal GQA, sliding window, ModernBERT's local band, f32), the q/k
prologue, the GEGLU MLP, the SPLADE head and the gated-delta-net layer. Whole
encodes: token ids in, unit vectors out, for the Qwen3 and EmbeddingGemma 2
runners. A case is a dict of plain values; ``exact`` computes the same outputs
in float64 with plain torch.
"""
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.getcwd(), "im-not-llm_amd")
if _PKG not in sys.path:
    sys.path.insert(1, _PKG)

import inl_hip  # noqa: E402

_BF16, _F32, _F64 = torch.bfloat16, torch.float32, torch.float64

# (query heads, K/V heads, head_dim, causal, window radius, scale)
FORMS = {
    "qwen3": (16, 8, 128, True, -1, 128 ** -0.5),
    "late": (16, 2, 256, True, -1, 256 ** -0.5),
    "gemma_window": (3, 1, 256, False, 512, 1.0),
    "gemma_full": (3, 1, 256, False, -1, 1.0),
    "modernbert_local": (12, 12, 64, False, 64, 64 ** -0.5),
    "modernbert_global": (12, 12, 64, False, -1, 64 ** -0.5),
    "vision": (16, 16, 64, False, -1, 1.0),
}
SPLADE_VOCAB, SPLADE_HIDDEN, SPLADE_TERMS = 50002, 768, 36282
GDN_HEADS, GDN_DIM, GDN_TAPS = 16, 128, 4
GEMMA_LAYERS, GEMMA_HIDDEN, GEMMA_FF, GEMMA_PLE, GEMMA_VOCAB = 24, 768, 1152, 256, 262144
QWEN = dict(vocab=151669, hidden=1024, intermediate=3072, layers=28, heads=16, kv_heads=8, head_dim=128,
            eps=1e-6, theta=1e6)


def listed():
    return [
        # One search query's attention layer by itself, schedule and all:
        # nothing but latency, the smallest call there is.
        dict(name="attn_one_query", kind="attn", form="qwen3", dtype="bf16", plan=False,
             texts=1, lo=23, hi=23, lens=0),
        # An indexing batch of passages: log-normal lengths, 64 texts (a
        # twelfth of the benchmark's 200k-token configuration 2), the schedule
        # kept for the layers of the encode.
        dict(name="attn_passages", kind="attn", form="qwen3", dtype="bf16", plan=True,
             texts=64, median=180.0, sigma=1.0, most=2048, lens=0),
        # Documents through an EmbeddingGemma sliding layer.
        dict(name="attn_window_docs", kind="attn", form="gemma_window", dtype="bf16", plan=True,
             texts=8, lo=64, hi=8192, lens=0),
        # A sparse engine's batch through a ModernBERT local layer (two in three).
        dict(name="attn_local_band", kind="attn", form="modernbert_local", dtype="bf16", plan=True,
             texts=32, lo=32, hi=2048, lens=0),
        # The f32 mode (the reference's own precision) on a batch of passages.
        dict(name="attn_passages_f32", kind="attn", form="qwen3", dtype="f32", plan=True,
             texts=32, median=180.0, sigma=1.0, most=2048, lens=1),
        # q/k norms and RoPE of the same 64 passages, on the fused projection row.
        dict(name="prologue_passages", kind="prologue", dtype="bf16",
             texts=64, median=180.0, sigma=1.0, most=2048, lens=0),
        # An EmbeddingGemma MLP over a batch of documents, ragged row count.
        dict(name="mlp_docs", kind="mlp", rows=20011, hidden=768, ff=1152),
        # The sparse engine's decoder, per-text maxima, finish and fold.
        dict(name="splade_head", kind="splade", texts=16, lo=32, hi=2048, lens=0),
        # The late engine's linear-attention layer over a batch of passages.
        dict(name="delta_layer", kind="gdn", dtype="bf16", texts=16, median=512.0, sigma=0.8, most=4096, lens=0),
        # One search query through the whole bf16 embedder.
        dict(name="encode_query", kind="qwen3", dtype="bf16", texts=1, lo=17, hi=17, lens=0),
        # Configuration 1: 8 texts of U[16, 256] tokens through the f32 embedder.
        dict(name="encode_batch_f32", kind="qwen3", dtype="f32", texts=8, lo=16, hi=256, lens=0),
        # Documents through the whole EmbeddingGemma 2 tower (configuration 3
        # with fewer texts).
        dict(name="encode_docs", kind="gemma", texts=6, lo=64, hi=8192, lens=0),
    ]


def draw(rng):
    """One more case: the same kinds, sizes over the whole range."""
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    def lengths_of(most_tokens, texts, median_lo, median_hi, most):
        # at most `most_tokens` tokens for certain: every length is under `most`
        n = log_int(1, texts)
        cap = max(1, min(most, most_tokens // n))
        return dict(texts=n, median=float(min(cap, log_int(median_lo, median_hi))),
                    sigma=rng.choice([0.0, 0.5, 1.0]), most=cap, lens=rng.randrange(1 << 30))

    kind = rng.choice(["attn", "attn", "attn", "prologue", "mlp", "splade", "gdn", "qwen3", "qwen3", "gemma"])
    if kind == "attn":
        form = rng.choice(sorted(FORMS))
        dtype = rng.choice(["bf16", "bf16", "bf16", "f32"])
        # quadratic forms at long texts: bounded so that no draw is over the
        # work of the largest listed case
        tokens = 8192 if dtype == "f32" else 32768
        return dict(kind="attn", form=form, dtype=dtype, plan=rng.random() < 0.7,
                    **lengths_of(tokens, 128, 12, 4096, 2048 if dtype == "f32" else 8192))
    if kind == "prologue":
        return dict(kind="prologue", dtype=rng.choice(["bf16", "bf16", "f32"]),
                    **lengths_of(32768, 128, 12, 2048, 8192))
    if kind == "mlp":
        hidden, ff = rng.choice([(768, 1152), (1024, 3072)])
        return dict(kind="mlp", rows=log_int(1, 32768), hidden=hidden, ff=ff)
    if kind == "splade":
        return dict(kind="splade", **lengths_of(16384, 64, 12, 1024, 2048))
    if kind == "gdn":
        return dict(kind="gdn", dtype=rng.choice(["bf16", "bf16", "f32"]), **lengths_of(12288, 32, 12, 2048, 4096))
    if kind == "qwen3":
        dtype = rng.choice(["bf16", "f32"])
        return dict(kind="qwen3", dtype=dtype, **lengths_of(1024, 32, 8, 256, 512))
    return dict(kind="gemma", **lengths_of(16384, 32, 64, 2048, 8192))


# --------------------------------------------------------------------------
# Inputs
# --------------------------------------------------------------------------

def _lengths(case):
    rng = np.random.default_rng(case["lens"])
    if "lo" in case:
        return [int(t) for t in rng.integers(case["lo"], case["hi"] + 1, size=case["texts"])]
    t = np.round(rng.lognormal(math.log(case["median"]), case["sigma"], size=case["texts"]))
    return [int(x) for x in np.clip(t, 1, case["most"])]


def _cu(lengths):
    return [0] + [int(x) for x in np.cumsum(lengths)]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _dt(case):
    return _BF16 if case["dtype"] == "bf16" else _F32


def _attn_inputs(case, seed):
    """q, k, v as slices of one fused projection row, as the runners hold
    them: q and k after a per-head RMSNorm with weights in [0.9, 1.1]."""
    hq, hkv, d, _, _, scale = FORMS[case["form"]]
    g, n = _gen(seed), sum(_lengths(case))
    x = torch.randn(n, hq + 2 * hkv, d, generator=g, device="cuda")
    w = 1.0 + 0.2 * (torch.rand(hq + 2 * hkv, d, generator=g, device="cuda") - 0.5)
    x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w
    x[:, :hq] *= d ** -0.5 / scale
    x = x.to(_dt(case))
    return x[:, :hq], x[:, hq:hq + hkv], x[:, hq + hkv:]


def _prologue_inputs(case, seed):
    g, lens = _gen(seed), _lengths(case)
    x = (torch.randn(sum(lens), 32, 128, generator=g, device="cuda") * 1.5).to(_dt(case))
    qw, kw = ((1.0 + 0.2 * (torch.rand(128, generator=g, device="cuda") - 0.5)).to(_dt(case)) for _ in range(2))
    rows = torch.from_numpy(np.concatenate([np.arange(t) for t in lens]).astype(np.int32)).cuda()
    inv = 1e6 ** (-np.arange(0, 128, 2) / 128.0)
    ang = np.arange(max(lens))[:, None] * inv[None, :]
    cos, sin = (torch.from_numpy(f(ang).astype(np.float32)).cuda() for f in (np.cos, np.sin))
    return x, qw, kw, rows, cos, sin


def _mlp_inputs(case, seed):
    g, h, f = _gen(seed), case["hidden"], case["ff"]
    x = torch.randn(case["rows"], h, generator=g, device="cuda").to(_BF16)
    gu = (torch.randn(2 * f, h, generator=g, device="cuda") * h ** -0.5).to(_BF16)
    down = (torch.randn(h, f, generator=g, device="cuda") * f ** -0.5).to(_BF16)
    return x, gu, down


def _splade_inputs(case, seed):
    g, lens = _gen(seed), _lengths(case)
    head = torch.randn(sum(lens), SPLADE_HIDDEN, generator=g, device="cuda").to(_BF16)
    w = (torch.randn(SPLADE_VOCAB, SPLADE_HIDDEN, generator=g, device="cuda") * (4.0 / SPLADE_HIDDEN ** 0.5)).to(_BF16)
    bias = torch.randn(SPLADE_VOCAB, generator=g, device="cuda")
    perm = torch.randperm(SPLADE_TERMS, generator=g, device="cuda")
    more = torch.randint(0, SPLADE_TERMS, (SPLADE_VOCAB - SPLADE_TERMS,), generator=g, device="cuda")
    return head, w, bias, torch.cat([perm, more]).to(torch.int32)


def _gdn_inputs(case, seed):
    g, n, dt = _gen(seed), sum(_lengths(case)), _dt(case)
    H, D = GDN_HEADS, GDN_DIM
    rand = lambda *s: torch.randn(*s, generator=g, device="cuda")
    proj = rand(n, 3 * H * D).to(dt)
    taps = (rand(3 * H * D, GDN_TAPS) * 0.5).to(dt)
    a, b = (rand(n, H) * 0.5).to(dt), rand(n, H).to(dt)
    # decay rates as such layers are initialised: A in [1, 16], step in [0.001, 0.1]
    step = torch.exp(torch.rand(H, generator=g, device="cuda") * math.log(100.0) + math.log(1e-3))
    dt_bias = torch.log(torch.expm1(step))
    neg_a = -(1.0 + 15.0 * torch.rand(H, generator=g, device="cuda"))
    z = rand(n, H, D).to(dt)
    w = (1.0 + 0.2 * (torch.rand(D, generator=g, device="cuda") - 0.5)).to(dt)
    return proj, taps, a, b, dt_bias, neg_a, z, w


def _qwen3_inputs(case, seed):
    """Weights drawn as this repository's random-init encoder draws them:
    matrices u * 2 / sqrt(fan_in), norm weights 1 + 0.2 u, u in [-0.5, 0.5)."""
    g, dt, c = _gen(seed), _dt(case), QWEN

    def mat(rows, cols):
        return ((torch.rand(rows, cols, generator=g, device="cuda") - 0.5) * (2 / cols ** 0.5)).to(dt)

    def norm(dim):
        return (1 + 0.2 * (torch.rand(dim, generator=g, device="cuda") - 0.5)).to(dt)

    hs, ff = c["hidden"], c["intermediate"]
    qd, kvd = c["heads"] * c["head_dim"], c["kv_heads"] * c["head_dim"]
    W = {"embed_tokens.weight": mat(c["vocab"], hs), "norm.weight": norm(hs)}
    for i in range(c["layers"]):
        p = f"layers.{i}."
        W.update({p + "self_attn.q_proj.weight": mat(qd, hs), p + "self_attn.k_proj.weight": mat(kvd, hs),
                  p + "self_attn.v_proj.weight": mat(kvd, hs), p + "self_attn.o_proj.weight": mat(hs, qd),
                  p + "self_attn.q_norm.weight": norm(c["head_dim"]),
                  p + "self_attn.k_norm.weight": norm(c["head_dim"]),
                  p + "mlp.gate_proj.weight": mat(ff, hs), p + "mlp.up_proj.weight": mat(ff, hs),
                  p + "mlp.down_proj.weight": mat(hs, ff), p + "input_layernorm.weight": norm(hs),
                  p + "post_attention_layernorm.weight": norm(hs)})
    ids = np.random.default_rng(seed).integers(0, c["vocab"], size=sum(_lengths(case))).astype(np.int32)
    return W, ids


def _gemma_config():
    return {
        "vocab_size": GEMMA_VOCAB, "hidden_size": GEMMA_HIDDEN, "intermediate_size": GEMMA_FF,
        "num_hidden_layers": GEMMA_LAYERS, "num_attention_heads": 3, "num_key_value_heads": 1, "head_dim": 256,
        "rms_norm_eps": 1e-6, "sliding_window": 512,
        "layer_types": ["full_attention" if (i + 1) % 6 == 0 else "sliding_attention" for i in range(GEMMA_LAYERS)],
        "hidden_size_per_layer_input": GEMMA_PLE, "embedding_dim": 768,
        "rope_parameters": {"sliding_attention": {"rope_theta": 1e4}, "full_attention": {"rope_theta": 1e6}},
        "per_layer_config": {}, "max_position_embeddings": 8192,
    }


def _gemma_inputs(case, seed):
    """Projections N(0, 1/fan_in), norm weights near 1 (q/k norms near 0.25:
    the attention is unscaled), embeddings N(0, 0.05^2)."""
    g = _gen(seed)
    mat = lambda r, c: (torch.randn(r, c, generator=g, device="cuda") * c ** -0.5).to(_BF16)
    norm = lambda d, s=1.0: (s * (1 + 0.05 * torch.randn(d, generator=g, device="cuda"))).to(_BF16)
    hs, ff, ple, L = GEMMA_HIDDEN, GEMMA_FF, GEMMA_PLE, GEMMA_LAYERS
    W = {"embed_tokens.weight": (torch.randn(GEMMA_VOCAB, hs, generator=g, device="cuda") * 0.05).to(_BF16),
         "ple.per_layer_model_projection.weight": mat(L * ple, hs),
         "ple.per_layer_projection_norm.weight": norm(ple), "norm.weight": norm(hs),
         "embedding_projection.weight": mat(768, hs)}
    for i in range(L):
        p = f"layers.{i}."
        W.update({p + "self_attn.q_proj.weight": mat(768, hs), p + "self_attn.k_proj.weight": mat(256, hs),
                  p + "self_attn.v_proj.weight": mat(256, hs), p + "self_attn.o_proj.weight": mat(hs, 768),
                  p + "self_attn.q_norm.weight": norm(256, 0.25), p + "self_attn.k_norm.weight": norm(256, 0.25),
                  p + "input_layernorm.weight": norm(hs), p + "post_attention_layernorm.weight": norm(hs),
                  p + "pre_feedforward_layernorm.weight": norm(hs), p + "post_feedforward_layernorm.weight": norm(hs),
                  p + "mlp.gate_proj.weight": mat(ff, hs), p + "mlp.up_proj.weight": mat(ff, hs),
                  p + "mlp.down_proj.weight": mat(hs, ff), p + "ple_block.per_layer_input_gate.weight": mat(ple, hs),
                  p + "ple_block.per_layer_projection.weight": mat(hs, ple),
                  p + "ple_block.post_per_layer_input_norm.weight": norm(hs),
                  p + "layer_scalar": (0.5 + 0.5 * torch.rand(1, generator=g, device="cuda")).to(_BF16)})
    ids = np.random.default_rng(seed).integers(0, GEMMA_VOCAB, size=sum(_lengths(case))).astype(np.int32)
    return W, ids


# --------------------------------------------------------------------------
# The calls
# --------------------------------------------------------------------------

class _QwenShape:
    def __init__(self):
        self.__dict__.update(QWEN)


def prepare(case, seed):
    s = {"case": case}
    kind = case["kind"]
    if kind == "attn":
        q, k, v = s["qkv"] = _attn_inputs(case, seed)
        s["cu"] = _cu(_lengths(case))
        if case["plan"]:
            hq, hkv, d, causal, window, scale = FORMS[case["form"]]
            desc = inl_hip.make_attn_desc(s["cu"], hq, hkv, d, causal=causal, window=window, scale=scale,
                                          dtype=case["dtype"], q_row_stride=q.stride(0), k_row_stride=k.stride(0),
                                          v_row_stride=v.stride(0))
            s["plan"] = inl_hip.AttnPlan(desc)
            s["out"] = torch.empty(q.shape, dtype=q.dtype, device=q.device)
    elif kind == "prologue":
        s["in"] = _prologue_inputs(case, seed)
    elif kind == "mlp":
        s["in"] = _mlp_inputs(case, seed)
    elif kind == "splade":
        s["in"] = _splade_inputs(case, seed)
        s["cu"] = np.asarray(_cu(_lengths(case)), dtype=np.int32)
    elif kind == "gdn":
        s["in"] = _gdn_inputs(case, seed)
        s["cu"] = torch.tensor(_cu(_lengths(case)), dtype=torch.int32, device="cuda")
    elif kind == "qwen3":
        W, s["ids"] = _qwen3_inputs(case, seed)
        s["cu"] = _cu(_lengths(case))
        s["enc"] = inl_hip.Qwen3Encoder(_QwenShape(), W)
    else:
        W, s["ids"] = _gemma_inputs(case, seed)
        s["cu"] = _cu(_lengths(case))
        s["enc"] = inl_hip.Gemma2Encoder(_gemma_config(), W)
    return s


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "attn":
        q, k, v = state["qkv"]
        if case["plan"]:
            state["plan"].run(q, k, v, state["out"])
            return state["out"]
        _, _, _, causal, window, scale = FORMS[case["form"]]
        return inl_hip.varlen_attention(q, k, v, state["cu"], causal=causal, window=window, scale=scale)
    if kind == "prologue":
        x, qw, kw, rows, cos, sin = state["in"]
        return inl_hip.norm_rope_qk(x[:, :24], 16, rows, cos, sin, q_weight=qw, k_weight=kw, eps=1e-6)
    if kind == "mlp":
        x, gu, down = state["in"]
        act = inl_hip.gemm_bf16_gated(x, gu, "geglu")
        return act, inl_hip.gemm_bf16(act, down, out_dtype=_F32)
    if kind == "splade":
        head, w, bias, canonical = state["in"]
        maxima = inl_hip.splade_decoder_max(head, w, state["cu"])
        return maxima, inl_hip.splade_finish(maxima, bias=bias, shift=10.0, masked_ids=(50000, 50001),
                                             canonical=canonical, out_dim=SPLADE_TERMS)
    if kind == "gdn":
        proj, taps, a, b, dt_bias, neg_a, z, w = state["in"]
        H, D, cu = GDN_HEADS, GDN_DIM, state["cu"]
        mixed = inl_hip.gdn_conv(proj, cu, taps)
        g, beta = inl_hip.gdn_gates(a, b, dt_bias, neg_a)
        core = inl_hip.gdn_rule(mixed, cu, H, H, D, D, g, beta)
        return core, inl_hip.gdn_gated_norm(core, z, w, 1e-6)
    return state["enc"].encode(state["ids"], state["cu"])


# --------------------------------------------------------------------------
# What a pass cannot do without
# --------------------------------------------------------------------------

def _visible(case):
    """Visible (query, key) pairs of one head."""
    causal, window = FORMS[case["form"]][3:5]
    return sum(_pairs(t, causal, window) for t in _lengths(case))


def _pairs(t, causal, window):
    if window < 0 or window >= t:
        return t * (t + 1) // 2 if causal else t * t
    q = np.arange(t)
    hi = np.minimum(t, q + window + 1) if not causal else q + 1
    return int((hi - np.maximum(0, q - window)).sum())


def work(case):
    kind = case["kind"]
    if kind == "mlp":
        m, h, f = case["rows"], case["hidden"], case["ff"]
        return {"bytes": m * h * 2 + 3 * h * f * 2 + m * f * 2 + m * h * 4, "flops": 6 * m * h * f}
    lens = _lengths(case)
    n = sum(lens)
    if kind == "attn":
        hq, hkv, d = FORMS[case["form"]][:3]
        size = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": n * d * (2 * hq + 2 * hkv) * size, "flops": 4 * hq * d * _visible(case)}
    if kind == "prologue":
        size = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": n * 24 * 128 * size * 2 + n * 4 + max(lens) * 64 * 8, "flops": n * 24 * 128 * 7}
    if kind == "splade":
        V, H, B = SPLADE_VOCAB, SPLADE_HIDDEN, len(lens)
        return {"bytes": n * H * 2 + V * H * 2 + B * V * 4 + V * 8 + B * SPLADE_TERMS * 4, "flops": 2 * n * V * H}
    if kind == "gdn":
        H, D = GDN_HEADS, GDN_DIM
        size = 2 if case["dtype"] == "bf16" else 4
        # projections and z in, the rule's output and the layer's out
        return {"bytes": n * H * (D * (3 * size + size + 4 + size) + 2 * size),
                "flops": 7 * n * H * D * D + n * 3 * H * D * (2 * GDN_TAPS + 4)}
    if kind == "qwen3":
        c = QWEN
        per = c["hidden"] * (c["heads"] + 2 * c["kv_heads"]) * c["head_dim"] + c["heads"] * c["head_dim"] * c["hidden"] \
            + 3 * c["hidden"] * c["intermediate"]
        pairs = sum(_pairs(t, True, -1) for t in lens)
        size = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": c["layers"] * per * size + n * c["hidden"] * size + len(lens) * c["hidden"] * 4,
                "flops": c["layers"] * (2 * per * n + 4 * c["heads"] * c["head_dim"] * pairs)}
    hs, ff, ple, L = GEMMA_HIDDEN, GEMMA_FF, GEMMA_PLE, GEMMA_LAYERS
    per = hs * (1280 + 768 + 3 * ff + 3 * ple)
    sliding = sum(_pairs(t, False, 512) for t in lens)
    full = sum(_pairs(t, False, -1) for t in lens)
    return {"bytes": L * per * 2 + n * hs * 2 + len(lens) * 768 * 4,
            "flops": 2 * L * per * n + 4 * 3 * 256 * (L // 6 * full + (L - L // 6) * sliding)}


def tolerance(case):
    """About four times the distance from ``exact`` that was measured per
    kind and type (bf16: the rounding of the outputs, and in the layers and
    encodes of the values in between; f32: the order of the sums)."""
    f32 = case.get("dtype") == "f32"
    if case["kind"] == "gdn":
        return {"rel": 3e-6 if f32 else 2.5e-2}
    if case["kind"] == "qwen3":
        return {"rel": 8e-6 if f32 else 2.4e-2}
    if case["kind"] == "gemma":
        return {"rel": 3e-2}
    if case["kind"] == "splade":
        return {"rel": 3e-6}
    return {"rel": 2e-6 if f32 else 7e-3}


# --------------------------------------------------------------------------
# The same outputs in 64 bits
# --------------------------------------------------------------------------

def _attend(q, k, v, lens, causal, window, scale):
    """f64 attention over packed rows [n, heads, d]."""
    out, start = torch.empty(q.shape, dtype=_F64, device=q.device), 0
    rep = q.shape[1] // k.shape[1]
    for t in lens:
        e = start + t
        for h in range(q.shape[1]):
            s = (q[start:e, h] @ k[start:e, h // rep].T) * scale
            if causal or window >= 0:
                i = torch.arange(t, device=q.device)
                d = i[:, None] - i[None, :]
                hide = (d < 0) if causal else torch.zeros_like(d, dtype=torch.bool)
                if window >= 0:
                    hide = hide | (d.abs() > window)
                s = s.masked_fill(hide, -math.inf)
            out[start:e, h] = torch.softmax(s, -1) @ v[start:e, h // rep]
        start = e
    return out


def _rms(x, w=None, eps=1e-6):
    y = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
    return y if w is None else y * w


def _rope(x, cos, sin):
    half = x.shape[-1] // 2
    a, b, c, s = x[..., :half], x[..., half:], cos[:, None, :], sin[:, None, :]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _angles(lens, theta, d):
    pos = torch.from_numpy(np.concatenate([np.arange(t) for t in lens])).cuda().double()
    inv = theta ** (-torch.arange(0, d, 2, device="cuda", dtype=_F64) / d)
    a = pos[:, None] * inv[None, :]
    return torch.cos(a), torch.sin(a)


def _gelu(x):
    return torch.nn.functional.gelu(x, approximate="tanh")


def exact(case, seed):
    kind = case["kind"]
    if kind == "mlp":
        x, gu, down = (t.double() for t in _mlp_inputs(case, seed))
        f = case["ff"]
        act = _gelu(x @ gu[:f].T) * (x @ gu[f:].T)
        return act, act @ down.T
    lens = _lengths(case)
    if kind == "attn":
        q, k, v = (t.double() for t in _attn_inputs(case, seed))
        return _attend(q, k, v, lens, *FORMS[case["form"]][3:])
    if kind == "prologue":
        x, qw, kw, rows, cos, sin = _prologue_inputs(case, seed)
        c, s = cos.double()[rows.long()], sin.double()[rows.long()]
        x = x[:, :24].double()
        return torch.cat([_rope(_rms(x[:, :16], qw.double()), c, s), _rope(_rms(x[:, 16:], kw.double()), c, s)], 1)
    if kind == "splade":
        head, w, bias, canonical = _splade_inputs(case, seed)
        w, start, rows = w.double(), 0, []
        for t in lens:
            rows.append((head[start:start + t].double() @ w.T).amax(0))
            start += t
        maxima = torch.stack(rows)
        y = torch.log1p(torch.relu(maxima + bias.double() - 10.0))
        y[:, 50000:50002] = 0
        out = torch.zeros(len(lens), SPLADE_TERMS, dtype=_F64, device="cuda")
        return maxima, out.scatter_reduce(1, canonical.long()[None, :].expand(len(lens), -1), y, "amax")
    if kind == "gdn":
        return _gdn_exact(case, seed, lens)
    if kind == "qwen3":
        return _qwen3_exact(case, seed, lens)
    return _gemma_exact(case, seed, lens)


def _gdn_exact(case, seed, lens):
    proj, taps, a, b, dt_bias, neg_a, z, w = (t.double() for t in _gdn_inputs(case, seed))
    H, D, n, T = GDN_HEADS, GDN_DIM, sum(lens), max(lens)
    cu = _cu(lens)
    x = torch.zeros(len(lens), T, 3 * H * D, dtype=_F64, device="cuda")
    for i, t in enumerate(lens):
        p = torch.nn.functional.pad(proj[cu[i]:cu[i + 1]], (0, 0, GDN_TAPS - 1, 0))
        x[i, :t] = torch.nn.functional.silu(sum(p[j:j + t] * taps[:, j] for j in range(GDN_TAPS)))
    spread = torch.cat([torch.arange(t) + i * T for i, t in enumerate(lens)]).cuda()

    def padded(v):
        out = torch.zeros(len(lens) * T, H, dtype=_F64, device="cuda")
        out[spread] = v
        return out.view(len(lens), T, H)

    decay = torch.exp(padded(torch.nn.functional.softplus(a + dt_bias) * neg_a))
    beta = padded(torch.sigmoid(b))
    q, k, v = (x[..., i * H * D:(i + 1) * H * D].view(len(lens), T, H, D) for i in range(3))
    q = q * torch.rsqrt((q * q).sum(-1, keepdim=True) + 1e-6) * D ** -0.5
    k = k * torch.rsqrt((k * k).sum(-1, keepdim=True) + 1e-6)
    S = torch.zeros(len(lens), H, D, D, dtype=_F64, device="cuda")
    core = torch.empty(len(lens), T, H, D, dtype=_F64, device="cuda")
    for t in range(T):
        S = S * decay[:, t, :, None, None]
        kt = k[:, t, :, :, None]
        u = (v[:, t] - (S * kt).sum(2)) * beta[:, t, :, None]
        S = S + kt * u[:, :, None, :]
        core[:, t] = (S * q[:, t, :, :, None]).sum(2)
    core = core.view(len(lens) * T, H, D)[spread]
    return core, _rms(core, w) * torch.nn.functional.silu(z)


def _qwen3_exact(case, seed, lens):
    W, ids = _qwen3_inputs(case, seed)
    c, w = QWEN, lambda name: W[name].double()
    n, hq, hkv, d = sum(lens), c["heads"], c["kv_heads"], c["head_dim"]
    cos, sin = _angles(lens, c["theta"], d)
    h = W["embed_tokens.weight"][torch.from_numpy(ids).cuda().long()].double()
    for i in range(c["layers"]):
        p = f"layers.{i}."
        x = _rms(h, w(p + "input_layernorm.weight"))
        q, k, v = ((x @ w(p + f"self_attn.{m}_proj.weight").T).view(n, -1, d) for m in "qkv")
        q = _rope(_rms(q, w(p + "self_attn.q_norm.weight")), cos, sin)
        k = _rope(_rms(k, w(p + "self_attn.k_norm.weight")), cos, sin)
        a = _attend(q, k, v, lens, True, -1, d ** -0.5).view(n, hq * d)
        h = h + a @ w(p + "self_attn.o_proj.weight").T
        x = _rms(h, w(p + "post_attention_layernorm.weight"))
        x = torch.nn.functional.silu(x @ w(p + "mlp.gate_proj.weight").T) * (x @ w(p + "mlp.up_proj.weight").T)
        h = h + x @ w(p + "mlp.down_proj.weight").T
    last = torch.tensor(_cu(lens)[1:], device="cuda") - 1
    return torch.nn.functional.normalize(_rms(h[last], w("norm.weight")), dim=-1)


def _gemma_exact(case, seed, lens):
    W, ids = _gemma_inputs(case, seed)
    w = lambda name: W[name].double()
    tc, n, eps = _gemma_config(), sum(lens), 1e-6
    tables = {kind: _angles(lens, p["rope_theta"], 256) for kind, p in tc["rope_parameters"].items()}
    h = W["embed_tokens.weight"][torch.from_numpy(ids).cuda().long()].double() * GEMMA_HIDDEN ** 0.5
    emb = h
    for i in range(GEMMA_LAYERS):
        p = f"layers.{i}."
        wp = w("ple.per_layer_model_projection.weight")[i * GEMMA_PLE:(i + 1) * GEMMA_PLE]
        ple = _rms(emb @ wp.T * GEMMA_HIDDEN ** -0.5, w("ple.per_layer_projection_norm.weight"), eps)
        x = _rms(h, w(p + "input_layernorm.weight"))
        q, k, v = ((x @ w(p + f"self_attn.{m}_proj.weight").T).view(n, -1, 256) for m in "qkv")
        kind = tc["layer_types"][i]
        q = _rope(_rms(q, w(p + "self_attn.q_norm.weight")), *tables[kind])
        k = _rope(_rms(k, w(p + "self_attn.k_norm.weight")), *tables[kind])
        a = _attend(q, k, _rms(v), lens, False, 512 if kind == "sliding_attention" else -1, 1.0).view(n, 768)
        h = h + _rms(a @ w(p + "self_attn.o_proj.weight").T, w(p + "post_attention_layernorm.weight"))
        x = _rms(h, w(p + "pre_feedforward_layernorm.weight"))
        x = _gelu(x @ w(p + "mlp.gate_proj.weight").T) * (x @ w(p + "mlp.up_proj.weight").T)
        h = h + _rms(x @ w(p + "mlp.down_proj.weight").T, w(p + "post_feedforward_layernorm.weight"))
        x = _gelu(h @ w(p + "ple_block.per_layer_input_gate.weight").T) * ple
        h = h + _rms(x @ w(p + "ple_block.per_layer_projection.weight").T,
                     w(p + "ple_block.post_per_layer_input_norm.weight"))
        h = h * w(p + "layer_scalar")
    h = _rms(h, w("norm.weight"))
    cu = _cu(lens)
    mean = torch.stack([h[cu[b]:cu[b + 1]].mean(0) for b in range(len(lens))])
    return torch.nn.functional.normalize(mean @ w("embedding_projection.weight").T, dim=-1)
