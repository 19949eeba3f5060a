"""Performance cases: what a program built on ncmorph_amd has it do.

Every case is one pass through the package's public entry points on data that
is already where such a program holds it: device tensors for activations,
weights and tables; token ids on the host, which is where the forwards take
them. `listed()` holds the fixed cases, `draw(rng)` gives further ones of the
same ranges. Kinds:

  linear       one bf16 projection y = x W^T (+ bias)
  mlp          RMSNorm, gate|up projection with SwiGLU, down projection with
               the residual add: a decoder layer's second half
  attn         RMSNorm, q|k|v projection with RoPE, causal grouped-query
               attention, output projection with the residual add: a decoder
               layer's first half
  decoder      token ids to logits, bf16 mode, whole model
  decoder_f32  the same in the f32 mode (checkpoints that are not all BF16)
  ncm          the NCM level-parallel step: body and codebook-tied code heads
  rvq          multiscale residual VQ, encode (codes, reconstruction) then
               decode (codes to reconstruction)
  tok_encode   VQ-VAE tokenizer, token ids to codes and latent
  tok_decode   VQ-VAE tokenizer, codes to logits
"""
from __future__ import annotations

import math

import numpy as np
import torch

from ncmorph_amd import decoder, kernels, ncm, vq, vq_tokenizer

DEV = "cuda:0"

# hidden, intermediate, vocab, q heads, kv heads, head_dim, layers of the
# checkpoints whose configurations the test suite holds.
MODELS = {
    "smollm2-135m": (576, 1536, 49152, 9, 3, 64, 30),
    "qwen2.5-0.5b": (896, 4864, 151936, 14, 2, 64, 24),
    "qwen3-0.6b": (1024, 3072, 151936, 16, 8, 128, 28),
    "llama-3.2-1b": (2048, 8192, 128256, 32, 8, 64, 16),
    "llama-3.0-8b": (4096, 14336, 128256, 32, 8, 128, 32),
}


def listed():
    return [
        # A short prompt through one square projection: too little work to
        # fill the GPU, so launch and latency count.
        dict(name="linear_short", kind="linear", m=17, k=2048, n=2048, out_mode="bf16_f32",
             bias=False),
        # The FFN up projection of a 2048-token prefill, fp32 output.
        dict(name="linear_ffn", kind="linear", m=2048, k=2048, n=8192, out_mode="f32",
             bias=False),
        # The MLP half of a layer for a prompt of ragged, ordinary length.
        dict(name="mlp_prompt", kind="mlp", model="llama-3.2-1b", rows=203),
        # The attention half of a layer in a batched prefill.
        dict(name="attn_prefill", kind="attn", model="llama-3.2-1b", batch=4, seq=1024,
             window=0),
        # A whole model on one chat-sized prompt.
        dict(name="decoder_prompt", kind="decoder", model="llama-3.2-1b", layers=16, batch=1,
             seq=77),
        # A whole model on a batch of long prompts (the prefill benchmark).
        dict(name="decoder_batch", kind="decoder", model="llama-3.2-1b", layers=16, batch=4,
             seq=1024),
        # A small checkpoint with float32 tensors: the f32 mode.
        dict(name="decoder_f32", kind="decoder_f32", model="smollm2-135m", layers=30, batch=1,
             seq=200),
        # Two layers of the 8B-shaped NCM body and the eight code heads over
        # the levels of a 4096-position sequence.
        dict(name="ncm_step", kind="ncm", model="llama-3.0-8b", layers=2, prefix=64,
             positions=4096, levels=8, codes=8192, mask="block_causal"),
        # One short sequence, every level at full resolution: latency.
        dict(name="rvq_small", kind="rvq", b=1, t=128, d=256, v=512, levels=4, top_stride=1),
        # The tokenizer of a training pipeline: a large batch, eight scales.
        dict(name="rvq_large", kind="rvq", b=16, t=2048, d=2048, v=4096, levels=8,
             top_stride=128),
        # Tokenizing and detokenizing batches of sentences.
        dict(name="tok_encode", kind="tok_encode", b=96),
        dict(name="tok_decode", kind="tok_decode", b=24),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["linear", "linear", "mlp", "attn", "decoder", "decoder", "decoder_f32",
                       "ncm", "rvq", "rvq", "tok_encode", "tok_decode"])
    if kind == "linear":
        hidden, inter, _, hq, hkv, hd, _ = MODELS[rng.choice(sorted(MODELS))]
        k, n = rng.choice([(hidden, hidden), (hidden, inter), (inter, hidden),
                           (hidden, (hq + 2 * hkv) * hd)])
        return dict(kind=kind, m=_log(rng, 1, 4096), k=k, n=n,
                    out_mode=rng.choice(["f32", "bf16_f32", "bf16"]), bias=rng.random() < 0.3)
    if kind == "mlp":
        return dict(kind=kind, model=rng.choice(sorted(MODELS)), rows=_log(rng, 1, 4096))
    if kind == "attn":
        batch = rng.choice([1, 1, 2, 3, 4])
        return dict(kind=kind, model=rng.choice(sorted(MODELS)), batch=batch,
                    seq=_log(rng, 8, 4096 // batch), window=rng.choice([0, 0, 0, 256]))
    if kind == "decoder":
        model = rng.choice(["smollm2-135m", "qwen2.5-0.5b", "qwen3-0.6b", "llama-3.2-1b"])
        batch = rng.choice([1, 1, 2, 4])
        return dict(kind=kind, model=model, layers=MODELS[model][6], batch=batch,
                    seq=_log(rng, 4, 2048 // batch))
    if kind == "decoder_f32":
        model = rng.choice(["smollm2-135m", "qwen2.5-0.5b"])
        return dict(kind=kind, model=model, layers=MODELS[model][6], batch=rng.choice([1, 1, 2]),
                    seq=_log(rng, 4, 300))
    if kind == "ncm":
        levels = rng.randint(3, 8)
        return dict(kind=kind, model=rng.choice(["qwen3-0.6b", "llama-3.2-1b", "llama-3.0-8b"]),
                    layers=2, prefix=_log(rng, 5, 128), levels=levels,
                    positions=rng.randint(1, 3584 >> (levels - 1)) << (levels - 1),
                    codes=rng.choice([1000, 4096, 8192]),
                    mask=rng.choice(["block_causal", "block_diagonal"]))
    if kind == "rvq":
        levels = rng.randint(2, 8)
        top = 1 << rng.randint(0, levels - 1)
        return dict(kind=kind, b=_log(rng, 1, 12), t=top * rng.randint(1, max(1, 2048 // top)),
                    d=64 * rng.randint(2, 32), v=rng.choice([512, 1000, 2048, 4096]),
                    levels=levels, top_stride=top)
    if kind == "tok_encode":
        return dict(kind=kind, b=_log(rng, 1, 500))
    return dict(kind=kind, b=_log(rng, 1, 64))


# ------------------------------------------------------------------ helpers

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV) * std


def _bf16(g, *shape, std=1.0):
    return _randn(g, *shape, std=std).to(torch.bfloat16)


def _spec(case):
    hidden, inter, vocab, hq, hkv, hd, _ = MODELS[case["model"]]
    return decoder.DecoderSpec(hidden=hidden, intermediate=inter, vocab=vocab, q_heads=hq,
                               kv_heads=hkv, head_dim=hd, layers=case.get("layers", 1),
                               window=case.get("window", 0))


def _ncm_spec(case):
    hidden, inter, vocab, hq, hkv, hd, _ = MODELS[case["model"]]
    return ncm.NcmSpec(hidden=hidden, vq_width=hidden, intermediate=inter, q_heads=hq,
                       kv_heads=hkv, head_dim=hd, layers=case["layers"],
                       level_lengths=ncm.multiscale_levels(case["positions"], case["levels"]),
                       prefix_length=case["prefix"], prefix_vocab=vocab, mask=case["mask"])


def _strides(case):
    """Non-increasing powers of two from top_stride down to 1, the finest
    scale repeated when there are more levels than scales."""
    return [max(1, case["top_stride"] >> l) for l in range(case["levels"])]


def _tables(spec, positions):
    cos, sin = decoder.rope_tables(spec, positions)
    return torch.from_numpy(cos).to(DEV), torch.from_numpy(sin).to(DEV)


def _f32_weights(spec, g):
    """Float32 checkpoint tensors in the layout of decoder.forward_f32."""
    h, i, qw = spec.hidden, spec.intermediate, spec.q_heads * spec.head_dim

    def w(*shape):
        return _randn(g, *shape, std=0.02)

    layers = [{"input_norm": 1.0 + w(h), "qkv_weight": w(spec.qkv_width, h), "o_weight": w(h, qw),
               "post_attention_norm": 1.0 + w(h), "gate_weight": w(i, h), "up_weight": w(i, h),
               "down_weight": w(h, i)} for _ in range(spec.layers)]
    return decoder.DecoderWeights(embed=w(spec.vocab, h), final_norm=1.0 + w(h), layers=layers,
                                  mode="f32")


# ------------------------------------------------------------------ prepare

def prepare(case, seed):
    g = _gen(seed)
    kind = case["kind"]
    s = {"case": case}
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        s.update(x=_bf16(g, m, k), w=_bf16(g, n, k, std=0.02),
                 bias=_bf16(g, n, std=0.02) if case["bias"] else None)
    elif kind == "mlp":
        sp = _spec(case)
        s.update(spec=sp, h=_bf16(g, case["rows"], sp.hidden).float(),
                 norm=1.0 + _randn(g, sp.hidden, std=0.02),
                 gate_up=_bf16(g, 2 * sp.intermediate, sp.hidden, std=0.02),
                 down=_bf16(g, sp.hidden, sp.intermediate, std=0.02))
    elif kind == "attn":
        sp = _spec(case)
        s.update(spec=sp, h=_bf16(g, case["batch"] * case["seq"], sp.hidden).float(),
                 norm=1.0 + _randn(g, sp.hidden, std=0.02),
                 qkv=_bf16(g, sp.qkv_width, sp.hidden, std=0.02),
                 o=_bf16(g, sp.hidden, sp.q_heads * sp.head_dim, std=0.02),
                 tables=_tables(sp, case["seq"]))
    elif kind in ("decoder", "decoder_f32"):
        sp = _spec(case)
        ids = np.random.default_rng(seed).integers(0, sp.vocab, (case["batch"], case["seq"]))
        weights = (decoder.random_weights(sp, DEV, seed=seed) if kind == "decoder"
                   else _f32_weights(sp, g))
        s.update(spec=sp, weights=weights, ids=ids, tables=_tables(sp, case["seq"]))
    elif kind == "ncm":
        sp = _ncm_spec(case)
        nl, v = len(sp.level_lengths), case["codes"]
        cos, sin = ncm.rope_tables(sp)
        books = _bf16(g, nl, v, sp.hidden, std=sp.hidden ** -0.5)
        s.update(spec=sp, weights=ncm.random_weights(sp, DEV, seed=seed),
                 ids=np.random.default_rng(seed).integers(0, sp.prefix_vocab, sp.prefix_length),
                 target=_randn(g, sum(sp.level_lengths), sp.vq_width),
                 tables=(torch.from_numpy(cos).to(DEV), torch.from_numpy(sin).to(DEV)),
                 z=_bf16(g, nl, sp.hidden, sp.hidden, std=0.02), books=books,
                 csq=vq.prepare(books))
    elif kind == "rvq":
        d, v = case["d"], case["v"]
        books = _bf16(g, case["levels"], v, d, std=d ** -0.5)
        s.update(x=_randn(g, case["b"], case["t"], d), books=books, csq=vq.prepare(books),
                 strides=_strides(case))
    else:
        cfg = vq_tokenizer.WMT14
        rng = np.random.default_rng(seed)
        s["tok"] = vq_tokenizer.Tokenizer(
            cfg, vq_tokenizer.random_state(cfg, DEV, seed=seed, decoder=kind == "tok_decode"))
        if kind == "tok_encode":
            s["ids"] = rng.integers(0, cfg.in_vocab, (case["b"], cfg.seq_len))
        else:
            codes = np.concatenate([rng.integers(0, v, (case["b"], n)) for n, v in
                                    zip(cfg.levels, cfg.vocab_sizes)], axis=1)
            s["codes"] = torch.from_numpy(codes.astype(np.int32)).to(DEV)
    return s


# ---------------------------------------------------------------------- run

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "linear":
        if case["out_mode"] == "bf16":
            y = torch.empty(case["m"], case["n"], dtype=torch.bfloat16, device=DEV)
            return kernels.linear_bf16(s["x"], s["w"], bias=s["bias"], out=y, out_mode="bf16")
        return kernels.linear_bf16(s["x"], s["w"], bias=s["bias"], out_mode=case["out_mode"])
    if kind == "mlp":
        sp = s["spec"]
        n = kernels.rms_norm_rows(s["h"], s["norm"], sp.rms_eps, out_mode="bf16")
        a = kernels.linear_bf16_swiglu(n, s["gate_up"])
        return {"act": a, "hidden": kernels.linear_bf16_residual(a, s["down"], s["h"])}
    if kind == "attn":
        sp, (cos, sin) = s["spec"], s["tables"]
        b, t, hd = case["batch"], case["seq"], sp.head_dim
        qw, kw = sp.q_heads * hd, sp.kv_heads * hd
        n = kernels.rms_norm_rows(s["h"], s["norm"], sp.rms_eps, out_mode="bf16")
        if hd == 64:
            qkv = kernels.linear_bf16_rope64(n, s["qkv"], qw + kw, t, cos, sin)
        else:
            qkv = torch.empty(b * t, sp.qkv_width, dtype=torch.bfloat16, device=DEV)
            kernels.linear_bf16(n, s["qkv"], out=qkv, out_mode="bf16")
            kernels.rope_rotate(qkv[:, :qw], sp.q_heads, hd, t, cos, sin)
            kernels.rope_rotate(qkv[:, qw:qw + kw], sp.kv_heads, hd, t, cos, sin)
        ctx = kernels.attention_bf16(qkv[:, :qw], qkv[:, qw:qw + kw], qkv[:, qw + kw:], b, t,
                                     sp.q_heads, sp.kv_heads, hd, window=sp.window,
                                     out_mode="bf16")
        return {"qkv": qkv, "context": ctx,
                "hidden": kernels.linear_bf16_residual(ctx, s["o"], s["h"])}
    if kind in ("decoder", "decoder_f32"):
        return decoder.run(s["spec"], s["weights"], s["ids"], *s["tables"])
    if kind == "ncm":
        sp = s["spec"]
        h = ncm.forward(sp, s["weights"], s["ids"], s["target"], *s["tables"])
        return {"hidden": h, "logits": ncm.code_head_logits(sp, h, s["z"], s["books"], s["csq"])}
    if kind == "rvq":
        r = vq.encode(s["x"], s["books"], s["strides"], csq=s["csq"], want_gap=False)
        back = vq.decode(r["codes"], s["books"], s["strides"], case["t"])
        return {"codes": r["codes"], "recon": r["recon"], "decoded": back}
    if kind == "tok_encode":
        r = s["tok"].encode(s["ids"])
        return {"codes": r["codes"], "zhat": r["zhat"]}
    zhat = s["tok"].reconstruct(s["codes"])
    return {"zhat": zhat, "logits": s["tok"].decode(zhat)}


# --------------------------------------------------------------------- work

def _causal_pairs(seq, window):
    if window <= 0 or window >= seq:
        return seq * (seq + 1) // 2
    return window * (window + 1) // 2 + (seq - window) * window


def _level_pairs(sp):
    """Allowed (query, key) pairs of the level mask: prefix keys for every
    position, and the own level (block_diagonal) or every level up to it."""
    pairs, seen = sp.seq_len * sp.prefix_length, 0
    for n in sp.level_lengths:
        seen += n
        pairs += n * (n if sp.mask == "block_diagonal" else seen)
    return pairs


def _layer_params(sp):
    return (sp.hidden * (sp.qkv_width + sp.q_heads * sp.head_dim)
            + 3 * sp.hidden * sp.intermediate)


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        out = 2 if case["out_mode"] == "bf16" else 4
        return {"bytes": 2 * (m * k + n * k) + out * m * n + (2 * n if case["bias"] else 0),
                "flops": 2 * m * n * k}
    if kind == "mlp":
        sp, m = _spec(case), case["rows"]
        p = 3 * sp.hidden * sp.intermediate
        return {"bytes": 2 * p + m * (8 * sp.hidden + 2 * sp.intermediate) + 4 * sp.hidden,
                "flops": 2 * m * p}
    if kind == "attn":
        sp, m = _spec(case), case["batch"] * case["seq"]
        qw = sp.q_heads * sp.head_dim
        p = sp.hidden * (sp.qkv_width + qw)
        pairs = case["batch"] * _causal_pairs(case["seq"], sp.window)
        return {"bytes": 2 * p + m * (8 * sp.hidden + 2 * sp.qkv_width + 2 * qw)
                + 8 * case["seq"] * sp.head_dim + 4 * sp.hidden,
                "flops": 2 * m * p + 4 * sp.head_dim * sp.q_heads * pairs}
    if kind in ("decoder", "decoder_f32"):
        sp, m = _spec(case), case["batch"] * case["seq"]
        esz = 2 if kind == "decoder" else 4
        p = sp.layers * _layer_params(sp) + sp.vocab * sp.hidden
        pairs = case["batch"] * _causal_pairs(case["seq"], 0)
        return {"bytes": esz * p + 4 * m * sp.vocab + 8 * m,
                "flops": 2 * m * p + sp.layers * 4 * sp.head_dim * sp.q_heads * pairs}
    if kind == "ncm":
        sp, v = _ncm_spec(case), case["codes"]
        S, T, nl = sp.seq_len, sum(sp.level_lengths), len(sp.level_lengths)
        p = sp.layers * _layer_params(sp) + sp.hidden * sp.vq_width
        head = sp.hidden * sp.hidden + v * sp.hidden
        return {"bytes": 2 * p + 2 * nl * head + 4 * T * (sp.vq_width + v) + 4 * S * sp.hidden,
                "flops": 2 * S * p + 2 * T * head
                + sp.layers * 4 * sp.head_dim * sp.q_heads * _level_pairs(sp)}
    if kind == "rvq":
        b, t, d, v = case["b"], case["t"], case["d"], case["v"]
        rows = sum(t // x for x in _strides(case))
        return {"bytes": 4 * b * t * d * 3 + 2 * case["levels"] * v * d + 8 * b * rows,
                "flops": 2 * b * rows * v * d}
    cfg, b = vq_tokenizer.WMT14, case["b"]
    L, d, books = cfg.seq_len, cfg.embed_dim, sum(cfg.vocab_sizes)
    convs, codes = cfg.n_levels * 3 * d * d, cfg.codes_per_sequence
    if kind == "tok_encode":
        f = vq_tokenizer.flops_per_sequence(cfg)["total"]
        return {"bytes": 4 * d * (books + b * L * 2) + 4 * convs + b * (8 * L + 4 * codes),
                "flops": b * f}
    f = vq_tokenizer.flops_per_sequence(cfg)
    dense = 12 * d * d + d * cfg.in_vocab
    return {"bytes": 4 * (convs + dense) + 4 * b * (L * (cfg.in_vocab + d) + codes),
            "flops": b * (f["phi"] + f["cascade"] / 2 + 2 * L * dense + 4 * L * L * d)}


# ---------------------------------------------------------------- tolerance

def tolerance(case):
    """Relative 2-norm errors that a change of summation order may bring.

    Products of bf16 values are exact in fp32, so an fp32 result moves by its
    sum's rounding only (3e-7 from float64 at K = 2048, up to three times that
    at K = 14336); a bf16 result by a step of 2^-8 where the sum lies at a
    rounding boundary (about one in thirty does); a block of several bf16
    stages by a few such steps (blocks are 2e-3 to 9e-3 from float64), and a
    whole bf16 model by the steps of all its layers (2e-2 to 3e-2 from
    float64; another order moves the result by about half of that). The f32
    model and the tokenizer's decoder are 1e-6 and 5e-7 from float64. The
    RVQ's codes and sums follow one fixed fp32 order, so they are whole. The
    VQ-VAE tokenizer's codes may differ where two float32 distances tie, and
    the rest of that sequence with them."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 3e-6} if case["out_mode"] == "f32" else {"rel": 3e-3, "max": 2e-2}
    if kind in ("mlp", "attn"):
        return {"rel": 1e-2, "max": 0.2}
    if kind == "decoder":
        return {"rel": 3e-2, "max": 0.5}
    if kind == "decoder_f32":
        return {"rel": 1e-5, "max": 4e-4}
    if kind == "ncm":
        return {"rel": 2e-2, "max": 0.4}
    if kind == "rvq":
        return "exact"
    if kind == "tok_encode":
        return {"rel": 2e-2, "max": 0.9, "differ": 1e-2}
    return {"rel": 5e-6, "max": 2e-4}


# -------------------------------------------------------------------- exact

def _norm64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()


def _rotate64(x, cos, sin):
    """x [rows, heads, hd] rotated by table rows [rows, hd]."""
    half = x.shape[-1] // 2
    turned = torch.cat([-x[..., half:], x[..., :half]], dim=-1)
    return x * cos[:, None, :] + turned * sin[:, None, :]


def _attend64(q, k, v, mask):
    """softmax(q k^T / sqrt(hd)) v per head; q [T, Hq, hd], k, v [T, Hkv, hd]."""
    T, hq, hd = q.shape
    group = hq // k.shape[1]
    out = torch.empty_like(q)
    for h in range(hq):
        s = (q[:, h] @ k[:, h // group].t().contiguous()) * hd ** -0.5
        p = torch.softmax(s.masked_fill(~mask, -math.inf), dim=-1)
        out[:, h] = p @ v[:, h // group].contiguous()
    return out.reshape(T, hq * hd)


def _attn64(sp, x, L, cos, sin, batch, mask):
    """(q|k|v rows after the rotation, context) of normed rows x."""
    qw, kw, hd = sp.q_heads * sp.head_dim, sp.kv_heads * sp.head_dim, sp.head_dim
    qkv = x @ L["qkv_weight"].double().t()
    T = x.shape[0] // batch
    ctx = []
    for b in range(batch):
        rows = qkv[b * T:(b + 1) * T]
        q = _rotate64(rows[:, :qw].reshape(T, -1, hd), cos, sin)
        k = _rotate64(rows[:, qw:qw + kw].reshape(T, -1, hd), cos, sin)
        rows[:, :qw], rows[:, qw:qw + kw] = q.reshape(T, qw), k.reshape(T, kw)
        ctx.append(_attend64(q, k, rows[:, qw + kw:].reshape(T, -1, hd), mask))
    return qkv, torch.cat(ctx)


def _swiglu64(x, gate_up):
    """gate and up rows interleaved in groups of 32."""
    gu = (x @ gate_up.double().t()).reshape(x.shape[0], -1, 2, 32)
    return (torch.nn.functional.silu(gu[:, :, 0]) * gu[:, :, 1]).reshape(x.shape[0], -1)


def _mlp64(x, L):
    if "gate_up_weight" in L:
        return _swiglu64(x, L["gate_up_weight"]) @ L["down_weight"].double().t()
    g, u = x @ L["gate_weight"].double().t(), x @ L["up_weight"].double().t()
    return (torch.nn.functional.silu(g) * u) @ L["down_weight"].double().t()


def _layers64(sp, h, layers, cos, sin, batch, mask):
    for L in layers:
        _, ctx = _attn64(sp, _norm64(h, L["input_norm"], sp.rms_eps), L, cos, sin, batch, mask)
        h = h + ctx @ L["o_weight"].double().t()
        h = h + _mlp64(_norm64(h, L["post_attention_norm"], sp.rms_eps), L)
    return h


def _causal(T, window):
    i = torch.arange(T, device=DEV)
    ok = i[None, :] <= i[:, None]
    return ok & (i[None, :] > i[:, None] - window) if window > 0 else ok


def _rvq64(s, case):
    x, books = s["x"].double(), s["books"].double()
    b, t, d = x.shape
    total, codes = torch.zeros_like(x), []
    for l, stride in enumerate(s["strides"]):
        u = (x - total).reshape(b, t // stride, stride, d).mean(2).reshape(-1, d)
        c = books[l]
        idx = torch.cat([((c * c).sum(1)[None] - 2.0 * (r @ c.t())).argmin(1)
                         for r in u.split(8192)])
        total += c[idx].reshape(b, t // stride, 1, d).expand(-1, -1, stride, -1).reshape(b, t, d)
        codes.append(idx.reshape(b, -1))
    return {"codes": torch.cat(codes, 1).to(torch.int32), "recon": total, "decoded": total}


def _conv3_64(h, w, bias):
    hp = torch.nn.functional.pad(h, (0, 0, 1, 1))
    L = h.shape[1]
    return bias + sum(hp[:, k:k + L] @ w[:, :, k].t() for k in range(3))


def _tok_state64(case, seed):
    cfg = vq_tokenizer.WMT14
    st = vq_tokenizer.random_state(cfg, DEV, seed=seed)
    return cfg, {n: t.double() for n, t in st.items()}


def _group_norm64(x, groups, eps):
    return torch.nn.functional.group_norm(x.transpose(1, 2), groups, eps=eps).transpose(1, 2)


def _tok_decode64(case, seed, codes):
    cfg, w = _tok_state64(case, seed)
    F = torch.nn.functional
    zhat, off = 0.0, 0
    for l, n in enumerate(cfg.levels):
        h = w[f"vq.embeddings.{l}.weight"][codes[:, off:off + n].long()]
        off += n
        if l == 0:
            strides = cfg.cascade_strides()
            for j in range(len(strides)):
                conv = f"vq.learned_up_l1.{2 * j}."  # a GroupNorm after each inner conv
                h = F.conv_transpose1d(h.transpose(1, 2), w[conv + "weight"], w[conv + "bias"],
                                       stride=strides[j]).transpose(1, 2)
                if cfg.cascade_norm and j < len(strides) - 1:
                    h = _group_norm64(h, cfg.groups, cfg.group_eps)
        elif n != cfg.seq_len:
            h = F.interpolate(h.transpose(1, 2), size=cfg.seq_len, mode="linear").transpose(1, 2)
        r = cfg.resi_ratio
        zhat = zhat + (1 - r) * h + r * _conv3_64(h, w[f"vq.quant_resi.{l}.weight"],
                                                  w[f"vq.quant_resi.{l}.bias"])
    p, d, hn = "decoder.middle_block.", cfg.embed_dim, cfg.n_head
    b, t = zhat.shape[:2]

    def rms(x, name):
        return x * torch.rsqrt((x * x).mean(-1, keepdim=True) + cfg.qk_eps) * w[name]

    x = zhat
    h = F.layer_norm(x, (d,), w[p + "ln_1.weight"], w[p + "ln_1.bias"], cfg.ln_eps)
    qkv = h @ w[p + "attn.c_attn.weight"].t() + w[p + "attn.c_attn.bias"]
    q, k, v = (y.reshape(b, t, hn, d // hn).transpose(1, 2) for y in qkv.split(d, dim=-1))
    q, k = rms(q, p + "attn.q_norm.weight"), rms(k, p + "attn.k_norm.weight")
    s = torch.softmax((q @ k.transpose(2, 3).contiguous()) * (d // hn) ** -0.5, dim=-1)
    a = (s @ v.contiguous()).transpose(1, 2).reshape(b, t, d)
    x = x + a @ w[p + "attn.c_proj.weight"].t() + w[p + "attn.c_proj.bias"]
    h = F.layer_norm(x, (d,), w[p + "ln_2.weight"], w[p + "ln_2.bias"], cfg.ln_eps)
    h = F.gelu(h @ w[p + "mlp.c_fc.weight"].t() + w[p + "mlp.c_fc.bias"])
    x = x + h @ w[p + "mlp.c_proj.weight"].t() + w[p + "mlp.c_proj.bias"]
    x = F.layer_norm(x, (d,), w["decoder.ln_f.weight"], None, cfg.ln_eps)
    return {"zhat": zhat, "logits": x @ w["decoder.output_layer.weight"].t()}


def exact(case, seed):
    """The same outputs in float64 with no rounding between the stages. None
    for the tokenizer's encode: its latent is a function of codes that are
    chosen by comparing distances, so it has no value of its own."""
    kind = case["kind"]
    if kind == "tok_encode":
        return None
    s = prepare(case, seed)
    if kind == "linear":
        y = s["x"].double() @ s["w"].double().t()
        return y if s["bias"] is None else y + s["bias"].double()
    if kind == "mlp":
        h = s["h"].double()
        a = _swiglu64(_norm64(h, s["norm"], s["spec"].rms_eps), s["gate_up"])
        return {"act": a, "hidden": h + a @ s["down"].double().t()}
    if kind == "attn":
        sp, h = s["spec"], s["h"].double()
        cos, sin = (x.double() for x in s["tables"])
        qkv, ctx = _attn64(sp, _norm64(h, s["norm"], sp.rms_eps), {"qkv_weight": s["qkv"]}, cos,
                           sin, case["batch"], _causal(case["seq"], sp.window))
        return {"qkv": qkv, "context": ctx, "hidden": h + ctx @ s["o"].double().t()}
    if kind in ("decoder", "decoder_f32"):
        sp, w = s["spec"], s["weights"]
        h = w.embed[torch.from_numpy(s["ids"].ravel()).to(DEV)].double()
        cos, sin = (x.double() for x in s["tables"])
        h = _layers64(sp, h, w.layers, cos, sin, case["batch"], _causal(case["seq"], 0))
        return _norm64(h, w.final_norm, sp.rms_eps) @ w.embed.double().t()
    if kind == "ncm":
        sp, w = s["spec"], s["weights"]
        n0, P = sp.level_lengths[0], sp.prefix_length
        x = torch.cat([w.prefix_token_embedding[torch.from_numpy(s["ids"]).to(DEV)].double(),
                       w.l0_queries.double(), s["target"][n0:].double()])
        h = x @ w.input_projection.double().t() + w.input_projection_bias.double()
        level = torch.repeat_interleave(torch.arange(len(sp.level_lengths), device=DEV),
                                        torch.tensor(sp.level_lengths, device=DEV))
        h[P:] += w.level_embedding.double()[level]
        of = torch.cat([torch.full((P,), -1, device=DEV), level])
        same = (of[None, :] == of[:, None] if sp.mask == "block_diagonal"
                else of[None, :] <= of[:, None])
        mask = same & (of[:, None] >= 0) | (of[None, :] < 0)
        cos, sin = (y.double() for y in s["tables"])
        h = _norm64(_layers64(sp, h, w.layers, cos, sin, 1, mask), w.final_norm, sp.rms_eps)
        logits = []
        for l, rows in enumerate(h[P:].split(list(sp.level_lengths))):
            e = s["books"][l].double()
            esq = (e * e).sum(1)
            logits.append((2.0 * (rows @ s["z"][l].double().t()) @ e.t() - esq) / esq.mean())
        return {"hidden": h, "logits": torch.cat(logits)}
    if kind == "rvq":
        return _rvq64(s, case)
    return _tok_decode64(case, seed, s["codes"])
