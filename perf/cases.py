"""The work that a user has this framework do, as cases that can be timed and compared.

Every case goes through a public entry point: the linears and quantizers of
nanoinfer_amd.quant, the decoder of nanoinfer_amd.model, and the C++ decoder
behind nanoinfer_amd.nicpp. Kinds:

  linear    one projection: quant.linear_q8 / linear_q4g / linear_q4 / linear_w8a8
            over 1 (one decoded token) to 2048 (a prompt) activation rows
  quantize  weights made at load time: quant.quantize_q8 / quantize_q4g
  block     one decoder layer of nanoinfer_amd.model on the hidden states of a
            prompt: norms, RoPE, attention and the W8A8 projections
  decoder   nicpp.Model.forward: token ids in, logits out, weight-only projections
            between fp32 activations

Inputs are synthetic: weights N(0, 0.02), activations N(0, 1), random token ids.
"""
import math
import os
import shutil
import tempfile

import numpy as np
import torch

from nanoinfer_amd import model, quant

DEV = "cuda"
DTYPE = {"f32": torch.float32, "f16": torch.float16}


def linear(name, fmt, m, n, k, x="f16", y=None, group=32, scale="f32", bias=False):
    """group and scale are read by q4g only (q4: one group per row)."""
    case = {"kind": "linear", "fmt": fmt, "m": m, "n": n, "k": k, "x": x, "y": y or x,
            "group": group if fmt == "q4g" else 0, "scale": scale if fmt == "q4g" else "f32", "bias": bias}
    return dict(case, name=name) if name else case


def listed():
    return [
        # The smallest: one decoded token through one MLP projection of a 0.5B model,
        # fp32 activations as the reference keeps them.
        linear("decode_q8_f32", "q8", 1, 4864, 896, x="f32"),
        # One decoded token through a 1.5B model's down projection, int4 groups of 32.
        linear("decode_q4g", "q4g", 1, 1536, 8960, scale="f16"),
        # Sixteen sequences decoded together through the gate / up projection.
        linear("batch_w8a8", "w8a8", 16, 8960, 1536),
        # The LM head of one decoded token: the largest weight a decode step reads.
        linear("lm_head", "q8", 1, 151936, 1536, y="f32"),
        # Sizes that are a multiple of nothing, as a model with odd dimensions has
        # them: a few rows, a bias, fp32 activations.
        linear("ragged_q8", "q8", 7, 1001, 1003, x="f32", bias=True),
        # The down projection over a short prompt in fp32, as the C++ decoder and the
        # reference run it, one row past whole tiles.
        linear("prompt_q8_f32", "q8", 333, 1536, 8960, x="f32"),
        # A long prompt through the gate / up projection, int8 activations.
        linear("prefill_w8a8", "w8a8", 2048, 8960, 1536),
        # The same with weight-only int4, the format that fits the most in memory.
        linear("prefill_q4g", "q4g", 2048, 8960, 1536, scale="f16"),
        # Loading a checkpoint: one fused gate|up weight to int4.
        {"name": "load_q4g", "kind": "quantize", "fmt": "q4g", "n": 17920, "k": 1536, "group": 32, "scale": "f16"},
        # One 1.5B decoder layer over a prompt.
        {"name": "block_512", "kind": "block", "s": 512, "x": "f16"},
        # The same over a few tokens, where launches count.
        {"name": "block_24", "kind": "block", "s": 24, "x": "f16"},
        # A prompt through the C++ decoder, two layers of 0.5B sizes.
        {"name": "decoder_q4g", "kind": "decoder", "fmt": "q4g", "s": 384},
    ]


# ---- drawn cases -----------------------------------------------------------------------

MAX_FLOPS = 2.0 * 2048 * 8960 * 1536


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A feature count: mostly multiples of 64 as models have them, else of 8, else any."""
    v, r = _log(rng, lo, hi), rng.random()
    step = 64 if r < 0.6 else 8 if r < 0.8 else 1
    return max(step, v // step * step)


def draw(rng):
    kind = rng.choices(["linear", "quantize", "block", "decoder"], [12, 2, 3, 3])[0]
    if kind == "linear":
        fmt = rng.choices(["q8", "q4g", "q4", "w8a8"], [4, 4, 1, 4])[0]
        n, k = _width(rng, 128, 18432), _width(rng, 128, 9216)
        if fmt == "q8" and rng.random() < 0.15:  # an LM head
            n = rng.randint(32000, 151936)
        m = _log(rng, 1, 2048)
        while 2.0 * m * n * k > MAX_FLOPS or n * k > 151936 * 1536:
            m, n, k = max(1, m // 2), n if m > 1 else n // 2, k
        x = rng.choice(["f32", "f16"])
        return linear(None, fmt, m, n, k, x=x, y=rng.choice([x, x, "f32"]),
                      group=rng.choice([32, 32, 64, 128]), scale=rng.choice(["f32", "f16"]), bias=rng.random() < 0.3)
    if kind == "quantize":
        fmt = rng.choice(["q8", "q4g"])
        return {"kind": kind, "fmt": fmt, "n": _width(rng, 256, 18432), "k": _width(rng, 256, 9216),
                "group": rng.choice([32, 64, 128]) if fmt == "q4g" else 0,
                "scale": rng.choice(["f32", "f16"]) if fmt == "q4g" else "f32"}
    if kind == "block":
        return {"kind": kind, "s": _log(rng, 2, 1024), "x": rng.choice(["f16", "f16", "f32"])}
    return {"kind": kind, "fmt": rng.choice(["q8", "q4g", "q4"]), "s": _log(rng, 2, 640)}


# ---- inputs ----------------------------------------------------------------------------

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device=DEV).mul_(std)


def _linear_inputs(case, seed):
    g = _gen(seed)
    w = _normal(g, case["n"], case["k"], std=0.02)
    x = _normal(g, case["m"], case["k"]).to(DTYPE[case["x"]])
    b = _normal(g, case["n"]) if case["bias"] else None
    return x, w, b


BLOCK = model.Config(hidden=1536, heads=12, kv_heads=2, head_dim=128, intermediate=8960, layers=1, vocab=128,
                     max_pos=1024)
DECODER = model.Config(hidden=896, heads=14, kv_heads=2, head_dim=64, intermediate=4864, layers=2, vocab=8192,
                       max_pos=1024)


def _weights(cfg, seed):
    """Random-init weights of a decoder under the exporter's names."""
    g = _gen(seed)
    w = {"embed_tokens.weight": _normal(g, cfg.vocab, cfg.hidden, std=0.02),
         "norm.weight": 1.0 + _normal(g, cfg.hidden, std=0.02)}
    for li in range(cfg.layers):
        L = f"layers.{li}."
        for p, (o, i) in model.proj_shapes(cfg).items():
            w[L + p + ".weight"] = _normal(g, o, i, std=0.02)
        for p in ("q_proj", "k_proj", "v_proj"):
            w[L + f"self_attn.{p}.bias"] = _normal(g, model.proj_shapes(cfg)[f"self_attn.{p}"][0], std=0.02)
        for p in ("input_layernorm", "post_attention_layernorm"):
            w[L + p + ".weight"] = 1.0 + _normal(g, cfg.hidden, std=0.02)
    return w


def _decoder_weights(seed):
    """Values that a bf16 checkpoint holds."""
    return {k: v.bfloat16().float() for k, v in _weights(DECODER, seed).items()}


def _ids(case, seed):
    r = np.random.default_rng(int(seed))
    return [int(t) for t in r.integers(0, DECODER.vocab, case["s"])]


def _write_checkpoint(path, cfg, weights):
    """config.txt and one bf16 NIT1 file per tensor."""
    fields = {"vocab_size": cfg.vocab, "hidden_size": cfg.hidden, "intermediate_size": cfg.intermediate,
              "num_layers": cfg.layers, "num_attention_heads": cfg.heads, "num_kv_heads": cfg.kv_heads,
              "head_dim": cfg.head_dim, "max_position_embeddings": cfg.max_pos, "rms_norm_eps": cfg.eps,
              "rope_theta": cfg.rope_theta, "tie_word_embeddings": 1, "eos_token_id": -1, "qkv_bias": 1}
    with open(os.path.join(path, "config.txt"), "w") as f:
        f.writelines(f"{k} {v}\n" for k, v in fields.items())
    for name, t in weights.items():
        with open(os.path.join(path, name + ".bin"), "wb") as f:
            f.write(b"NIT1" + np.int32([1, t.dim(), *t.shape]).tobytes())
            f.write(t.bfloat16().view(torch.int16).cpu().numpy().tobytes())


def prepare(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, b = _linear_inputs(case, seed)
        if case["fmt"] == "q4g":
            op, qw = quant.linear_q4g, quant.quantize_q4g(w, case["group"], DTYPE[case["scale"]])
        elif case["fmt"] == "q4":
            op, qw = quant.linear_q4, quant.quantize_q4(w)
        else:
            op, qw = (quant.linear_q8 if case["fmt"] == "q8" else quant.linear_w8a8), quant.quantize_q8(w)
        return {"kind": kind, "op": op, "x": x, "w": qw, "b": b, "y": DTYPE[case["y"]]}
    if kind == "quantize":
        return {"kind": kind, "case": case, "w": _normal(_gen(seed), case["n"], case["k"], std=0.02)}
    if kind == "block":
        dt = DTYPE[case["x"]]
        m = model.Model(BLOCK, _weights(BLOCK, seed), quant.QuantMode.W8A8, act_dtype=dt)
        return {"kind": kind, "model": m, "x": _normal(_gen(seed + 1000), case["s"], BLOCK.hidden).to(dt)}
    from nanoinfer_amd import nicpp
    path = tempfile.mkdtemp(prefix="decoder_")
    try:
        _write_checkpoint(path, DECODER, _decoder_weights(seed))
        m = nicpp.Model(path, nicpp.quant_mode(case["fmt"]), "hip")
    finally:
        shutil.rmtree(path)
    return {"kind": kind, "model": m, "ids": _ids(case, seed)}


def run(state):
    kind = state["kind"]
    if kind == "linear":
        return state["op"](state["x"], state["w"], state["b"], state["y"])
    if kind == "quantize":
        c = state["case"]
        q = quant.quantize_q8(state["w"]) if c["fmt"] == "q8" else quant.quantize_q4g(state["w"], c["group"],
                                                                                    DTYPE[c["scale"]])
        return {"codes": q.q, "scale": q.scale}
    if kind == "block":
        return state["model"].run_layers(state["x"])
    return state["model"].forward(state["ids"])


# ---- what a pass cannot do without -----------------------------------------------------

def _weight_bytes(fmt, n, k, group=32, scale="f32"):
    if fmt in ("q8", "w8a8"):
        return n * k + 4 * n
    g = k if fmt == "q4" else group
    return n * ((k + 1) // 2) + n * ((k + g - 1) // g) * (2 if scale == "f16" else 4)


def _size(dt):
    return 2 if dt == "f16" else 4


def _layer_flops(cfg, s):
    proj = sum(2.0 * s * o * i for o, i in model.proj_shapes(cfg).values())
    return proj + 4.0 * cfg.heads * cfg.head_dim * s * (s + 1) / 2


def work(case):
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        b = (_weight_bytes(case["fmt"], n, k, case["group"], case["scale"]) + m * k * _size(case["x"]) +
             m * n * _size(case["y"]) + (4 * n if case["bias"] else 0))
        return {"bytes": b, "flops": 2.0 * m * n * k}
    if kind == "quantize":
        return {"bytes": 4 * case["n"] * case["k"] +
                _weight_bytes(case["fmt"], case["n"], case["k"], case["group"], case["scale"]), "flops": 0}
    cfg, s = (BLOCK, case["s"]) if kind == "block" else (DECODER, case["s"])
    fmt = "w8a8" if kind == "block" else case["fmt"]
    b = cfg.layers * sum(_weight_bytes(fmt, o, i) for o, i in model.proj_shapes(cfg).values())
    if kind == "block":
        return {"bytes": b + 2 * s * cfg.hidden * _size(case["x"]), "flops": _layer_flops(cfg, s)}
    head = _weight_bytes("q8", cfg.vocab, cfg.hidden)
    return {"bytes": b + head + 4 * s * cfg.vocab,
            "flops": cfg.layers * _layer_flops(cfg, s) + 2.0 * s * cfg.vocab * cfg.hidden}


def tolerance(case):
    kind = case["kind"]
    if kind == "quantize":
        return "exact"
    if kind == "linear":
        return {"rel": 1e-5, "max": 1e-4} if case["y"] == "f32" else {"rel": 1e-3, "max": 5e-3}
    if kind == "block":
        return {"rel": 3e-2, "max": 0.5}  # each act quant can round a code the other way
    return {"rel": 1e-5, "max": 1e-4}


# ---- the same in 64 bits ---------------------------------------------------------------

def _div32(a, b):
    """The fp32 quotient of fp32 values, rounded once."""
    return (a.double() / b).float()


def _codes_q8(w):
    """Per row: scale = absmax / 127 in fp32, codes round-half-even of the fp32 quotient."""
    s = _div32(w.float().abs().amax(1), 127.0)
    q = torch.where(s[:, None] > 0, torch.round(_div32(w.float(), s[:, None])).clamp_(-127, 127), 0.0)
    return q, s


def _dequant_q4(w, group, scale):
    n, k = w.shape
    pad = (-k) % group
    v = torch.nn.functional.pad(w, (0, pad)).view(n, -1, group)
    s = _div32(v.abs().amax(2, keepdim=True), 7.0)
    q = torch.where(s > 0, torch.round(_div32(v, s)).clamp_(-7, 7), 0.0)
    return s.to(scale).squeeze(2), (q.double() * s.to(scale).double()).view(n, -1)[:, :k]


def _dequant(w, fmt, group=32, scale=torch.float32):
    if fmt in ("q8", "w8a8"):
        q, s = _codes_q8(w)
        return q.double() * s.double()[:, None]
    return _dequant_q4(w, w.shape[1] if fmt == "q4" else group, scale)[1]


def _linear64(x, w, b, fmt, group=32, scale=torch.float32):
    if fmt == "w8a8":
        q, s = _codes_q8(x)
        x = q.double() * s.double()[:, None]
    y = x.double() @ _dequant(w, fmt, group, scale).t()
    return y if b is None else y + b.double()


def _norm64(x, w, eps):
    return x * torch.rsqrt((x * x).mean(1, keepdim=True) + eps) * w.double()


def _attention64(cfg, q, k, v):
    s = q.shape[0]
    half = cfg.head_dim // 2
    inv = cfg.rope_theta ** (-torch.arange(half, device=DEV, dtype=torch.float64) * 2.0 / cfg.head_dim)
    ang = torch.arange(s, device=DEV, dtype=torch.float64)[:, None] * inv
    cos, sin = torch.cat([ang.cos()] * 2, 1), torch.cat([ang.sin()] * 2, 1)

    def heads(t, h, rope):
        t = t.reshape(s, h, cfg.head_dim).transpose(0, 1)
        if rope:
            t = t * cos + torch.cat([-t[..., half:], t[..., :half]], 2) * sin
        return t.repeat_interleave(cfg.heads // h, 0).contiguous()

    q, k, v = heads(q, cfg.heads, True), heads(k, cfg.kv_heads, True), heads(v, cfg.kv_heads, False)
    a = torch.empty_like(q)
    mask = torch.ones(s, s, dtype=torch.bool, device=DEV).triu(1)
    for h in range(cfg.heads):
        sc = (q[h] @ k[h].t().contiguous()) / math.sqrt(cfg.head_dim)
        a[h] = torch.softmax(sc.masked_fill(mask, -math.inf), 1) @ v[h]
    return a.transpose(0, 1).reshape(s, -1)


def _layers64(cfg, w, x, fmt):
    for li in range(cfg.layers):
        L = f"layers.{li}."

        def project(h, p):
            return _linear64(h, w[L + p + ".weight"], w.get(L + p + ".bias"), fmt)

        h = _norm64(x, w[L + "input_layernorm.weight"], cfg.eps)
        a = _attention64(cfg, *(project(h, f"self_attn.{p}_proj") for p in "qkv"))
        x = x + project(a, "self_attn.o_proj")
        h = _norm64(x, w[L + "post_attention_layernorm.weight"], cfg.eps)
        g = torch.nn.functional.silu(project(h, "mlp.gate_proj")) * project(h, "mlp.up_proj")
        x = x + project(g, "mlp.down_proj")
    return x


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, w, b = _linear_inputs(case, seed)
        return _linear64(x, w, b, case["fmt"], case["group"], DTYPE[case["scale"]])
    if kind == "quantize":
        w = _normal(_gen(seed), case["n"], case["k"], std=0.02)
        scale = _codes_q8(w)[1] if case["fmt"] == "q8" else _dequant_q4(w, case["group"], DTYPE[case["scale"]])[0]
        return {"codes": None, "scale": scale.double()}
    if kind == "block":
        x = _normal(_gen(seed + 1000), case["s"], BLOCK.hidden).to(DTYPE[case["x"]])
        return _layers64(BLOCK, _weights(BLOCK, seed), x.double(), "w8a8")
    w = _decoder_weights(seed)
    emb = _dequant(w["embed_tokens.weight"], "q8")
    x = _layers64(DECODER, w, emb[torch.tensor(_ids(case, seed), device=DEV)], case["fmt"])
    return _norm64(x, w["norm.weight"], DECODER.eps) @ emb.t()
