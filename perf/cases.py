"""The framework's work in use, as a list of cases: its primitives through the C ABI (include/rai_hip.h) and its decoders
through rai_amd.models.Decoder, from the smallest call to a long prompt, forward prefill and step-by-step decoding, bf16,
f16 and f32.  Sizes are those of the models the decoders serve (Phi-2, Qwen2-1.5B, Gemma-2B, Bezadra layers), of the
primitive sweep, and odd ones between them.

A case is a dict of plain values.  Its `kind` is one of
  linear     act(x W^T + bias) + residual                       rai_hip_linear
  matmul     batched product, right operand as it lies ([K, N]) or as a transposed view of [N, K]     rai_hip_matmul
  attention  causal scaled-dot-product attention, grouped query heads                          rai_hip_attention
  rows       a norm or a softmax over the last axis              rai_hip_layer_norm / rms_norm / softmax
  model      a request: prompt, greedy tokens, and the logits behind the last of them           rai_hip_decoder_*
"""
import math

import numpy as np
import torch

from rai_amd._lib import BF16, F16, F32, UNARY, call
from rai_amd.hip import HipTensor, sync
from rai_amd.models import Decoder

DTYPE = {"bf16": (BF16, torch.bfloat16, 2), "f16": (F16, torch.float16, 2), "f32": (F32, torch.float32, 4)}
VOCAB = 32768


def listed():
    return [
        # The MLP projection of a Phi-2 prefill: large product, bias and activation.
        dict(name="linear_bf16_mlp", kind="linear", dtype="bf16", m=4096, k=2560, n=10240, act="new_gelu", bias=True, residual=False),
        # An o_proj-like product of a short, odd prompt: few rows, bias-free, residual added.
        dict(name="linear_bf16_ragged", kind="linear", dtype="bf16", m=333, k=1536, n=8960, act="", bias=False, residual=True),
        # The same projection in f32, rai's default element type.
        dict(name="linear_f32_mlp", kind="linear", dtype="f32", m=1024, k=2560, n=10240, act="new_gelu", bias=True, residual=False),
        # Scores of 32 heads as a program that builds its own attention out of primitives writes them: Q K^T, K a view.
        dict(name="matmul_bf16_scores", kind="matmul", dtype="bf16", batch=32, m=512, k=80, n=512, b_t=True),
        # Attention of one Qwen2-1.5B layer over 16 prompts.
        dict(name="attention_bf16_gqa", kind="attention", dtype="bf16", batch=16, heads=12, kv_heads=2, s=1024, t=1024, dim=128, f32_scores=False),
        # Attention of one Phi-2 layer in f32 over an odd prompt.
        dict(name="attention_f32_mha", kind="attention", dtype="f32", batch=1, heads=32, kv_heads=32, s=333, t=333, dim=80, f32_scores=True),
        # The smallest call: the norm of a decoding step's single row.
        dict(name="rms_norm_row", kind="rows", op="rms_norm", dtype="bf16", rows=1, cols=1536),
        # One Phi-2 layer in f32: a 128-token prompt and eight tokens.
        model("phi2_f32_layer", "phi2", "f32", 2560, layers=1, batch=1, prompt=128, new=8),
        # A chat turn: 512-token prompt, 32 tokens, one sequence.
        model("phi2_bf16_turn", "phi2", "bf16", 2560, layers=4, batch=1, prompt=512, new=32),
        # Prompt processing of a full batch (scoring, embedding, the first token of many requests).
        model("qwen2_bf16_prefill", "qwen2", "bf16", 1536, layers=4, batch=16, prompt=1024, new=0),
        # Batched serving: 24 short prompts decoded together.
        model("gemma_bf16_batch", "gemma", "bf16", 2048, layers=4, batch=24, prompt=50, new=32),
        # A hybrid decoder: attention and delta-rule layers, three of them looped; odd prompt.
        model("bezadra_bf16_mixed", "bezadra", "bf16", 2048, layers=4, batch=1, prompt=777, new=16),
    ]


def model(name, arch, dtype, width, layers, batch, prompt, new):
    c = dict(name=name) if name else {}
    c.update(kind="model", arch=arch, dtype=dtype, width=width, layers=layers, batch=batch, prompt=prompt, new=new)
    return c


# (heads, key/value heads, head width, MLP width) by family and width
SHAPES = {
    ("phi2", 2560): (32, 32, 80, 10240), ("phi2", 2048): (32, 32, 64, 8192),
    ("qwen2", 1024): (8, 8, 128, 4096), ("qwen2", 1536): (12, 2, 128, 8960), ("qwen2", 2048): (16, 16, 128, 8192),
    ("gemma", 2048): (8, 1, 256, 16384),
    ("bezadra", 1024): (8, 8, 128, 4096), ("bezadra", 2048): (16, 16, 128, 8192),
}
MOST_FLOPS = 4e12  # a drawn case's work; the largest listed one has over 6e12


def _log(rng, lo, hi):
    """A whole number, even over the logarithm of the range."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    while True:
        c = _draw(rng)
        if work(c)["flops"] <= MOST_FLOPS * (1 if c["dtype"] != "f32" else 0.02):
            return c


def _draw(rng):
    kind = rng.choice(["linear", "linear", "matmul", "attention", "rows", "model", "model", "model"])
    if kind == "linear":
        dt = rng.choice(["bf16", "bf16", "f32"])
        return dict(kind=kind, dtype=dt, m=_log(rng, 1, 8192), k=32 * _log(rng, 8, 320), n=8 * _log(rng, 32, 2048),
                    act=rng.choice(["", "", "new_gelu", "silu", "gelu"]), bias=rng.random() < 0.5, residual=rng.random() < 0.3)
    if kind == "matmul":
        dt = rng.choice(["bf16", "bf16", "f32", "f16"])
        return dict(kind=kind, dtype=dt, batch=_log(rng, 2, 64), m=_log(rng, 1, 1024), k=_log(rng, 16, 1024), n=_log(rng, 16, 1024),
                    b_t=rng.random() < 0.5)
    if kind == "attention":
        kv = rng.choice([1, 2, 4, 8, 32])
        s = _log(rng, 1, 1024)
        return dict(kind=kind, dtype=rng.choice(["bf16", "bf16", "f32"]), batch=_log(rng, 1, 8), heads=kv * rng.choice([1, 1, 4, 6]) if kv < 32 else 32,
                    kv_heads=kv, s=s, t=s + (0 if rng.random() < 0.6 else _log(rng, 1, 1024)), dim=rng.choice([64, 80, 128, 256]),
                    f32_scores=rng.random() < 0.5)
    if kind == "rows":
        return dict(kind=kind, op=rng.choice(["layer_norm", "rms_norm", "softmax"]), dtype=rng.choice(["bf16", "f32"]),
                    rows=_log(rng, 1, 8192), cols=_log(rng, 64, 4096))
    arch, width = rng.choice(sorted(SHAPES))
    dt = "f32" if arch in ("phi2", "qwen2") and rng.random() < 0.3 else "bf16"
    return model(None, arch, dt, width, layers=4 if arch == "bezadra" else rng.randint(1, 4), batch=_log(rng, 1, 32), prompt=_log(rng, 1, 1024),
                 new=rng.choice([0, _log(rng, 1, 32), _log(rng, 1, 32)]))


# ------------------------------------------------------------------ inputs
class _Borrowed:
    """The memory of a torch tensor as a HipTensor's buffer."""

    def __init__(self, t):
        self.t, self.ptr, self.dev = t, t.data_ptr(), 0


def _tensor(t):
    return HipTensor(_Borrowed(t), {torch.bfloat16: BF16, torch.float16: F16, torch.float32: F32}[t.dtype], t.shape)


def _values(case, seed):
    """Inputs of a primitive in its element type: activations N(0, 1), weights scaled by their fan-in."""
    g = torch.Generator("cuda").manual_seed(int(seed) * 1000003 + 17)
    dt = DTYPE[case["dtype"]][1]

    def normal(*shape, std=1.0):
        return (torch.randn(shape, generator=g, device="cuda") * std).to(dt)

    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(x=normal(m, k), w=normal(n, k, std=k ** -0.5), bias=normal(n, std=0.1) if case["bias"] else None,
                    residual=normal(m, n) if case["residual"] else None)
    if kind == "matmul":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        return dict(a=normal(b, m, k), b=normal(b, n, k) if case["b_t"] else normal(b, k, n))
    if kind == "attention":
        b, d = case["batch"], case["dim"]
        return dict(q=normal(b, case["heads"], case["s"], d), k=normal(b, case["kv_heads"], case["t"], d), v=normal(b, case["kv_heads"], case["t"], d))
    x = normal(case["rows"], case["cols"], std=2.0)
    if case["op"] == "softmax":
        return dict(x=x)
    w = (1 + 0.1 * torch.randn(case["cols"], generator=g, device="cuda")).to(dt)
    return dict(x=x, w=w, b=normal(case["cols"], std=0.1) if case["op"] == "layer_norm" else None)


def _out_shape(case):
    kind = case["kind"]
    if kind == "linear":
        return case["m"], case["n"]
    if kind == "matmul":
        return case["batch"], case["m"], case["n"]
    if kind == "attention":
        return case["batch"], case["s"], case["heads"] * case["dim"]
    return case["rows"], case["cols"]


def _param_shapes(case):
    """Parameter name -> shape, as the decoder of this family names them."""
    h, L = case["width"], case["layers"]
    heads, kvh, hd, ff = SHAPES[case["arch"], h]
    qd, kd, out = heads * hd, kvh * hd, {}
    if case["arch"] == "bezadra":
        out.update({"embed": (VOCAB, h), "loop.in": (h, 2 * h), "loop.step": (2, h)})
        for i in range(L):
            p = f"l{i}."
            out[p + "norm1"] = (h,)
            out.update({p + "mix.q": (qd, h), p + "mix.k": (kd, h), p + "mix.v": (kd, h), p + "mix.o": (h, qd)})
            if i == 0:
                out.update({p + "mix.sink": (heads,), p + "mix.g": (qd, h)})
            else:
                out.update({p + f"mix.{c}.conv": (qd, 4) for c in "qkv"})
                out.update({p + "mix.b": (heads, h), p + "mix.A_log": (heads,), p + "mix.norm": (hd,), p + "mix.a1": (128, h), p + "mix.a2": (qd, 128),
                            p + "mix.dt_bias": (qd,), p + "mix.g1": (128, h), p + "mix.g2": (qd, 128)})
            out.update({p + "mlp.gate": (ff, h), p + "mlp.up": (ff, h), p + "mlp.down": (h, ff)})
        out["final.norm"] = (h,)
        return out
    out["model.embed_tokens.weight"] = (VOCAB, h)
    for i in range(L):
        p = f"model.layers.{i}."
        for name, rows, cols in (("q_proj", qd, h), ("k_proj", kd, h), ("v_proj", kd, h), ("dense" if case["arch"] == "phi2" else "o_proj", h, qd)):
            out[p + f"self_attn.{name}.weight"] = (rows, cols)
            if case["arch"] == "phi2" or (case["arch"] == "qwen2" and name != "o_proj"):
                out[p + f"self_attn.{name}.bias"] = (rows,)
        if case["arch"] == "phi2":
            out.update({p + "mlp.fc1.weight": (ff, h), p + "mlp.fc1.bias": (ff,), p + "mlp.fc2.weight": (h, ff), p + "mlp.fc2.bias": (h,),
                        p + "input_layernorm.weight": (h,), p + "input_layernorm.bias": (h,)})
        else:
            out.update({p + "mlp.gate_proj.weight": (ff, h), p + "mlp.up_proj.weight": (ff, h), p + "mlp.down_proj.weight": (h, ff),
                        p + "input_layernorm.weight": (h,), p + "post_attention_layernorm.weight": (h,)})
    if case["arch"] == "phi2":
        out.update({"model.final_layernorm.weight": (h,), "model.final_layernorm.bias": (h,)})
    else:
        out["model.norm.weight"] = (h,)
    return out


def _params(case, seed):
    """Random weights on the GPU, in the model's element type.  Matrices N(0, 0.02); embedding rows, which also are the
    head (tied), large enough beside the layers' contributions that a greedy choice has no near ties."""
    g = torch.Generator("cuda").manual_seed(int(seed) * 1000003 + 29)
    dt = DTYPE[case["dtype"]][1]
    for name, shape in _param_shapes(case).items():
        a = torch.randn(shape, generator=g, device="cuda")
        last = name.rsplit(".", 1)[-1]
        if "embed" in name:
            a *= 0.02 if case["arch"] == "gemma" else 1.0  # Gemma scales its embeddings by sqrt(width)
        elif last in ("norm", "norm1") or name.endswith("norm.weight"):
            a = 0.1 * a + (0.0 if case["arch"] == "gemma" else 1.0)
        elif last == "A_log":
            a *= 0.5
        elif last == "dt_bias":
            a = 1.5 * a - 3.0
        elif last == "conv":
            a *= 0.5
        elif name == "loop.in":
            h = shape[0]
            a *= 0.005
            a[:, :h] += 0.7 * torch.eye(h, device="cuda")
            a[:, h:] += 0.3 * torch.eye(h, device="cuda")
        elif last != "sink":
            a *= 0.02
        yield name, a.to(dt)


def _decoder(case):
    h, L = case["width"], case["layers"]
    heads, kvh, hd, ff = SHAPES[case["arch"], h]
    room = dict(max_batch=case["batch"], max_context=case["prompt"] + case["new"] + 1)
    if case["arch"] == "bezadra":
        mlp = dict(mlp_kind="dense", intermediate=ff, mlp_limit=7.0, mlp_alpha=1.702)
        attn = dict(mixer="attention", heads=heads, kv_heads=kvh, qk_dim=hd, v_dim=hd, rot_dims=hd, rot_base=5e5, rot_factor=8.0, rot_low=1.0,
                    rot_high=4.0, rot_original=8192, attn_scale=hd ** -0.5, softcap=30.0, **mlp)
        delta = dict(mixer="channel_delta", heads=heads, kv_heads=kvh, qk_dim=hd, v_dim=hd, conv_taps=4, decay_rank=128, gate_rank=128, **mlp)
        return Decoder.hybrid(case["dtype"], vocab_size=VOCAB, width=h, layers=[attn] + [delta] * (L - 1), norm_eps=1e-6, loop=(1, L, 2), **room)
    return Decoder(case["arch"], case["dtype"], vocab_size=VOCAB, hidden_size=h, intermediate_size=ff, num_hidden_layers=L,
                   num_attention_heads=heads, num_key_value_heads=kvh, head_dim=hd, rotary_dim=int(0.4 * hd) if case["arch"] == "phi2" else hd,
                   max_position_embeddings=2048, hidden_act={"phi2": "gelu_new", "qwen2": "silu", "gemma": "gelu"}[case["arch"]],
                   tie_word_embeddings=True, norm_eps=1e-5 if case["arch"] == "phi2" else 1e-6, **room)


def _prompt(case, seed):
    return np.random.Generator(np.random.PCG64(int(seed))).integers(0, VOCAB, (case["batch"], case["prompt"])).astype(np.uint32)


def prepare(case, seed):
    if case["kind"] == "model":
        dec = _decoder(case)
        for name, a in _params(case, seed):
            dec.load_param(name, (a.view(torch.int16) if a.dtype == torch.bfloat16 else a).cpu().numpy())
        sync()
        return dict(case=case, dec=dec, prompt=_prompt(case, seed))
    # A program that keeps its tensors: inputs and the output on the GPU, and their descriptors.
    values = _values(case, seed)
    out = torch.empty(_out_shape(case), dtype=DTYPE[case["dtype"]][1], device="cuda")
    call("rai_hip_init", 0)
    desc = {n: None if t is None else _tensor(t).desc() for n, t in values.items()}
    if case["kind"] == "matmul" and case["b_t"]:
        desc["b"] = _tensor(values["b"]).transpose(1, 2).desc()
    torch.cuda.synchronize()
    return dict(case=case, values=values, out=out, desc=desc, out_desc=_tensor(out).desc(), eps=1e-5)


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "model":
        dec = state["dec"]
        if case["new"] == 0:
            dec.clear_kv_cache()
            logits, tokens = dec.forward(state["prompt"])
        else:
            tokens, _, _ = dec.generate(state["prompt"], case["new"])
            logits, _ = dec.forward(tokens[:, -1:])
        return dict(tokens=tokens, logits=logits)
    d, o = state["desc"], state["out_desc"]
    if kind == "linear":
        call("rai_hip_linear", 0, d["x"], d["w"], d["bias"], UNARY[case["act"]] if case["act"] else -1, d["residual"], o)
    elif kind == "matmul":
        call("rai_hip_matmul", 0, d["a"], d["b"], o)
    elif kind == "attention":
        call("rai_hip_attention", 0, d["q"], d["k"], d["v"], case["dim"] ** -0.5, 1, int(case["f32_scores"]), o)
    elif case["op"] == "layer_norm":
        call("rai_hip_layer_norm", 0, d["x"], d["w"], d["b"], state["eps"], o)
    elif case["op"] == "rms_norm":
        call("rai_hip_rms_norm", 0, d["x"], d["w"], state["eps"], 0, o)
    else:
        call("rai_hip_softmax", 0, d["x"], 1, o)
    return state["out"]


# ------------------------------------------------------------------ what a pass cannot do without
def work(case):
    es = DTYPE[case["dtype"]][2]
    kind = case["kind"]
    if kind == "linear":
        m, k, n = case["m"], case["k"], case["n"]
        return dict(bytes=es * (m * k + n * k + m * n * (2 if case["residual"] else 1) + (n if case["bias"] else 0)), flops=2.0 * m * k * n)
    if kind == "matmul":
        b, m, k, n = case["batch"], case["m"], case["k"], case["n"]
        return dict(bytes=es * b * (m * k + k * n + m * n), flops=2.0 * b * m * k * n)
    if kind == "attention":
        b, h, s, t, d = case["batch"], case["heads"], case["s"], case["t"], case["dim"]
        seen = s * (t - s) + s * (s + 1) / 2.0
        return dict(bytes=es * b * d * (2 * h * s + 2 * case["kv_heads"] * t), flops=4.0 * b * h * seen * d)
    if kind == "rows":
        return dict(bytes=es * case["rows"] * case["cols"] * 2, flops=8.0 * case["rows"] * case["cols"])
    heads, kvh, hd, ff = SHAPES[case["arch"], case["width"]]
    h, qd, kd, L = case["width"], heads * hd, kvh * hd, case["layers"]
    b, p, new = case["batch"], case["prompt"], case["new"]
    params = sum(math.prod(s) for n, s in _param_shapes(case).items() if "embed" not in n)
    runs = [(params / L, 1)] * L  # (weights of a layer, whether it holds keys)
    if case["arch"] == "bezadra":
        runs = [(params / L, 1)] + [(params / L, 0)] * (2 * (L - 1))
    keys = sum(k for _, k in runs)
    calls = 1 + new                                  # the prompt, then one token at a time
    # a looped layer's weights are read once a call: the passes follow one another
    weights = calls * (params + VOCAB * h) * es
    cached = sum(2 * kd * (p + i) for i in range(1, new + 1)) * keys * b * es + 2 * kd * (p + new) * keys * b * es
    tokens = b * (p + new)
    seen = b * ((p + new) * (p + new + 1) / 2.0)
    flops = 2.0 * tokens * sum(w for w, _ in runs) + 4.0 * seen * qd * keys + 2.0 * b * calls * VOCAB * h
    return dict(bytes=weights + cached + tokens * h * es + 4 * b * VOCAB, flops=flops)


# ------------------------------------------------------------------ how far another correct implementation may be off
# Measured against 64 bits: f32 products 1e-6, f32 models 2e-6, bf16 primitives 0.002 to 0.0044 (attention), bf16 models
# 0.005 to 0.011.
def tolerance(case):
    if case["kind"] == "model":
        return {"rel": 1e-5, "differ": 0.0} if case["dtype"] == "f32" else {"rel": 0.03, "differ": 0.0}
    if case["dtype"] == "f32":
        return {"rel": 5e-6}
    return {"rel": 8e-3, "max": 0.1}


# ------------------------------------------------------------------ the same in 64 bits
def _act(name, x):
    if name == "new_gelu":
        return 0.5 * x * (1 + torch.tanh(math.sqrt(2 / math.pi) * (x + 0.044715 * x ** 3)))
    if name == "gelu":
        return 0.5 * x * (1 + torch.erf(x / math.sqrt(2)))
    return x * torch.sigmoid(x) if name == "silu" else x


def _attend(q, k, v, scale, cap=0.0, sink=None):
    """q [b, h, s, d], k and v [b, kv, t, d]: the last s of t positions, causal."""
    b, h, s, d = q.shape
    t, out = k.shape[2], torch.empty_like(q)
    see = torch.arange(t, device=q.device)[None, :] <= torch.arange(t - s, t, device=q.device)[:, None]
    for i in range(h):
        j = i // (h // k.shape[1])
        w = q[:, i] @ k[:, j].transpose(1, 2).contiguous() * scale
        if cap:
            w = cap * torch.tanh(w / cap)
        w = w.masked_fill(~see, -math.inf)
        if sink is not None:
            w = torch.cat([w, sink[i].expand(b, s, 1)], 2)
        out[:, i] = torch.softmax(w, 2)[..., :t] @ v[:, j]
    return out


def exact(case, seed):
    if case["kind"] == "model":
        return _exact_model(case, seed)
    v = {n: None if t is None else t.double() for n, t in _values(case, seed).items()}
    kind = case["kind"]
    if kind == "linear":
        y = v["x"] @ v["w"].T
        y = _act(case["act"], y if v["bias"] is None else y + v["bias"])
        return y if v["residual"] is None else y + v["residual"]
    if kind == "matmul":
        return v["a"] @ (v["b"].transpose(1, 2).contiguous() if case["b_t"] else v["b"])
    if kind == "attention":
        y = _attend(v["q"], v["k"], v["v"], case["dim"] ** -0.5)
        return y.transpose(1, 2).reshape(_out_shape(case))
    if case["op"] == "softmax":
        return torch.softmax(v["x"], 1)
    return _norm(v["x"], v["w"], v["b"], 1e-5, case["op"] == "layer_norm")


def _norm(x, w, b, eps, centre):
    if centre:
        x = x - x.mean(-1, keepdim=True)
    y = x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w
    return y if b is None else y + b


def _turn(x, angle, table):
    """x [b, h, s, d]: features i and i + len(angle[0]) turned by angle [s, n]; `table` rounds cosines and sines."""
    n = angle.shape[1]
    c, s = table(torch.cos(angle)), table(torch.sin(angle))
    u, v = x[..., :n], x[..., n:2 * n]
    return torch.cat([u * c - v * s, v * c + u * s, x[..., 2 * n:]], -1)


def _angles(case, length, dims):
    """Rotary angles as these families define them: in the model's element type, positions and products rounded to it."""
    dt = DTYPE[case["dtype"]][1]
    inv = torch.tensor([1.0 / 10000.0 ** (2 * i / dims) for i in range(dims // 2)], dtype=torch.float32, device="cuda").to(dt)
    pos = torch.arange(length, device="cuda").float().to(dt)
    return (pos.float()[:, None] * inv.float()[None, :]).to(dt).double()


def _exact_model(case, seed):
    p = dict(_params(case, seed))
    prompt = torch.from_numpy(_prompt(case, seed).astype(np.int64)).cuda()
    new, n = case["new"], case["prompt"]
    layers = _bezadra if case["arch"] == "bezadra" else _decoder_layers
    table = p["embed" if case["arch"] == "bezadra" else "model.embed_tokens.weight"].double()
    # Guess that the last token repeats (see _params), evaluate the whole sequence at once and put right what was wrong.
    tokens = prompt[:, -1:].repeat(1, max(1, new))
    while True:
        ids = torch.cat([prompt, tokens[:, :new]], 1)
        logits = layers(case, p, table[ids])[:, n - 1:] @ table.T
        chosen = logits[:, :max(1, new)].argmax(-1)
        wrong = (chosen != tokens).any(0).nonzero()
        if not len(wrong):
            return dict(tokens=tokens.cpu().numpy().astype(np.uint32), logits=logits[:, -1].float().cpu().numpy())
        at = int(wrong[0])
        tokens[:, at:] = chosen[:, at:at + 1]


def _heads(x, n):
    return x.reshape(x.shape[0], x.shape[1], n, -1).transpose(1, 2)


def _decoder_layers(case, p, x):
    """Phi-2 (parallel block, layer norm), Qwen2 and Gemma (sequential block, RMS norm): the normed last hidden rows."""
    arch, (heads, kvh, hd, _) = case["arch"], SHAPES[case["arch"], case["width"]]
    eps = 1e-5 if arch == "phi2" else 1e-6
    if arch == "gemma":
        x = x * math.sqrt(case["width"])
    dt = DTYPE[case["dtype"]][1]
    angle = _angles(case, x.shape[1], int(0.4 * hd) if arch == "phi2" else hd)

    def lin(name, h):
        y = h @ p[name + ".weight"].double().T
        return y + p[name + ".bias"].double() if name + ".bias" in p else y

    def norm(name, h):
        w = p[name + ".weight"].double()
        return _norm(h, 1 + w if arch == "gemma" else w, p[name + ".bias"].double() if arch == "phi2" else None, eps, arch == "phi2")

    for i in range(case["layers"]):
        pre = f"model.layers.{i}."
        h = norm(pre + "input_layernorm", x)
        q, k, v = (_heads(lin(pre + f"self_attn.{c}_proj", h), n) for c, n in (("q", heads), ("k", kvh), ("v", kvh)))
        rounded = lambda t: t.to(dt).double()  # noqa: E731
        y = _attend(_turn(q, angle, rounded), _turn(k, angle, rounded), v, hd ** -0.5).transpose(1, 2).reshape(x.shape[0], x.shape[1], -1)
        if arch == "phi2":
            x = x + lin(pre + "self_attn.dense", y) + lin(pre + "mlp.fc2", _act("new_gelu", lin(pre + "mlp.fc1", h)))
            continue
        x = x + lin(pre + "self_attn.o_proj", y)
        h = norm(pre + "post_attention_layernorm", x)
        x = x + lin(pre + "mlp.down_proj", _act("silu" if arch == "qwen2" else "gelu", lin(pre + "mlp.gate_proj", h)) * lin(pre + "mlp.up_proj", h))
    return norm("model.final_layernorm" if arch == "phi2" else "model.norm", x)


def _bezadra(case, p, x):
    heads, kvh, hd, _ = SHAPES[case["arch"], case["width"]]
    L, (B, T, H) = case["layers"], x.shape
    w = lambda name: p[name].double()  # noqa: E731
    norm = lambda h, name: _norm(h, w(name), None, 1e-6, True)  # noqa: E731
    f = 5e5 ** (-2.0 * torch.arange(hd // 2, device="cuda", dtype=torch.float64) / hd)
    blend = ((8192 * f / (2 * math.pi) - 1.0) / 3.0).clamp(0, 1)   # waves between 8192 and 8192 / 4 positions long
    angle = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * ((1 - blend) * f / 8.0 + blend * f)

    def attention(h, q):
        a, k, v = (_heads(h @ w(q + c).T, n) for c, n in (("q", heads), ("k", kvh), ("v", kvh)))
        y = _attend(_turn(a, angle, lambda t: t), _turn(k, angle, lambda t: t), v, hd ** -0.5, 30.0, w(q + "sink"))
        return (y.transpose(1, 2).reshape(B, T, -1) * torch.sigmoid(h @ w(q + "g").T)) @ w(q + "o").T

    def delta(h, q):
        def conv(c):
            y, taps = torch.nn.functional.pad(h @ w(q + c).T, (0, 0, 3, 0)), w(q + c + ".conv")
            return _heads(_act("silu", sum(y[:, j:j + T] * taps[:, j] for j in range(4))), heads)

        unit = lambda t: t / torch.sqrt(t.square().sum(-1, keepdim=True) + 1e-6)  # noqa: E731
        a, k, v = unit(conv("q")) * hd ** -0.5, unit(conv("k")), conv("v")
        step = torch.nn.functional.softplus((h @ w(q + "a1").T) @ w(q + "a2").T + w(q + "dt_bias"), threshold=1e9)
        g = torch.exp(-torch.exp(w(q + "A_log"))[:, None, None] * _heads(step, heads))
        beta = torch.sigmoid(h @ w(q + "b").T).transpose(1, 2)
        S, out = torch.zeros(B, heads, hd, hd, device="cuda", dtype=torch.float64), torch.empty_like(v)
        for t in range(T):
            S = g[:, :, t, :, None] * S
            u = beta[:, :, t, None] * (v[:, :, t] - (S * k[:, :, t, :, None]).sum(2))
            S = S + k[:, :, t, :, None] * u[:, :, None, :]
            out[:, :, t] = (S * a[:, :, t, :, None]).sum(2)
        y = out / torch.sqrt(out.square().mean(-1, keepdim=True) + 1e-6) * w(q + "norm")
        y = y.transpose(1, 2).reshape(B, T, -1) * torch.sigmoid((h @ w(q + "g1").T) @ w(q + "g2").T)
        return y @ w(q + "o").T

    def layer(x, i):
        h, q = norm(x, f"l{i}.norm1"), f"l{i}."
        a, b = (h @ w(q + "mlp.gate").T).clamp(max=7.0), (h @ w(q + "mlp.up").T).clamp(-7.0, 7.0)
        return x + (attention if i == 0 else delta)(h, q + "mix.") + (a * torch.sigmoid(1.702 * a) * (b + 1)) @ w(q + "mlp.down").T

    x0 = x
    x = layer(x, 0)
    for t in range(2):
        x = torch.cat([x, x0], -1) @ w("loop.in").T + w("loop.step")[t]
        for i in range(1, L):
            x = layer(x, i)
    return norm(x, "final.norm")
