"""Performance cases: what a program that uses this framework has it do.

A case is a dict of plain values.  ``listed()`` names twelve of them, ``draw(rng)``
gives more of the same ranges, ``prepare`` makes what a user's program holds before
the call (weights, inputs, a decoding session), ``run`` is one pass through the
public entry points, ``work`` what a pass cannot do without, ``exact`` the same
result in float64 from plain torch.

The kinds of case, each over the models of ``GPTConfig``'s presets, 'medium'
(8 layers, d 512) and GPT-2 XL:

    forward     CutileGPT.forward: logits of a batch of prompts, or of one prompt
    decode      DecodeSession: prompt, then one KV-cache step for every given token
                (scoring a continuation; generate() drives the same calls)
    attention   cutile_causal_attention on (B, H, T, hd) tensors
    qkv         attention_qkv on the fused projection's output
    mlp         cutile_fused_mlp
    linear      cutile_linear (no bias: the LM head) / cutile_linear_bias
    layer_norm  cutile_layer_norm
    gelu        cutile_gelu
"""

from __future__ import annotations

import math

import torch
import torch.nn.functional as F

import cutilegpt_amd as cg
from cutilegpt_amd.decode import DecodeSession

_DTYPES = {"float32": torch.float32, "bfloat16": torch.bfloat16, "float16": torch.float16}

VOCAB = 50257

# (n_layer, n_head, n_embd, block_size): the presets, and the 'medium' of the benchmark.
MODELS = {
    "nano": (3, 3, 48, 128),
    "micro": (4, 4, 128, 256),
    "tile-medium": (6, 4, 128, 256),
    "mini": (6, 6, 192, 256),
    "tile-large": (8, 8, 256, 512),
    "medium": (8, 8, 512, 1024),
    "gpt2": (12, 12, 768, 1024),
    "gpt2-medium": (24, 16, 1024, 1024),
    "gpt2-large": (36, 20, 1280, 1024),
    "gpt2-xl": (48, 25, 1600, 1024),
}

# No drawn case costs more than this: the largest listed one (XL decode) in
# operations, a full-vocabulary forward in bytes moved.
MAX_FLOPS = 1.2e13
MAX_OUT_BYTES = 8.3e8


def listed():
    return [
        # A batch of full-context prompts through GPT-2 124M, every position's logits.
        dict(name="forward_batch", kind="forward", model="gpt2", dtype="bfloat16", B=4, T=1024),
        # One short prompt in the model's default dtype: a user at a prompt, launches count.
        dict(name="forward_prompt", kind="forward", model="gpt2", dtype="float32", B=1, T=87),
        # One sequence generated token by token after a half-context prompt.
        dict(name="decode_single", kind="decode", model="gpt2", dtype="bfloat16", B=1, T=500, new=24),
        # Batched serving: GPT-2 XL, 32 sequences after 128-token prompts.
        dict(name="decode_batch", kind="decode", model="gpt2-xl", dtype="bfloat16", B=32, T=128, new=16),
        # The attention of a full prefill batch, read straight from the projection.
        dict(name="attention_prefill", kind="qkv", dtype="bfloat16", B=16, H=12, T=1024, hd=64),
        # The attention kernel by itself in fp32, the reference's own benchmark shape.
        dict(name="attention_fp32", kind="attention", dtype="float32", B=8, H=12, T=512, hd=64),
        # An MLP block in the default dtype: 8 prompts of 512 tokens.
        dict(name="mlp_fp32", kind="mlp", dtype="float32", rows=4096, d=768),
        # GPT-2 XL's MLP block over the prompts of a decode batch.
        dict(name="mlp_xl", kind="mlp", dtype="bfloat16", rows=4096, d=1600),
        # The LM head on the vocabulary as checkpoints hold it (odd width, rows unpadded).
        dict(name="head_unpadded", kind="linear", dtype="bfloat16", rows=1000, n=VOCAB, d=768, bias=False),
        # A projection over three ragged prompts in fp16.
        dict(name="linear_ragged", kind="linear", dtype="float16", rows=591, n=2304, d=768, bias=True),
        # The normalisation of a full prefill batch.
        dict(name="layer_norm", kind="layer_norm", dtype="bfloat16", rows=16384, d=768),
        # The activation by itself, the reference's own benchmark shape.
        dict(name="gelu", kind="gelu", dtype="float32", rows=16384, d=768),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["forward", "forward", "decode", "decode", "attention", "qkv", "mlp", "mlp",
                       "linear", "linear", "layer_norm", "gelu"])
    while True:
        case = _draw_kind(rng, kind)
        if work(case)["flops"] <= MAX_FLOPS and _out_bytes(case) <= MAX_OUT_BYTES:
            return case


def _draw_kind(rng, kind):
    half = rng.choice(["bfloat16", "bfloat16", "float16"])
    drop_in = rng.choice(["float32", half])
    if kind in ("forward", "decode"):
        model = rng.choice(list(MODELS))
        block = MODELS[model][3]
        dtype = rng.choice(["float32", "bfloat16", "bfloat16"])
        if kind == "forward":
            T = _log_int(rng, 1, block)
            return dict(kind=kind, model=model, dtype=dtype, B=_log_int(rng, 1, 32), T=T)
        new = rng.randint(4, 24)
        return dict(kind=kind, model=model, dtype=dtype, B=_log_int(rng, 1, 64),
                    T=_log_int(rng, 4, block - new), new=new)
    if kind in ("attention", "qkv"):
        return dict(kind=kind, dtype=drop_in, B=_log_int(rng, 1, 32), H=rng.choice([3, 4, 6, 8, 12, 16, 20, 25]),
                    T=_log_int(rng, 1, 1024), hd=rng.choice([16, 32, 64, 64, 64]))
    d = rng.choice([m[2] for m in MODELS.values()])
    if kind == "mlp":
        return dict(kind=kind, dtype=drop_in, rows=_log_int(rng, 1, 16384), d=d)
    if kind == "linear":
        n, k = rng.choice([(3 * d, d), (d, d), (4 * d, d), (d, 4 * d), (VOCAB, d)])
        return dict(kind=kind, dtype=drop_in, rows=_log_int(rng, 1, 16384), n=n, d=k, bias=n != VOCAB)
    return dict(kind=kind, dtype=drop_in, rows=_log_int(rng, 1, 32768), d=d * (4 if kind == "gelu" else 1))


# ------------------------------------------------------------------- work


def _esize(case):
    return 4 if case["dtype"] == "float32" else 2


def _out_bytes(case):
    k = case["kind"]
    if k == "forward":
        return case["B"] * case["T"] * VOCAB * 4
    if k == "decode":
        return case["B"] * case["new"] * VOCAB * 4
    if k in ("attention", "qkv"):
        return case["B"] * case["H"] * case["T"] * case["hd"] * _esize(case)
    return case["rows"] * case.get("n", case["d"]) * _esize(case)


def work(case):
    """Each input read once, each output written once; causal attention counted as
    the half it is.  A decode pass reads the weights and the cache rows so far once
    a step (the prompt is a step of its own)."""
    k, e = case["kind"], _esize(case)
    if k in ("forward", "decode"):
        L, H, D, _ = MODELS[case["model"]]
        B, T = case["B"], case["T"]
        layers = 12 * L * D * D
        head = VOCAB * D
        attn = lambda t: 4 * L * D * t * (t + 1) // 2
        if k == "forward":
            flops = 2 * B * T * (layers + head) + B * attn(T)
            return {"bytes": (layers + head) * e + B * T * VOCAB * 4, "flops": flops}
        n = case["new"]
        S = T + n - 1
        flops = 2 * B * S * layers + 2 * B * n * head + B * attn(S)
        kv = sum(2 * L * D * B * (T + i) * e for i in range(n))
        return {"bytes": n * (layers + head) * e + kv + B * n * VOCAB * 4, "flops": flops}
    if k in ("attention", "qkv"):
        B, H, T, hd = case["B"], case["H"], case["T"], case["hd"]
        return {"bytes": 4 * B * H * T * hd * e, "flops": 4 * B * H * hd * T * (T + 1) // 2}
    r, d = case["rows"], case["d"]
    if k == "mlp":
        return {"bytes": (8 * d * d + 2 * r * d) * e, "flops": 16 * r * d * d}
    if k == "linear":
        n = case["n"]
        return {"bytes": (n * d + r * d + r * n) * e, "flops": 2 * r * n * d}
    return {"bytes": 2 * r * d * e, "flops": (8 if k == "layer_norm" else 12) * r * d}


# ----------------------------------------------------------------- inputs


class _Gen:
    """Seeded tensors on the GPU."""

    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(seed)

    def __call__(self, shape, dtype, std=1.0, mean=0.0):
        t = torch.empty(shape, dtype=torch.float32, device="cuda")
        return t.normal_(mean, std, generator=self.g).to(dtype)

    def tokens(self, shape):
        return torch.randint(0, VOCAB, shape, generator=self.g, device="cuda")


def _weights(case, gen):
    """Checkpoint-like parameters: GPT-2's initial scale for the matrices, biases
    and LayerNorm parameters that are neither zero nor one."""
    L, H, D, block = MODELS[case["model"]]
    dt = _DTYPES[case["dtype"]]
    proj = 0.02 / math.sqrt(2 * L)
    w = {"wte": gen((VOCAB, D), dt, 0.02), "wpe": gen((block, D), dt, 0.02)}
    for i in range(L):
        p = f"h.{i}."
        for ln in ("ln_1", "ln_2"):
            w[p + ln + ".weight"] = gen((D,), dt, 0.1, 1.0)
            w[p + ln + ".bias"] = gen((D,), dt, 0.1)
        for name, n, k, std in (("attn.c_attn", 3 * D, D, 0.02), ("attn.c_proj", D, D, proj),
                                ("mlp.c_fc", 4 * D, D, 0.02), ("mlp.c_proj", D, 4 * D, proj)):
            w[p + name + ".weight"] = gen((n, k), dt, std)
            w[p + name + ".bias"] = gen((n,), dt, 0.02)
    w["ln_f.weight"] = gen((D,), dt, 0.1, 1.0)
    w["ln_f.bias"] = gen((D,), dt, 0.1)
    return w


def _inputs(case, seed):
    gen = _Gen(seed)
    k = case["kind"]
    dt = _DTYPES[case["dtype"]]
    if k == "forward":
        return {"weights": _weights(case, gen), "idx": gen.tokens((case["B"], case["T"]))}
    if k == "decode":
        return {"weights": _weights(case, gen),
                "idx": gen.tokens((case["B"], case["T"] + case["new"] - 1))}
    if k == "attention":
        shape = (case["B"], case["H"], case["T"], case["hd"])
        return {n: gen(shape, dt) for n in "qkv"}
    if k == "qkv":
        return {"qkv": gen((case["B"], case["T"], 3 * case["H"] * case["hd"]), dt)}
    r, d = case["rows"], case["d"]
    x = gen((r, d), dt)
    if k == "mlp":
        return {"x": x, "w_fc": gen((4 * d, d), dt, 0.02), "b_fc": gen((4 * d,), dt, 0.02),
                "w_proj": gen((d, 4 * d), dt, 0.02), "b_proj": gen((d,), dt, 0.02)}
    if k == "linear":
        out = {"x": x, "w": gen((case["n"], d), dt, 0.02)}
        if case["bias"]:
            out["b"] = gen((case["n"],), dt, 0.02)
        return out
    if k == "layer_norm":
        return {"x": gen((r, d), dt, 2.0, 0.3), "w": gen((d,), dt, 0.1, 1.0), "b": gen((d,), dt, 0.1)}
    return {"x": x}


def prepare(case, seed):
    inp = _inputs(case, seed)
    if case["kind"] not in ("forward", "decode"):
        return {"case": case, **inp}
    L, H, D, block = MODELS[case["model"]]
    model = cg.CutileGPT(cg.GPTConfig(vocab_size=VOCAB, block_size=block, n_layer=L, n_head=H, n_embd=D),
                         dtype=_DTYPES[case["dtype"]], init_weights=False)
    model.load_weights(inp["weights"])
    state = {"case": case, "model": model, "idx": inp["idx"]}
    if case["kind"] == "decode":
        T = case["T"]
        state["prompt"] = inp["idx"][:, :T].contiguous()
        state["given"] = [inp["idx"][:, T + i].contiguous() for i in range(case["new"] - 1)]
        sess = DecodeSession(model, case["B"], T, case["new"])
        # A program keeps its session and the step it captured over its generations.
        sess.prefill(state["prompt"])
        sess.step.zero_()
        sess.next_logits()
        state["session"] = sess
    return state


def run(state):
    case = state["case"]
    k = case["kind"]
    if k == "forward":
        return state["model"](state["idx"])[0]
    if k == "decode":
        sess = state["session"]
        sess.prefill(state["prompt"])
        out = [sess.logits.clone()]
        sess.step.zero_()
        for tokens in state["given"]:
            sess.ids.copy_(tokens)
            sess.next_logits()
            sess.step.add_(1)
            out.append(sess.logits.clone())
        return torch.stack(out, 1)
    if k == "attention":
        return cg.cutile_causal_attention(state["q"], state["k"], state["v"], case["H"])
    if k == "qkv":
        return cg.attention_qkv(state["qkv"], case["H"])
    if k == "mlp":
        return cg.cutile_fused_mlp(state["x"], state["w_fc"], state["b_fc"], state["w_proj"], state["b_proj"])
    if k == "linear":
        if case["bias"]:
            return cg.cutile_linear_bias(state["x"], state["w"], state["b"])
        return cg.cutile_linear(state["x"], state["w"])
    if k == "layer_norm":
        return cg.cutile_layer_norm(state["x"], state["w"], state["b"])
    return cg.cutile_gelu(state["x"])


# ------------------------------------------------------------------ exact


def _attention64(q, k, v):
    """Causal attention of (B, H, T, hd) float64 tensors, a few sequences at a time."""
    T, hd = q.shape[2], q.shape[3]
    dead = torch.ones(T, T, dtype=torch.bool, device=q.device).triu_(1)
    out = torch.empty_like(q)
    for b in range(q.shape[0]):
        s = (q[b] @ k[b].transpose(1, 2).contiguous()) / math.sqrt(hd)
        out[b] = torch.softmax(s.masked_fill_(dead, float("-inf")), -1) @ v[b]
    return out


def _heads(x, B, T, H):
    return x.view(B, T, H, -1).transpose(1, 2).contiguous()


def _hidden64(case, w, idx):
    """Final LayerNorm output (B, T, D) of the model in float64."""
    L, H, D, _ = MODELS[case["model"]]
    B, T = idx.shape
    W = lambda k: w[k].double()
    ln = lambda x, k: F.layer_norm(x, (D,), W(k + ".weight"), W(k + ".bias"), 1e-5)
    lin = lambda x, k: F.linear(x, W(k + ".weight"), W(k + ".bias"))
    x = (w["wte"][idx].double() + w["wpe"][:T].double()).view(B * T, D)
    for i in range(L):
        p = f"h.{i}."
        q, k, v = (_heads(t, B, T, H) for t in lin(ln(x, p + "ln_1"), p + "attn.c_attn").split(D, 1))
        a = _attention64(q, k, v).transpose(1, 2).reshape(B * T, D)
        x = x + lin(a, p + "attn.c_proj")
        f = F.gelu(lin(ln(x, p + "ln_2"), p + "mlp.c_fc"), approximate="tanh")
        x = x + lin(f, p + "mlp.c_proj")
    return ln(x, "ln_f").view(B, T, D)


@torch.no_grad()
def exact(case, seed):
    inp = _inputs(case, seed)
    k = case["kind"]
    if k == "forward":
        return _hidden64(case, inp["weights"], inp["idx"]) @ inp["weights"]["wte"].double().t()
    if k == "decode":
        h = _hidden64(case, inp["weights"], inp["idx"])
        return h[:, case["T"] - 1:] @ inp["weights"]["wte"].double().t()
    if k == "attention":
        return _attention64(inp["q"].double(), inp["k"].double(), inp["v"].double())
    if k == "qkv":
        B, T, H = case["B"], case["T"], case["H"]
        q, kk, v = (_heads(t, B, T, H) for t in inp["qkv"].double().chunk(3, 2))
        return _attention64(q, kk, v).transpose(1, 2).reshape(B, T, -1)
    x = inp["x"].double()
    if k == "mlp":
        h = F.gelu(F.linear(x, inp["w_fc"].double(), inp["b_fc"].double()), approximate="tanh")
        return F.linear(h, inp["w_proj"].double(), inp["b_proj"].double())
    if k == "linear":
        return F.linear(x, inp["w"].double(), inp["b"].double() if case["bias"] else None)
    if k == "layer_norm":
        return F.layer_norm(x, (case["d"],), inp["w"].double(), inp["b"].double(), 1e-5)
    return F.gelu(x, approximate="tanh")


# About four times what the paths differ from float64 by, measured over the listed
# cases and forty drawn ones: (2-norm, largest difference over the result's root mean
# square).  The float32 figures are those of the longest sums (K = 6400, 48 layers);
# the 16-bit ones are the rounding of the outputs and, for models, of every layer.
_TOL = {
    "forward": {"float32": (8e-6, 6e-5), "bfloat16": (1.8e-2, 0.12)},
    "decode": {"float32": (8e-6, 6e-5), "bfloat16": (1.8e-2, 0.12)},
    "attention": {"float32": (2e-6, 4e-5), "bfloat16": (8e-3, 8e-2), "float16": (1e-3, 1e-2)},
    "mlp": {"float32": (8e-6, 6e-5), "bfloat16": (9e-3, 4e-2), "float16": (1.2e-3, 6e-3)},
    "linear": {"float32": (8e-6, 6e-5), "bfloat16": (7e-3, 1.6e-2), "float16": (9e-4, 2e-3)},
    "layer_norm": {"float32": (4e-7, 4e-6), "bfloat16": (7e-3, 1.6e-2), "float16": (9e-4, 2e-3)},
    "gelu": {"float32": (3e-7, 2e-6), "bfloat16": (7e-3, 1.6e-2), "float16": (9e-4, 2e-3)},
}


def tolerance(case):
    kind = "attention" if case["kind"] == "qkv" else case["kind"]
    rel, most = _TOL[kind][case["dtype"]]
    return {"rel": rel, "max": most}
