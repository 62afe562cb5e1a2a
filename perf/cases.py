"""Performance cases: the work a user of this framework has it do.

Five kinds, each through a public entry point of velomind_hip (the Python
binding of include/vm_hip.h and include/vm_llama.h):

  qmm                Op::QuantizedMatMul: activations [m, k] times INT8 or
                     INT4 weights [k, n].  m = 1..4 is decode, more rows are
                     prompts and batched decode.
  pack               the weight packers, run over every linear at load time.
  attention          FusedAttention on contiguous q, k, v, as the graph
                     engine runs it.
  attention_prefill  causal attention over the resident decoder's KV cache.
  llama              whole calls of the resident decoder.

Inputs and expected values are made with torch alone.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import numpy as np
import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "velo-mind_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

import velomind_hip as H  # noqa: E402
from velomind_hip import llama as L  # noqa: E402

DEV = "cuda"
_TORCH = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_CODE = {"f32": H.DTYPE_F32, "f16": H.DTYPE_F16, "bf16": H.DTYPE_BF16}
_BYTES = {"f32": 4, "f16": 2, "bf16": 2}

# Architectures of this repository's end-to-end benchmark.
TINYLLAMA = dict(vocab=32000, hidden=2048, inter=5632, layers=22, heads=32, kv_heads=4, theta=10000.0)
SMOLLM2 = dict(vocab=49152, hidden=960, inter=2560, layers=32, heads=15, kv_heads=5, theta=100000.0)


def _qmm(name, dtype, quant, block, m, k, n, half_scale=False):
    return dict(name=name, kind="qmm", dtype=dtype, half_scale=half_scale, quant=quant, block=block, m=m, k=k, n=n)


def listed():
    return [
        # The smallest call in use: one INT8 projection of one decode token.
        _qmm("qmm_int8_m1_576x1536", "f32", 8, 0, 1, 576, 1536),
        # TinyLlama's gate (or up) projection of one decode token, the shape
        # that takes the most time of an INT4 decode step.
        _qmm("qmm_int4_m1_2048x5632", "f32", 4, 32, 1, 2048, 5632),
        # The same projection of a 70B-class model: bandwidth, not latency.
        _qmm("qmm_int4_m1_8192x28672", "f32", 4, 32, 1, 8192, 28672),
        # Batched decode of 16 sequences.
        _qmm("qmm_int4_m16_2048x5632", "f32", 4, 32, 16, 2048, 5632),
        # A 512-token prompt, INT8 per column.
        _qmm("qmm_int8_m512_2048x5632", "f32", 8, 0, 512, 2048, 5632),
        # TinyLlama's down projection with bfloat16 activations and outputs,
        # a prompt whose length is no multiple of a tile.
        _qmm("qmm_int4_bf16_m333_5632x2048", "bf16", 4, 32, 333, 5632, 2048),
        # A vocabulary with three tokens added by a fine-tune: the logits of
        # eight positions, an output width that is no multiple of anything.
        _qmm("qmm_int8_m8_2048x32003", "f32", 8, 0, 8, 2048, 32003),
        # Packing TinyLlama's lm_head at load time.
        dict(name="pack_int4_2048x32000", kind="pack", quant=4, block=32, k=2048, n=32000),
        # One layer's attention of a 512-token TinyLlama prompt, resident cache.
        dict(name="attention_prefill_512", kind="attention_prefill", rows=512, past=0, heads=32, kv_heads=4),
        # One layer's FusedAttention of a 512-token SmolLM2 prompt.
        dict(name="attention_512x512", kind="attention", batch=1, heads=15, kv_heads=5, sq=512, sk=512, d=64),
        # A 512-token TinyLlama INT4 prompt, whole model: logits.
        dict(name="llama_int4_prefill_512", kind="llama", quant=4, block=32, prompt=512, steps=0, **TINYLLAMA),
        # SmolLM2 INT8: a 128-token prompt and 32 greedy tokens, then the
        # logits of one more step.
        dict(name="llama_int8_generate_32", kind="llama", quant=8, block=0, prompt=128, steps=32, **SMOLLM2),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _size(rng, lo, hi, multiple):
    """Log-uniform size; one in four is any integer, the rest multiples."""
    v = _log(rng, lo, hi)
    return v if rng.random() < 0.25 else max(multiple, v // multiple * multiple)


def draw(rng):
    kind = rng.choice(["qmm"] * 6 + ["pack", "attention", "attention_prefill", "llama"])
    if kind == "qmm":
        m = _log(rng, 1, 8) if rng.random() < 0.4 else _log(rng, 5, 1024)
        quant = rng.choice([4, 8])
        block = rng.choice([32, 32, 64, 128]) if quant == 4 else rng.choice([0, 0, 0, 128])
        dtype = rng.choice(["f32", "f32", "f16", "bf16"])
        hi_n = 32768 if m <= 64 else 12288
        c = _qmm("", dtype, quant, block, m, _size(rng, 256, 8192, 32), _size(rng, 256, hi_n, 16),
                 dtype != "f32" and rng.random() < 0.5)
        del c["name"]
        return c
    if kind == "pack":
        quant = rng.choice([4, 8])
        return dict(kind="pack", quant=quant, block=rng.choice([32, 64, 128]) if quant == 4 else 0,
                    k=_size(rng, 256, 8192, 32), n=_size(rng, 256, 32768, 16))
    kv_heads = rng.choice([1, 2, 4, 5, 8])
    heads = kv_heads * rng.choice([1, 2, 3, 4, 8])
    if kind == "attention":
        sq = 1 if rng.random() < 0.3 else _log(rng, 5, 1024)
        sk = sq + (_log(rng, 16, 2048) if sq == 1 or rng.random() < 0.3 else 0)
        return dict(kind="attention", batch=rng.choice([1, 1, 2]), heads=heads, kv_heads=kv_heads, sq=sq, sk=sk,
                    d=rng.choice([64, 128]))
    if kind == "attention_prefill":
        return dict(kind="attention_prefill", rows=_log(rng, 5, 1536), past=rng.choice([0, 0, _log(rng, 1, 1024)]),
                    heads=heads, kv_heads=kv_heads)
    heads = rng.choice([9, 12, 15, 16])
    quant = rng.choice([4, 8])
    return dict(kind="llama", quant=quant, block=rng.choice([32, 64]) if quant == 4 else 0,
                prompt=_log(rng, 5, 500), steps=rng.choice([0, _log(rng, 2, 16)]), vocab=_log(rng, 2000, 32000) // 16 * 16,
                hidden=heads * 64, inter=rng.choice([1536, 2560, 4096]), layers=rng.randint(2, 8), heads=heads,
                kv_heads=rng.choice([h for h in (3, 4, 5) if heads % h == 0]), theta=10000.0)


# ---- inputs -----------------------------------------------------------------

def _gen(seed, salt=0):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed * 1009 + salt)
    return g


def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _quantize(w, quant, block):
    """quant.cpp's symmetric packing of w [k, n]: (codes, scales, code values)."""
    k, n = w.shape
    top = 7.0 if quant == 4 else 127.0
    low = -8.0 if quant == 4 else -127.0
    b = block if block > 0 else k
    nb = -(-k // b)
    pad = torch.zeros(nb * b, n, device=DEV)
    pad[:k] = w
    pad = pad.view(nb, b, n)
    amax = pad.abs().amax(1)
    one = torch.ones_like(amax)
    # tensor by tensor: torch divides by a Python number as a product with its
    # reciprocal, which moves codes that lie at a half
    s = torch.where(amax > 0, amax / (one * top), one)
    x = (pad * (one / s)[:, None]).view(nb * b, n)[:k]
    v = (torch.trunc(x.abs().double() + 0.5) * x.sign()).clamp_(low, top).to(torch.int8)
    if quant == 8:
        return v, s, v
    if k % 2:
        v = torch.cat([v, torch.zeros(1, n, device=DEV, dtype=torch.int8)])
    packed = (v[0::2] & 15) | (v[1::2] << 4)
    return packed.contiguous(), s, v[:k]


def _dense(values, scales, block):
    k = values.shape[0]
    b = block if block > 0 else k
    return values.double() * scales.double().repeat_interleave(b, 0)[:k]


def _qmm_inputs(case, seed):
    g = _gen(seed)
    w = _randn(g, case["k"], case["n"]) * 0.02
    codes, scales, values = _quantize(w, case["quant"], case["block"])
    a = _randn(g, case["m"], case["k"]).to(_TORCH[case["dtype"]])
    if case["half_scale"]:
        scales = scales.to(_TORCH[case["dtype"]])
    return a, codes, scales, values


def _attention_inputs(case, seed):
    g = _gen(seed)
    b, hq, hk, d = case["batch"], case["heads"], case["kv_heads"], case["d"]
    return (_randn(g, b, hq, case["sq"], d), _randn(g, b, hk, case["sk"], d), _randn(g, b, hk, case["sk"], d))


def _attention_prefill_inputs(case, seed):
    g = _gen(seed)
    total = case["past"] + case["rows"]
    # q carries 1/sqrt(head_dim), as the model loaders fold it into q_proj
    return (_randn(g, case["heads"], case["rows"], 64) * 0.125, _randn(g, case["kv_heads"], total, 64),
            _randn(g, case["kv_heads"], total, 64))


class _Config:
    """The fields that velomind_hip.llama reads from a model config."""

    def __init__(self, case):
        self.vocab_size, self.hidden_size, self.intermediate_size = case["vocab"], case["hidden"], case["inter"]
        self.num_layers, self.num_heads, self.num_kv_heads = case["layers"], case["heads"], case["kv_heads"]
        self.rms_norm_eps, self.rope_theta = 1e-5, case["theta"]


def _llama_weights(case, seed):
    """(kind, layer, fp32 tensor) of every weight in the graph's layout."""
    h, i, v = case["hidden"], case["inter"], case["vocab"]
    kv = h // case["heads"] * case["kv_heads"]
    g = _gen(seed)
    yield L.W_EMBED, 0, _randn(g, v, h) * 0.02
    yield L.W_FINAL_NORM, 0, 1 + 0.02 * _randn(g, h)
    yield L.W_LM_HEAD, 0, _randn(g, h, v) * 0.02
    for layer in range(case["layers"]):
        yield L.W_ATTN_NORM, layer, 1 + 0.02 * _randn(g, h)
        yield L.W_FFN_NORM, layer, 1 + 0.02 * _randn(g, h)
        yield L.W_Q, layer, _randn(g, h, h) * (0.02 * 0.125)
        for kind, rows, cols in ((L.W_K, h, kv), (L.W_V, h, kv), (L.W_O, h, h), (L.W_GATE, h, i), (L.W_UP, h, i),
                                 (L.W_DOWN, i, h)):
            yield kind, layer, _randn(g, rows, cols) * 0.02


def _prompt(case, seed):
    return np.random.default_rng(seed).integers(0, case["vocab"], case["prompt"]).astype(np.int32)


# ---- the calls --------------------------------------------------------------

def prepare(case, seed):
    H.load()
    kind = case["kind"]
    if kind == "qmm":
        a, codes, scales, _ = _qmm_inputs(case, seed)
        out = torch.empty(case["m"], case["n"], device=DEV, dtype=a.dtype)
        return dict(case=case, a=a, codes=codes, scales=scales, out=out)
    if kind == "pack":
        k, n, quant = case["k"], case["n"], case["quant"]
        w = _randn(_gen(seed), k, n) * 0.02
        codes = torch.empty((k + 1) // 2 if quant == 4 else k, n, device=DEV, dtype=torch.int8)
        blocks = -(-k // case["block"]) if quant == 4 else 1
        return dict(case=case, w=w, codes=codes, scales=torch.empty(blocks, n, device=DEV))
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        return dict(case=case, q=q, k=k, v=v, out=torch.empty_like(q))
    if kind == "attention_prefill":
        q, k, v = _attention_prefill_inputs(case, seed)
        pos = torch.tensor([case["past"]], device=DEV, dtype=torch.int32)
        return dict(case=case, q=q, k=k, v=v, pos=pos, out=torch.empty(case["rows"], case["heads"] * 64, device=DEV))
    cfg = _Config(case)
    weights = L.Weights(cfg)
    for what, layer, t in _llama_weights(case, seed):
        weights.set(what, layer, t.cpu().numpy())
    packed = L.PackedWeights.pack(weights, H.QUANT_INT4 if case["quant"] == 4 else H.QUANT_INT8, case["block"])
    session = L.Session.from_packed(packed, case["prompt"] + case["steps"] + 2)
    return dict(case=case, session=session, prompt=_prompt(case, seed))


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "qmm":
        a, codes, scales, out = state["a"], state["codes"], state["scales"], state["out"]
        quant = H.QUANT_INT4 if case["quant"] == 4 else H.QUANT_INT8
        m, k, n, block = case["m"], case["k"], case["n"], case["block"]
        if case["dtype"] == "f32":
            H.qmm_f32(a.data_ptr(), codes.data_ptr(), scales.data_ptr(), out.data_ptr(), m, k, n, quant, block)
        else:
            code = _CODE[case["dtype"]]
            H.qmm(a.data_ptr(), code, codes.data_ptr(), scales.data_ptr(), code if case["half_scale"] else H.DTYPE_F32,
                  out.data_ptr(), code, m, k, n, quant, block)
        return out
    if kind == "pack":
        w, codes, scales = state["w"], state["codes"], state["scales"]
        if case["quant"] == 4:
            H.pack_int4(w.data_ptr(), codes.data_ptr(), scales.data_ptr(), case["k"], case["n"], case["block"])
        else:
            H.pack_int8(w.data_ptr(), codes.data_ptr(), scales.data_ptr(), case["k"], case["n"])
        return {"codes": codes, "scales": scales}
    if kind == "attention":
        q, k, v, out = state["q"], state["k"], state["v"], state["out"]
        H.check(H.open_library().vm_hip_attention_f32(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), out.data_ptr(), case["batch"], case["heads"], case["kv_heads"],
            case["sq"], case["sk"], case["d"], case["d"], ctypes.c_float(0.0), 1, None))
        return out
    if kind == "attention_prefill":
        q, k, v, pos, out = state["q"], state["k"], state["v"], state["pos"], state["out"]
        H.check(H.open_library().vm_hip_attention_prefill_f32(
            q.data_ptr(), k.data_ptr(), v.data_ptr(), pos.data_ptr(), out.data_ptr(), case["rows"], case["heads"],
            case["kv_heads"], 64, case["past"] + case["rows"], ctypes.c_float(1.0), None))
        return out
    session, prompt, steps = state["session"], state["prompt"], case["steps"]
    if not steps:
        return {"logits": session.prefill(prompt)}
    tokens, _ = session.generate(prompt, steps)
    return {"logits": session.forward_step(int(tokens[-1]), len(prompt) + steps), "tokens": tokens}


# ---- what a pass cannot do without ------------------------------------------

def _weight_bytes(k, n, quant, block, scale_bytes=4):
    codes = (k + 1) // 2 * n if quant == 4 else k * n
    return codes + (-(-k // block) if block > 0 else 1) * n * scale_bytes


def work(case):
    kind = case["kind"]
    if kind == "qmm":
        m, k, n, e = case["m"], case["k"], case["n"], _BYTES[case["dtype"]]
        weights = _weight_bytes(k, n, case["quant"], case["block"], e if case["half_scale"] else 4)
        return {"bytes": weights + e * m * (k + n), "flops": 2 * m * k * n}
    if kind == "pack":
        k, n = case["k"], case["n"]
        return {"bytes": 4 * k * n + _weight_bytes(k, n, case["quant"], case["block"]), "flops": 3 * k * n}
    if kind in ("attention", "attention_prefill"):
        if kind == "attention":
            b, sq, sk, d = case["batch"], case["sq"], case["sk"], case["d"]
        else:
            b, sq, sk, d = 1, case["rows"], case["past"] + case["rows"], 64
        seen = sq * (sk - sq) + sq * (sq + 1) // 2  # visible (query, key) pairs of a head
        hq, hk = case["heads"], case["kv_heads"]
        return {"bytes": 4 * b * d * (2 * hq * sq + 2 * hk * sk), "flops": 4 * b * hq * seen * d}
    h, i, v, layers = case["hidden"], case["inter"], case["vocab"], case["layers"]
    kv = h // case["heads"] * case["kv_heads"]
    linears = [(h, h + 2 * kv), (h, h), (h, 2 * i), (i, h)]
    q, b = case["quant"], case["block"]
    layer_bytes = sum(_weight_bytes(r, c, q, b) for r, c in linears)
    macs = layers * sum(r * c for r, c in linears)
    rows, steps = case["prompt"], case["steps"] + 1 if case["steps"] else 0
    once = layers * layer_bytes + _weight_bytes(h, v, q, b)
    attn = 4 * layers * h * (rows * (rows + 1) // 2 + sum(rows + s + 1 for s in range(steps)))
    kv_bytes = 8 * layers * kv * (rows + sum(rows + s + 1 for s in range(steps)))
    return {"bytes": once * (1 + steps) + kv_bytes + 4 * h * rows + 4 * v,
            "flops": 2 * macs * (rows + steps) + 2 * h * v * (1 + steps) + attn}


def tolerance(case):
    kind = case["kind"]
    if kind == "pack":
        return "exact"
    if kind == "qmm" and case["dtype"] == "bf16":
        return {"rel": 7e-3}  # outputs rounded to 8 bits
    if kind == "qmm" and case["dtype"] == "f16":
        return {"rel": 8e-4}  # outputs rounded to 11 bits
    if kind == "llama":
        return {"rel": 2e-5, "differ": 0.01}  # 4e-6 from 64 bits after 22 layers
    return {"rel": 4e-6, "max": 1e-4}  # 32-bit sums, up to 8e-7 from 64 bits


# ---- the same in 64 bits ----------------------------------------------------

def _attend(q, k, v, scale):
    """q [b, hq, sq, d] over k, v [b, hk, sk, d]: causal, grouped heads."""
    rep = q.shape[1] // k.shape[1]
    k, v = k.repeat_interleave(rep, 1), v.repeat_interleave(rep, 1)
    sq, sk = q.shape[2], k.shape[2]
    s = torch.matmul(q * scale, k.transpose(2, 3).contiguous())
    hidden = torch.arange(sk, device=DEV)[None, :] > torch.arange(sq, device=DEV)[:, None] + (sk - sq)
    return torch.matmul(torch.softmax(s.masked_fill(hidden, -math.inf), -1), v)


def _norm(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w


def _rope(x, first, theta):
    """x [heads, rows, 64]; angles in 32 bits, as the rotary tables define them."""
    half = x.shape[-1] // 2
    inv = np.float32(1) / np.power(np.float32(theta), np.arange(half, dtype=np.float32) * 2 / np.float32(2 * half))
    t = np.arange(first, first + x.shape[1], dtype=np.float32)
    angle = torch.from_numpy((t[:, None] * inv.astype(np.float32)[None, :]).astype(np.float64)).to(DEV)
    c, s = torch.cos(angle), torch.sin(angle)
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _exact_llama(case, seed):
    linear = {L.W_LM_HEAD, L.W_Q, L.W_K, L.W_V, L.W_O, L.W_GATE, L.W_UP, L.W_DOWN}
    w = {}
    for kind, layer, t in _llama_weights(case, seed):
        if kind in linear:
            _, scales, values = _quantize(t, case["quant"], case["block"])
            w[kind, layer] = _dense(values, scales, case["block"])
        else:
            w[kind, layer] = t.double()
    heads, kv_heads, theta = case["heads"], case["kv_heads"], case["theta"]
    cache = [None] * case["layers"]

    def forward(tokens, first):
        h = w[L.W_EMBED, 0][torch.as_tensor(tokens, device=DEV, dtype=torch.long)]
        rows = h.shape[0]
        for layer in range(case["layers"]):
            x = _norm(h, w[L.W_ATTN_NORM, layer])
            q = (x @ w[L.W_Q, layer]).view(rows, heads, 64).transpose(0, 1)
            k = (x @ w[L.W_K, layer]).view(rows, kv_heads, 64).transpose(0, 1)
            v = (x @ w[L.W_V, layer]).view(rows, kv_heads, 64).transpose(0, 1)
            q, k = _rope(q, first, theta), _rope(k, first, theta)
            if cache[layer] is not None:
                k, v = torch.cat([cache[layer][0], k], 1), torch.cat([cache[layer][1], v], 1)
            cache[layer] = (k, v)
            ctx = _attend(q[None], k[None], v[None], 1.0)[0]
            h = h + ctx.transpose(0, 1).reshape(rows, -1) @ w[L.W_O, layer]
            x = _norm(h, w[L.W_FFN_NORM, layer])
            gate = x @ w[L.W_GATE, layer]
            h = h + (torch.sigmoid(gate) * gate * (x @ w[L.W_UP, layer])) @ w[L.W_DOWN, layer]
        return _norm(h[-1], w[L.W_FINAL_NORM, 0]) @ w[L.W_LM_HEAD, 0]

    prompt = _prompt(case, seed)
    logits = forward(prompt, 0)
    if not case["steps"]:
        return {"logits": logits}
    tokens = [int(logits.argmax())]
    for s in range(case["steps"]):
        tokens.append(int(forward(tokens[-1:], len(prompt) + s).argmax()))
    return {"logits": forward(tokens[-1:], len(prompt) + case["steps"]), "tokens": np.array(tokens, np.int32)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "qmm":
        a, _, scales, values = _qmm_inputs(case, seed)
        return a.double() @ _dense(values, scales, case["block"])
    if kind == "pack":
        k, n, quant = case["k"], case["n"], case["quant"]
        w = (_randn(_gen(seed), k, n) * 0.02).double()
        b = case["block"] if quant == 4 else k
        amax = torch.stack([p.abs().amax(0) for p in w.split(b)])
        return {"codes": None, "scales": torch.where(amax > 0, amax / (7.0 if quant == 4 else 127.0), 1.0)}
    if kind == "attention":
        q, k, v = _attention_inputs(case, seed)
        return _attend(q.double(), k.double(), v.double(), 1.0 / math.sqrt(case["d"]))
    if kind == "attention_prefill":
        q, k, v = _attention_prefill_inputs(case, seed)
        ctx = _attend(q[None].double(), k[None].double(), v[None].double(), 1.0)[0]
        return ctx.transpose(0, 1).reshape(case["rows"], -1)
    return _exact_llama(case, seed)
