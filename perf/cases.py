"""The work this library does for a program that runs a quantized Llama on it, as timed cases.

Every case is one call (or the calls of one step) through the public entry points of memvanta_amd.capi:
  matvec    y = W . x for one token: Context.matvec (device buffers, or host arrays as an application that keeps
            its activations on the host passes them)
  matmul    a prefill chunk against one weight: Context.matmul_batch_v06, in the default numerics (fp32
            activations) or with Q8 activations
  attend    one layer's attention over the paged cache: KVCache.write of the new rows, then attn_decode (one
            token) or attn_batch (a prefill chunk)
  prefill   Model.reset + Model.prefill of a prompt, logits of its last token
  request   Model.reset, prefill of a prompt, then greedy decoding: what serving one request does
Shapes are those of the three model configurations in memvanta_amd/synth.py (the 7B, TinyLlama-1.1B and 288-wide
shapes); the whole models are those shapes with fewer layers, so that one can be written and opened in a second.
"""
from __future__ import annotations

import dataclasses
import math
import os
import tempfile

import numpy as np
import torch

from memvanta_amd import capi, synth

TYPES = {"q4_0": synth.Q4_0, "q8_0": synth.Q8_0, "q6_k": synth.Q6_K}
BLOCK = {"q4_0": (32, 18), "q8_0": (32, 34), "q6_k": (256, 210)}
KV = {"f32": capi.MVH_KV_F32, "f16": capi.MVH_KV_F16, "q8": capi.MVH_KV_Q8}
ACT = {"ref": capi.MVH_ACT_REF, "q8": capi.MVH_ACT_Q8}
SHAPES = {"7b": synth.LLAMA7B, "1.1b": synth.TINYLLAMA_MIXED, "288": synth.TINY}


def listed():
    return [
        # decode, the smallest launch of a 7B layer: the attention output projection
        {"name": "matvec_q4_0_4096x4096", "kind": "matvec", "type": "q4_0", "k": 4096, "n": 4096, "host": False},
        # decode, the output head of both large shapes' vocabularies (Q6_K)
        {"name": "matvec_q6_k_4096x32000", "kind": "matvec", "type": "q6_k", "k": 4096, "n": 32000, "host": False},
        # decode, the TinyLlama shape's feed-forward up projection (Q8_0)
        {"name": "matvec_q8_0_2048x5632", "kind": "matvec", "type": "q8_0", "k": 2048, "n": 5632, "host": False},
        # an application whose activations are host vectors, calling tensor by tensor
        {"name": "matvec_host_q4_0_4096x11008", "kind": "matvec", "type": "q4_0", "k": 4096, "n": 11008, "host": True},
        # one 32-token prefill chunk against a 7B feed-forward weight, default numerics
        {"name": "matmul_q4_0_ref_m32", "kind": "matmul", "type": "q4_0", "act": "ref", "k": 4096, "n": 11008, "m": 32,
         "ffn": True},
        # the same chunk with Q8 activations, down projection
        {"name": "matmul_q4_0_q8_m32", "kind": "matmul", "type": "q4_0", "act": "q8", "k": 11008, "n": 4096, "m": 32,
         "ffn": True},
        # a prompt taken as one batch
        {"name": "matmul_q4_0_q8_m512", "kind": "matmul", "type": "q4_0", "act": "q8", "k": 4096, "n": 4096, "m": 512,
         "ffn": False},
        # the ragged last chunk of a prompt on the TinyLlama shape: tokens left over by the 8-token blocking
        {"name": "matmul_q8_0_ref_m77", "kind": "matmul", "type": "q8_0", "act": "ref", "k": 2048, "n": 5632, "m": 77,
         "ffn": True},
        # decode attention far into a conversation, 7B heads, fp16 pages
        {"name": "attend_decode_f16_pos1500", "kind": "attend", "kv": "f16", "heads": 32, "kv_heads": 32, "hd": 128,
         "pos": 1500, "tokens": 1, "page": 128},
        # a prefill chunk's attention at the end of a 512-token prompt
        {"name": "attend_chunk_f16_pos480", "kind": "attend", "kv": "f16", "heads": 32, "kv_heads": 32, "hd": 128,
         "pos": 480, "tokens": 32, "page": 128},
        # a prompt through the TinyLlama shape, default numerics, chunks of 32
        {"name": "prefill_1.1b_ref_512", "kind": "prefill", "shape": "1.1b", "layers": 8, "act": "ref", "kv": "f16",
         "prompt": 512, "batch": 32, "gen": 0},
        # one served request on the 7B shape: 128 prompt tokens, 64 greedy ones
        {"name": "request_7b_q8_128_64", "kind": "request", "shape": "7b", "layers": 4, "act": "q8", "kv": "f16",
         "prompt": 128, "batch": 32, "gen": 64},
    ]


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    """One more case: the same calls over the whole range of weights, batches, positions, cache types and options."""
    kind = rng.choice(["matvec", "matvec", "matmul", "matmul", "matmul", "attend", "attend", "attend", "prefill",
                       "request"])
    if kind in ("matvec", "matmul"):
        ty = rng.choice(["q4_0", "q4_0", "q8_0", "q6_k"])
        unit = 256 if ty == "q6_k" else rng.choice([32, 256])  # Q4_0 / Q8_0 rows need whole 32-element blocks only
        k = min(11008 // unit, max(1, round(_log(rng, 256, 11008) / unit))) * unit
        n = round(_log(rng, 64, 32000))
        if kind == "matvec":
            return {"kind": kind, "type": ty, "k": k, "n": n, "host": rng.random() < 0.25}
        m = round(_log(rng, 2, 512))
        return {"kind": kind, "type": ty, "act": rng.choice(["ref", "q8"]), "k": k, "n": min(n, 11008), "m": m,
                "ffn": rng.random() < 0.5}
    kv = rng.choice(["f16", "f16", "f32", "q8"])
    if kind == "attend":
        heads, kv_heads, hd = rng.choice([(32, 32, 128), (32, 4, 64), (32, 8, 128), (6, 6, 48)])
        tokens = rng.choice([1, 1, round(_log(rng, 2, 128))])
        return {"kind": kind, "kv": kv, "heads": heads, "kv_heads": kv_heads, "hd": hd,
                "pos": round(_log(rng, 1, 4000 if tokens == 1 else 1900)), "tokens": tokens,
                "page": rng.choice([16, 128])}
    prompt = round(_log(rng, 8, 512))
    return {"kind": kind, "shape": rng.choice(["7b", "1.1b", "288"]), "layers": rng.choice([1, 2, 3]),
            "act": rng.choice(["ref", "q8"]), "kv": kv, "prompt": prompt, "batch": rng.choice([8, 32, 32, 64]),
            "gen": round(_log(rng, 4, 60)) if kind == "request" else 0}


# ---- inputs -------------------------------------------------------------------------------------------------

def _gen(seed, salt=0):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000003 * int(seed) + salt)
    return g


def _weight(case, seed):
    """Block bytes of N(0, 0.02) weights, [n][row bytes]."""
    w = torch.randn((case["n"], case["k"]), generator=_gen(seed, 1), device="cuda") * 0.02
    return synth.quantize_torch(TYPES[case["type"]], w).contiguous()


def _activations(m, k, seed, salt):
    """N(0, 1) with one element in a thousand at +-20, as transformer activations have outliers."""
    g = _gen(seed, salt)
    x = torch.randn((m, k), generator=g, device="cuda")
    far = torch.rand((m, k), generator=g, device="cuda") < 0.001
    return torch.where(far, torch.where(x < 0, -20.0, 20.0), x).contiguous()


def _cache_rows(case, seed):
    kv_dim, n = case["kv_heads"] * case["hd"], case["pos"] + case["tokens"]
    g = _gen(seed, 3)
    k = torch.randn((n, kv_dim), generator=g, device="cuda")
    v = torch.randn((n, kv_dim), generator=g, device="cuda")
    q = torch.randn((case["tokens"], case["heads"] * case["hd"]), generator=g, device="cuda")
    return k, v, q


def _config(case):
    return dataclasses.replace(SHAPES[case["shape"]], layers=case["layers"], ctx=max(256, case["prompt"] + case["gen"]))


def _tokens(case, seed):
    return np.random.default_rng(seed).integers(0, 32000, size=case["prompt"]).astype(np.int32)


class _State:
    pass


def prepare(case, seed):
    s = _State()
    s.case = case
    if case["kind"] in ("prefill", "request"):
        fd, path = tempfile.mkstemp(suffix=".gguf")
        os.close(fd)
        try:
            synth.write_model(_config(case), path, seed=seed, device="cuda", digest=False)
            s.model = capi.Model(path, act_mode=ACT[case["act"]], max_batch=case["batch"], kv_type=KV[case["kv"]])
        finally:
            os.unlink(path)
        s.tokens = _tokens(case, seed)
        torch.cuda.synchronize()
        return s
    s.ctx = capi.Context(0)
    if case["kind"] == "attend":
        kv_dim, n = case["kv_heads"] * case["hd"], case["pos"] + case["tokens"]
        k, v, q = _cache_rows(case, seed)
        s.kv = s.ctx.kv_cache(1, kv_dim, page_tokens=case["page"], max_tokens=n, kv_type=KV[case["kv"]])
        torch.cuda.synchronize()
        if case["pos"]:
            s.kv.write(0, 0, k[: case["pos"]].contiguous(), v[: case["pos"]].contiguous())
        s.k, s.v, s.q = k[case["pos"]:].contiguous(), v[case["pos"]:].contiguous(), q
        s.out = torch.empty_like(q)
        s.ctx.synchronize()
        torch.cuda.synchronize()
        return s
    s.bytes = _weight(case, seed)
    name = "blk.0.ffn_up.weight" if case.get("ffn") else "blk.0.attn_q.weight"
    s.w = s.ctx.wrap(name, TYPES[case["type"]], case["k"], case["n"], s.bytes.data_ptr(), s.bytes.numel())
    m = case.get("m", 1)
    s.x = _activations(m, case["k"], seed, 2)
    s.y = torch.empty((m, case["n"]), device="cuda")
    if case["kind"] == "matvec":
        s.x, s.y = s.x[0], s.y[0]
        if case["host"]:
            s.x, s.y = s.x.cpu().numpy(), np.empty(case["n"], np.float32)
    torch.cuda.synchronize()
    return s


def run(s):
    case = s.case
    kind = case["kind"]
    if kind == "matvec":
        return s.ctx.matvec(s.w, s.x, s.y)
    if kind == "matmul":
        return s.ctx.matmul_batch_v06(s.w, s.x, ACT[case["act"]], s.y)
    if kind == "attend":
        s.kv.write(0, case["pos"], s.k, s.v)
        if case["tokens"] == 1:
            return s.kv.attn_decode(0, s.q, case["pos"], case["heads"], case["kv_heads"], case["hd"], s.out)
        return s.kv.attn_batch(0, s.q, case["pos"], case["tokens"], case["heads"], case["kv_heads"], case["hd"], s.out)
    s.model.reset()
    logits = s.model.prefill(s.tokens, batch=case["batch"])
    if kind == "prefill":
        return {"logits": logits}
    ids, last = s.model.generate_greedy(int(np.argmax(logits)), case["gen"], logits=True)
    return {"prompt_logits": logits, "last_logits": last, "ids": ids}


# ---- what a pass cannot do without ----------------------------------------------------------------------------

def _row_bytes(ty, k):
    e, b = BLOCK[ty]
    return k // e * b


def _attention_work(pos, tokens, heads, kv_heads, hd, kv):
    """K/V rows 0..pos+tokens-1 read once, the new ones written; 4 hd operations per head and causal (token, row)."""
    row = 2 * kv_heads * hd * {"f32": 4, "f16": 2, "q8": 1}[kv] + (8 if kv == "q8" else 0)
    pairs = tokens * pos + tokens * (tokens + 1) // 2
    return (pos + tokens) * row, 4 * hd * heads * pairs


def work(case):
    if case["kind"] in ("matvec", "matmul"):
        m, k, n = case.get("m", 1), case["k"], case["n"]
        return {"bytes": n * _row_bytes(case["type"], k) + 4 * m * (k + n), "flops": 2 * m * k * n}
    if case["kind"] == "attend":
        b, f = _attention_work(case["pos"], case["tokens"], case["heads"], case["kv_heads"], case["hd"], case["kv"])
        kv_dim = case["kv_heads"] * case["hd"]
        return {"bytes": b + 4 * case["tokens"] * 2 * (kv_dim + case["heads"] * case["hd"]), "flops": f}
    c = _config(case)
    name = {v: k for k, v in TYPES.items()}
    kv_dim = c.kv_heads * c.head_dim
    wt, dt = name[c.wtype], name[c.down_type if c.down_type is not None else c.wtype]
    layer_el = c.dim * (2 * c.dim + 2 * kv_dim) + 3 * c.dim * c.ffn
    layer_b = (2 * c.dim + 2 * kv_dim + 2 * c.ffn) * _row_bytes(wt, c.dim) + c.dim * _row_bytes(dt, c.ffn)
    head_b = c.vocab * _row_bytes(name[c.out_type], c.dim)
    a_b, a_f = _attention_work(0, case["prompt"], c.heads, c.kv_heads, c.head_dim, case["kv"])
    out = {"bytes": c.layers * (layer_b + a_b) + head_b,
           "flops": c.layers * (2 * case["prompt"] * layer_el + a_f) + 2 * c.vocab * c.dim}
    for i in range(case["gen"]):  # each decoded token reads every weight again
        a_b, a_f = _attention_work(case["prompt"] + i, 1, c.heads, c.kv_heads, c.head_dim, case["kv"])
        out["bytes"] += c.layers * (layer_b + a_b) + head_b
        out["flops"] += c.layers * (2 * layer_el + a_f) + 2 * c.vocab * c.dim
    return out


# About four times what the path shows against the same arithmetic in 64 bits: 32-bit chains over at most a few
# hundred blocks (Q4_0 / Q8_0 products: 4e-7 seen), a double sum rounded once to 32 bits (Q6_K: 3e-8), 32-bit chains
# over a few thousand positions (attention: 7e-7 at 1500).  Whole models: a 32-bit sum taken in another order moves
# single Q8 activations by a step, layer after layer; 1e-3 of the logits is what this library's own tests allow.
def tolerance(case):
    if case["kind"] in ("matvec", "matmul"):
        return {"rel": 2e-7 if case["type"] == "q6_k" else 2e-6}
    if case["kind"] == "attend":
        return {"rel": 4e-6}
    return {"rel": 1e-3, "differ": 0.02}


# ---- the same results in 64 bits ------------------------------------------------------------------------------

def _half(b):
    return b.contiguous().view(torch.float16)[..., 0].double()


def _dequantized(case, w):
    n, k = case["n"], case["k"]
    if case["type"] == "q4_0":
        b = w.reshape(n, k // 32, 18)
        q = torch.cat([b[..., 2:] & 15, b[..., 2:] >> 4], dim=2).double() - 8.0
        return (q * _half(b[..., :2])[..., None]).reshape(n, k)
    if case["type"] == "q8_0":
        b = w.reshape(n, k // 32, 34)
        return (b[..., 2:].contiguous().view(torch.int8).double() * _half(b[..., :2])[..., None]).reshape(n, k)
    # 6-bit codes: two 128-element halves, each four 32-element rows; scale per 16 elements
    b = w.reshape(n, k // 256, 210)
    rows = []
    for half in range(2):
        ql, qh = b[..., 64 * half:64 * half + 64], b[..., 128 + 32 * half:160 + 32 * half]
        for r in range(4):
            lo = (ql[..., 32 * (r % 2):32 * (r % 2) + 32] >> (4 * (r // 2))) & 15
            rows.append(lo | (((qh >> (2 * r)) & 3) << 4))
    q = torch.cat(rows, dim=2).double() - 32.0
    sc = b[..., 192:208].contiguous().view(torch.int8).double().repeat_interleave(16, dim=2)
    return (q * sc * _half(b[..., 208:])[..., None]).reshape(n, k)


def _q8_activations(x):
    """Q8 blocks of 32: d = max|x| / 127 (1 for a zero block), round(x * (1 / d)) half away from zero, in 32 bits."""
    b = x.reshape(-1, 32)
    top = b.abs().amax(dim=1, keepdim=True)
    one = torch.ones_like(top)
    d = torch.where(top > 0, top / (127.0 * one), one)  # tensor by tensor: a scalar divisor becomes a product
    z = b * (one / d)
    q = torch.clamp(torch.sign(z) * torch.floor(z.abs().double() + 0.5), -127, 127)
    return (q.double() * d.double()).reshape(x.shape)


def _as_stored(x, kv):
    """K/V rows as the cache holds them."""
    if kv == "f32":
        return x.double()
    if kv == "q8":  # one scale per row
        top = x.abs().amax(dim=1, keepdim=True)
        one = torch.ones_like(top)
        s = torch.where(top > 0, top / (127.0 * one), one)
        z = x / s
        return torch.clamp(torch.sign(z) * torch.floor(z.abs().double() + 0.5), -127, 127) * s.double()
    # fp16 bits as the format defines them: ties away from zero, a carry out of the mantissa OR-ed into the exponent
    i = x.contiguous().view(torch.int32)
    sign = torch.where(i < 0, 0x8000, 0)
    e, mant = ((i >> 23) & 255) - 112, i & 0x7FFFFF
    normal = (e.clamp(min=1) << 10) | ((mant + 0x1000) >> 13)
    small = ((((mant | 0x800000) >> (1 - e).clamp(0, 31)) + 0x1000) >> 13)
    bits = torch.where(e <= 0, torch.where(e < -10, torch.zeros_like(small), small), normal) | sign
    return bits.to(torch.int16).view(torch.float16).double()


def exact(case, seed):
    if case["kind"] in ("prefill", "request"):
        return None  # Q8 activations round at every layer: the logits have no 64-bit value of their own
    if case["kind"] == "attend":
        k, v, q = _cache_rows(case, seed)
        kd, vd = (_as_stored(t, case["kv"]).reshape(-1, case["kv_heads"], case["hd"]) for t in (k, v))
        group, t, pos = case["heads"] // case["kv_heads"], case["tokens"], case["pos"]
        qd = q.double().reshape(t, case["heads"], case["hd"])
        out = torch.empty_like(qd)
        late = torch.arange(pos + t, device="cuda")[None, :] > (pos + torch.arange(t, device="cuda"))[:, None]
        for h in range(case["heads"]):
            s = qd[:, h] @ kd[:, h // group].T.contiguous() / math.sqrt(case["hd"])
            out[:, h] = torch.softmax(s.masked_fill(late, -math.inf), dim=1) @ vd[:, h // group].contiguous()
        return out.reshape(t, -1)
    m = case.get("m", 1)
    x = _activations(m, case["k"], seed, 2)
    w = _dequantized(case, _weight(case, seed))
    q8 = case["type"] == "q4_0" and (case["kind"] == "matvec" or (case["act"] == "q8" and m >= 2))
    y = (_q8_activations(x) if q8 else x.double()) @ w.T.contiguous()
    if case["kind"] == "matvec":
        return y[0].cpu().numpy() if case["host"] else y[0]
    return y
