"""The work that TL programs have this backend do, as cases that can be timed and compared.

Each kind of case is one way a program reaches the library:

  linear   one quantized linear layer on device buffers (tl_hip_launch_quant_matvec for up to
           four rows, tl_hip_launch_quant_gemm beyond): decode rows, chat prompts, full prompts,
           the exact f32 path of tl_qtensor_matmul and the f16 matrix path
  decode   attention of one new token per sequence over an f16 KV cache
  prefill  causal attention of a prompt over an f16 KV cache
  sdpa     the scaled-dot-product-attention operator on f32 tensors
  rows     the row operators around the linears: norms, RoPE, SwiGLU, softmax
  layer    one decoder layer as chatbot.tl composes it, operator by operator
  model    a whole TinyLlama-shape decoder: prompt, then greedy decode, with its logits

Sizes are those of the benchmark and the tests (TinyLlama-1.1B, 4096 / 11008-wide Llama
layers) and odd ones between.  Everything is made from the seed on the GPU; quantized weights
are GGUF blocks whose values have the spread of a trained model's (about N(0, 0.02)).
"""
import math

import numpy as np
import torch

from tl_amd import HipDevice, QTensor
from tl_amd.llama import HipLlama, LlamaConfig, linear_type

TYPES = {"Q4_0": 2, "Q8_0": 8, "Q4_K": 12, "Q6_K": 14}
BLOCK_BYTES = {"Q4_0": 18, "Q8_0": 34, "Q4_K": 144, "Q6_K": 210}
BLOCK_ELEMS = {"Q4_0": 32, "Q8_0": 32, "Q4_K": 256, "Q6_K": 256}
STD = 0.02
EPS = 1e-5
LAYER_WEIGHTS = ("attn_q", "attn_k", "attn_v", "attn_output", "ffn_gate", "ffn_up", "ffn_down")

_device = None


def device():
    global _device
    if _device is None:
        _device = HipDevice(0)
    return _device


def listed():
    return [
        # one row through a 4096 x 4096 Q4_0 weight: a decode projection, the smallest call
        {"name": "matvec_q4_0", "kind": "linear", "type": "Q4_0", "m": 1, "n": 4096, "k": 4096, "f16": False},
        # a full prompt through an FFN projection by tl_qtensor_matmul: the exact f32 path
        {"name": "prompt_f32_q4_0", "kind": "linear", "type": "Q4_0", "m": 512, "n": 11008, "k": 4096, "f16": False},
        # a chat turn of 16 tokens through the down projection, exact f32 path, Q8_0
        {"name": "turn_f32_q8_0", "kind": "linear", "type": "Q8_0", "m": 16, "n": 4096, "k": 11008, "f16": False},
        # a ragged prompt through a Q6_K down projection (Q4_K_M files) on the f16 matrix path
        {"name": "prompt_f16_q6_k", "kind": "linear", "type": "Q6_K", "m": 301, "n": 2048, "k": 5632, "f16": True},
        # eight sequences decoding over 2048-token caches
        {"name": "decode_attention", "kind": "decode", "batch": 8, "len": 2048, "hq": 32, "hkv": 8, "d": 128},
        # a prompt that fills TinyLlama's 2048-token context
        {"name": "prefill_attention", "kind": "prefill", "n": 2048, "pos0": 0, "hq": 32, "hkv": 4, "d": 64},
        # the attention operator of a .tl program over a 512-token prompt, causal ones mask
        {"name": "sdpa_512", "kind": "sdpa", "heads": 32, "sq": 512, "sk": 512, "d": 64, "mask": True},
        # the row operators of a 512-token prompt
        {"name": "rows_512", "kind": "rows", "n": 512, "heads": 32, "hd": 128, "ffn": 11008, "vocab": 32000},
        # one TinyLlama layer of a 128-token prompt in the chatbot's operators (Q4_K weights)
        {"name": "layer_ops", "kind": "layer", "type": "Q4_K", "n": 128, "past": 0},
        # a 512-token prompt through the whole decoder with its default settings (exact f32 path)
        {"name": "model_prompt_f32", "kind": "model", "type": "Q4_0", "layers": 22, "n": 512, "steps": 0, "f16": False, "kv16": False},
        # the same prompt on the f16 path with an f16 cache, as the benchmark has it
        {"name": "model_prompt_f16", "kind": "model", "type": "Q4_0", "layers": 22, "n": 512, "steps": 0, "f16": True, "kv16": True},
        # a chat turn over a Q4_K_M file: 24 tokens in, 16 greedy tokens out (graph replay), f16 cache
        {"name": "model_chat", "kind": "model", "type": "Q4_K_M", "layers": 22, "n": 24, "steps": 16, "f16": False, "kv16": True},
    ]


def draw(rng):
    """One more case of the same ranges."""
    def log(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["linear"] * 4 + ["decode", "prefill", "sdpa", "rows", "layer", "model"])
    typ = rng.choice(sorted(TYPES))
    if kind == "linear":
        e = 256 if BLOCK_ELEMS[typ] == 256 else 32
        return {"kind": kind, "type": typ, "m": log(1, 512), "n": log(256, 11008), "k": e * log(256 // e, 11008 // e),
                "f16": rng.random() < 0.4}
    if kind == "decode":
        hkv, d = rng.choice([4, 8]), rng.choice([64, 128])
        return {"kind": kind, "batch": log(1, 8), "len": log(64, 4096), "hq": hkv * rng.choice([4, 8]), "hkv": hkv, "d": d}
    if kind == "prefill":
        n = log(5, 2048)
        hkv, d = rng.choice([4, 8]), rng.choice([64, 128])
        return {"kind": kind, "n": n, "pos0": rng.choice([0, 0, rng.randrange(0, 2049 - n)]), "hq": 32, "hkv": hkv, "d": d}
    if kind == "sdpa":
        sq = log(1, 512)
        return {"kind": kind, "heads": rng.choice([4, 8, 16, 32]), "sq": sq, "sk": sq + rng.choice([0, 0, log(1, 512)]),
                "d": rng.choice([32, 64, 80, 128]), "mask": rng.random() < 0.5}
    if kind == "rows":
        heads, hd = rng.choice([8, 16, 32]), rng.choice([64, 128])
        return {"kind": kind, "n": log(1, 512), "heads": heads, "hd": hd, "ffn": log(1000, 11008), "vocab": log(1000, 32000)}
    if kind == "layer":
        past = rng.choice([0, 0, log(1, 1024)])
        return {"kind": kind, "type": typ, "n": 1 if past else log(5, 512), "past": past}
    # tokens are generated after exact prompts only: on the f16 path two logits that differ by its
    # rounding may change places, and another token is another text
    f16 = rng.random() < 0.5
    return {"kind": kind, "type": rng.choice([typ, "Q4_K_M"]), "layers": rng.randrange(2, 7), "n": log(5, 512),
            "steps": 0 if f16 else rng.randrange(0, 17), "f16": f16, "kv16": f16 or rng.random() < 0.5}


# ------------------------------------------------------------------------- inputs ----
def generator(seed, *key):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 1000003 + sum((i + 1) * 7919 * int(v) for i, v in enumerate(key))) % (1 << 62))
    return g


def normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def whole(g, shape, mean, std, lo, hi):
    """Whole numbers around `mean`, clipped to [lo, hi], as uint8."""
    x = torch.empty(shape, device="cuda", dtype=torch.float16).normal_(mean, std, generator=g)
    return x.round_().clamp_(lo, hi).to(torch.int16).to(torch.uint8)


def half_bytes(x):
    return x.to(torch.float16).view(torch.uint8).view(*x.shape, 2)


def blocks(g, typ, n, k):
    """GGUF blocks of an [n, k] weight, uint8 [n, blocks, bytes] on the GPU."""
    nb = k // BLOCK_ELEMS[typ]
    spread = 0.8 + 0.4 * torch.rand(n, nb, generator=g, device="cuda")
    if typ == "Q4_0":
        q = whole(g, (n, nb, 32), 8, 2.7, 0, 15)
        return torch.cat([half_bytes(spread * (STD / 2.7)), q[..., :16] | (q[..., 16:] << 4)], dim=-1)
    if typ == "Q8_0":
        q = whole(g, (n, nb, 32), 128, 40, 1, 255) ^ 128  # two's complement of q - 128
        return torch.cat([half_bytes(spread * (STD / 40)), q], dim=-1)
    if typ == "Q4_K":
        q = whole(g, (n, nb, 4, 64), 8, 2.7, 0, 15)
        sc, mn = whole(g, (n, nb, 8), 44, 6, 20, 63), whole(g, (n, nb, 8), 44, 6, 20, 63)
        low, high = sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6)
        scales = torch.cat([low, high, (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], dim=-1)
        d = spread * (STD / 2.7 / 44)
        return torch.cat([half_bytes(d), half_bytes(8 * d), scales, (q[..., :32] | (q[..., 32:] << 4)).flatten(2)], dim=-1)
    q = whole(g, (n, nb, 2, 4, 32), 32, 9, 0, 63)  # the 128-weight halves, their four 32-weight rows
    lo, hi = q & 15, q >> 4
    ql = torch.cat([lo[..., 0, :] | (lo[..., 2, :] << 4), lo[..., 1, :] | (lo[..., 3, :] << 4)], dim=-1)
    qh = hi[..., 0, :] | (hi[..., 1, :] << 2) | (hi[..., 2, :] << 4) | (hi[..., 3, :] << 6)
    sc = whole(g, (n, nb, 16), 90, 15, 30, 127)
    return torch.cat([ql.flatten(2), qh.flatten(2), sc, half_bytes(spread * (STD / 9 / 90))], dim=-1)


def values(typ, raw):
    """The f64 values [n, k] of GGUF blocks."""
    def f(b):
        return b.contiguous().view(torch.float16).double()

    n = raw.shape[0]
    if typ == "Q4_0":
        q = raw[..., 2:]
        return (torch.cat([q & 15, q >> 4], dim=-1).double().sub_(8) * f(raw[..., :2])).view(n, -1)
    if typ == "Q8_0":
        return (raw[..., 2:].contiguous().view(torch.int8).double() * f(raw[..., :2])).view(n, -1)
    if typ == "Q4_K":
        s, q = raw[..., 4:16], raw[..., 16:].unflatten(-1, (4, 32))
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], dim=-1).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], dim=-1).double()
        q = torch.stack([q & 15, q >> 4], dim=-2).flatten(-3, -2).double()  # [n, nb, 8, 32]
        return (q * (sc * f(raw[..., :2]))[..., None] - (mn * f(raw[..., 2:4]))[..., None]).reshape(n, -1)
    ql, qh = raw[..., :128].unflatten(-1, (2, 2, 32)), raw[..., 128:192].unflatten(-1, (2, 32))
    lo = torch.cat([ql & 15, ql >> 4], dim=-2)  # [n, nb, 2, 4, 32]
    hi = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], dim=-2)
    q = (lo | (hi << 4)).double().sub_(32).view(*raw.shape[:2], 16, 16)
    sc = raw[..., 192:208].contiguous().view(torch.int8).double()
    return (q * (sc * f(raw[..., 208:210]))[..., None]).reshape(n, -1)


def host(t):
    return t.flatten().cpu().numpy()


def weight(typ, raw, n, k):
    q = QTensor(TYPES[typ], host(raw), (n, k))
    q.upload(device().lib)
    q.data = None  # the program keeps the device residency only
    return q


def tensor(t):
    return device().tensor_new(t.cpu().numpy())


class Shared:
    """A device tensor handle seen by torch without a copy; keeps the handle."""

    def __init__(self, t, shape):
        self.t = t
        self.__cuda_array_interface__ = {"shape": shape, "typestr": "<f4", "data": (t.data_ptr, False), "version": 2}


def seen(t, *shape):
    return torch.as_tensor(Shared(t, shape), device="cuda")


def linear_inputs(case, seed):
    g = generator(seed, 1)
    return normal(g, case["m"], case["k"]), blocks(g, case["type"], case["n"], case["k"])


def decode_inputs(case, seed):
    g = generator(seed, 2)
    shape = (case["batch"], case["hkv"], case["len"], case["d"])
    return normal(g, case["batch"], case["hq"], case["d"]), normal(g, *shape).half(), normal(g, *shape).half()


def prefill_inputs(case, seed):
    g = generator(seed, 3)
    shape = (case["hkv"], case["pos0"] + case["n"], case["d"])
    return normal(g, case["n"], case["hq"], case["d"]), normal(g, *shape).half(), normal(g, *shape).half()


def sdpa_inputs(case, seed):
    g = generator(seed, 4)
    h, sq, sk, d = case["heads"], case["sq"], case["sk"], case["d"]
    mask = torch.ones(sq, sk, device="cuda").tril(sk - sq) if case["mask"] else None
    return normal(g, 1, h, sq, d), normal(g, 1, h, sk, d), normal(g, 1, h, sk, d), mask


def rows_inputs(case, seed):
    g = generator(seed, 5)
    n, dim = case["n"], case["heads"] * case["hd"]
    return {"x": normal(g, n, dim), "r": normal(g, n, dim), "w": 0.5 + torch.rand(dim, generator=g, device="cuda"),
            "gate": normal(g, n, case["ffn"]), "up": normal(g, n, case["ffn"]), "logits": 3 * normal(g, n, case["vocab"])}


def shape_of(name):
    return LlamaConfig.tinyllama().linear_shape(name)


def layer_inputs(case, seed):
    g = generator(seed, 6)
    cfg = LlamaConfig.tinyllama()
    past = (1, cfg.n_kv_heads, case["past"], cfg.head_dim)
    s = {"x": normal(g, case["n"], cfg.d_model)}
    for i in ("w1", "w2"):
        s[i] = 0.5 + torch.rand(cfg.d_model, generator=g, device="cuda")
    s["k"], s["v"] = normal(g, *past), normal(g, *past)
    for name in LAYER_WEIGHTS:
        s[name] = blocks(g, case["type"], *shape_of(name))
    return s


def config(case):
    c = LlamaConfig.tinyllama()
    c.n_layers = case["layers"]
    return c


def model_type(case, layer, name):
    t = linear_type(TYPES.get(case["type"], case["type"]), config(case), layer, name)
    return next(i for i, v in TYPES.items() if v == t)


def model_linear(case, seed, layer, name):
    n, k = shape_of(name if layer >= 0 else "output")
    return blocks(generator(seed, 7, layer + 1, LAYER_WEIGHTS.index(name) if layer >= 0 else 7), model_type(case, layer, name), n, k)


def model_norm(case, seed, layer, which):
    return 0.5 + torch.rand(2048, generator=generator(seed, 8, layer + 1, which), device="cuda")


def model_embedding(case, seed):
    return normal(generator(seed, 9), 32000, 2048)


def model_prompt(case, seed):
    return torch.randint(0, 32000, (case["n"],), generator=generator(seed, 10), device="cuda").cpu().numpy().astype(np.int32)


def prepare(case, seed):
    dev, kind, s = device(), case["kind"], {"case": case}
    if kind == "linear":
        x, raw = linear_inputs(case, seed)
        s.update(x=x, w=weight(case["type"], raw, case["n"], case["k"]), y=torch.empty(case["m"], case["n"], device="cuda"))
    elif kind in ("decode", "prefill"):
        q, k, v = (decode_inputs if kind == "decode" else prefill_inputs)(case, seed)
        s.update(q=tensor(q), k=dev.tensor_new_f16(k.cpu().numpy()), v=dev.tensor_new_f16(v.cpu().numpy()))
    elif kind == "sdpa":
        q, k, v, mask = sdpa_inputs(case, seed)
        s.update(q=tensor(q), k=tensor(k), v=tensor(v), mask=tensor(mask) if mask is not None else None)
    elif kind == "rows":
        s.update({i: tensor(t) for i, t in rows_inputs(case, seed).items()})
        s["x3"] = dev.tensor_reshape(s["x"], (case["n"], case["heads"], case["hd"]))
        s["cos"], s["sin"] = (f(case["hd"], 2048, 10000.0) for f in (dev.tensor_rope_new_cos, dev.tensor_rope_new_sin))
    elif kind == "layer":
        for i, t in layer_inputs(case, seed).items():
            if i in LAYER_WEIGHTS:
                s[i] = weight(case["type"], t, *shape_of(i))
            elif t.numel():
                s[i] = tensor(t)
        s["cos"], s["sin"] = (f(64, 2048, 10000.0) for f in (dev.tensor_rope_new_cos, dev.tensor_rope_new_sin))
    else:
        m = HipLlama(config(case), kv_f16=case["kv16"])
        items = [("embedding", -1, 0, lambda: model_embedding(case, seed))]
        for l in range(case["layers"]):
            items += [("linear", l, i, lambda l=l, w=w: model_linear(case, seed, l, w)) for i, w in enumerate(LAYER_WEIGHTS)]
            items += [("norm", l, i, lambda l=l, i=i: model_norm(case, seed, l, i)) for i in (0, 1)]
        items += [("norm", -1, 0, lambda: model_norm(case, seed, -1, 0)), ("linear", -1, 0, lambda: model_linear(case, seed, -1, "output"))]
        m.load(((a, b, c, host(make())) for a, b, c, make in items), ggml_type=TYPES.get(case["type"], case["type"]))
        s.update(model=m, prompt=model_prompt(case, seed))
    return s


# --------------------------------------------------------------------------- runs ----
def run_linear(s):
    c, x, y = s["case"], s["x"], s["y"]
    lib, w = device().lib, s["w"].upload(device().lib)
    if c["m"] <= 4:
        rc = lib.tl_hip_launch_quant_matvec(w, x.data_ptr(), y.data_ptr(), c["m"], None)
    else:
        rc = lib.tl_hip_launch_quant_gemm(w, x.data_ptr(), y.data_ptr(), c["m"], int(c["f16"]), None)
    if rc:
        raise RuntimeError(lib.tl_hip_last_error().decode())
    return y


def run_decode(s):
    c = s["case"]
    o = device().attention_decode(s["q"], s["k"], s["v"], c["len"], 1 / math.sqrt(c["d"]))
    return seen(o, c["batch"], c["hq"], c["d"])


def run_prefill(s):
    c = s["case"]
    o = device().attention_prefill(s["q"], s["k"], s["v"], c["pos0"], 1 / math.sqrt(c["d"]))
    return seen(o, c["n"], c["hq"], c["d"])


def run_sdpa(s):
    c = s["case"]
    return seen(device().tensor_scaled_dot_product_attention(s["q"], s["k"], s["v"], s["mask"]), c["heads"], c["sq"], c["d"])


def run_rows(s):
    dev, c = device(), s["case"]
    n, dim = c["n"], c["heads"] * c["hd"]
    return {
        "norm": seen(dev.tensor_rms_norm(s["x"], s["w"], EPS), n, dim),
        "add_norm": seen(dev.fused_add_rms_norm(s["x"], s["r"], s["w"], EPS), n, dim),
        "rope": seen(dev.tensor_apply_rope_pos(s["x3"], s["cos"], s["sin"], 0, c["heads"]), n, c["heads"], c["hd"]),
        "swiglu": seen(dev.fused_silu_mul(s["gate"], s["up"]), n, c["ffn"]),
        "softmax": seen(dev.tensor_softmax(s["logits"], -1), n, c["vocab"]),
    }


def run_layer(s):
    """Block::forward of chatbot.tl in its own operators."""
    dev, c = device(), s["case"]
    n, past, heads, kv, hd = c["n"], c["past"], 32, 4, 64
    x = s["x"]
    h = dev.tensor_rms_norm(x, s["w1"], EPS)
    q = dev.tensor_reshape(dev.tl_qtensor_matmul(h, s["attn_q"]), (1, n, heads, hd))
    k = dev.tensor_reshape(dev.tl_qtensor_matmul(h, s["attn_k"]), (1, n, kv, hd))
    v = dev.tensor_reshape(dev.tl_qtensor_matmul(h, s["attn_v"]), (1, n, kv, hd))
    cos, sin = dev.tensor_narrow(s["cos"], 0, past, n), dev.tensor_narrow(s["sin"], 0, past, n)
    k = dev.tensor_transpose(dev.tensor_apply_rope(k, cos, sin), 1, 2)
    v = dev.tensor_transpose(v, 1, 2)
    if past:
        k, v = dev.tensor_cat(s["k"], k, 2), dev.tensor_cat(s["v"], v, 2)
    q = dev.tensor_transpose(dev.tensor_apply_rope(q, cos, sin), 1, 2)
    kw, vw = dev.tensor_repeat_interleave(k, heads // kv, 1), dev.tensor_repeat_interleave(v, heads // kv, 1)
    a = dev.tensor_scale(dev.tensor_matmul(q, dev.tensor_transpose(kw, 2, 3)), 0.125)
    if n > 1:
        a = dev.tensor_add(a, dev.tensor_reshape(dev.tensor_new_causal_mask(n), (1, 1, n, n)))
    o = dev.tensor_transpose(dev.tensor_matmul(dev.tensor_softmax(a, 3), vw), 1, 2)
    x = dev.tensor_add(x, dev.tl_qtensor_matmul(dev.tensor_reshape(o, (n, heads * hd)), s["attn_output"]))
    h = dev.tensor_rms_norm(x, s["w2"], EPS)
    u = dev.tensor_mul(dev.tensor_silu(dev.tl_qtensor_matmul(h, s["ffn_gate"])), dev.tl_qtensor_matmul(h, s["ffn_up"]))
    x = dev.tensor_add(x, dev.tl_qtensor_matmul(u, s["ffn_down"]))
    return {"x": seen(x, n, heads * hd), "k": seen(k, kv, past + n, hd), "v": seen(v, kv, past + n, hd)}


def run_model(s):
    m, c = s["model"], s["case"]
    m.reset()
    out = {"prompt": m.forward(s["prompt"], prefill_f16=c["f16"])}
    if c["steps"]:
        first = m.sample_greedy(1.1, s["prompt"])
        rest = m.generate(first, c["steps"], 1.1, history=s["prompt"])
        out["tokens"] = np.concatenate([[first], rest]).astype(np.int32)
        out["last"] = m.forward(rest[-1:])
    return out


RUN = {"linear": run_linear, "decode": run_decode, "prefill": run_prefill, "sdpa": run_sdpa, "rows": run_rows,
       "layer": run_layer, "model": run_model}


def run(s):
    return RUN[s["case"]["kind"]](s)


# -------------------------------------------------------------------- work, bounds ----
def linear_work(typ, m, n, k):
    return {"bytes": n * (k // BLOCK_ELEMS[typ]) * BLOCK_BYTES[typ] + 4 * m * (n + k), "flops": 2 * m * n * k}


def total(*parts):
    return {i: sum(p[i] for p in parts) for i in ("bytes", "flops")}


def work(case):
    kind = case["kind"]
    if kind == "linear":
        return linear_work(case["type"], case["m"], case["n"], case["k"])
    if kind == "decode":
        b, d = case["batch"], case["d"]
        return {"bytes": b * (4 * case["hkv"] * case["len"] * d + 8 * case["hq"] * d), "flops": 4 * b * case["hq"] * case["len"] * d}
    if kind == "prefill":
        n, d, keys = case["n"], case["d"], case["pos0"] + case["n"]
        pairs = n * case["pos0"] + n * (n + 1) // 2
        return {"bytes": 4 * case["hkv"] * keys * d + 8 * n * case["hq"] * d, "flops": 4 * case["hq"] * pairs * d}
    if kind == "sdpa":
        h, sq, sk, d = case["heads"], case["sq"], case["sk"], case["d"]
        return {"bytes": 4 * h * d * (2 * sq + 2 * sk) + (4 * sq * sk if case["mask"] else 0), "flops": 4 * h * sq * sk * d}
    if kind == "rows":
        n, dim = case["n"], case["heads"] * case["hd"]
        table = 8 * n * case["hd"]
        return {"bytes": 4 * n * (7 * dim + 3 * case["ffn"] + 2 * case["vocab"]) + 8 * dim + table, "flops": 20 * n * (dim + case["ffn"] + case["vocab"])}
    if kind == "layer":
        n, t = case["n"], case["past"] + case["n"]
        attn = {"bytes": 4 * (2 * 256 * (2 * t) + 2 * n * 2048), "flops": 4 * 2048 * n * t}
        return total(attn, *(linear_work(case["type"], n, *shape_of(w)) for w in LAYER_WEIGHTS))
    n, steps = case["n"], case["steps"]
    rounds = [n] + [1] * (steps + 1 if steps else 0)
    parts = []
    for m in rounds:
        parts += [linear_work(model_type(case, l, w), m, *shape_of(w)) for l in range(case["layers"]) for w in LAYER_WEIGHTS]
        parts.append(linear_work(model_type(case, -1, "output"), 1, *shape_of("output")))
        parts.append({"bytes": 4 * m * 2048, "flops": 2 * 2048 * m * n * case["layers"]})
    return total(*parts)


def tolerance(case):
    """About four times the distance from exact() that the paths were measured to have: f32 sums
    of up to 11008 products 1.9e-6, f16 operands 2.9e-4 (one linear or attention) and 1.4e-3 (22
    layers), f32 through 22 layers 5.1e-6, 6.2e-4 with the cache in f16."""
    kind = case["kind"]
    if kind == "linear":
        return {"rel": 1.2e-3} if case["f16"] and case["m"] > 4 else {"rel": 8e-6}
    if kind == "model":
        return {"rel": 6e-3} if case["f16"] else {"rel": 2.5e-3} if case["kv16"] else {"rel": 2.5e-5}
    return {"rel": {"decode": 2e-6, "prefill": 1e-3, "sdpa": 2e-6, "rows": 2e-6, "layer": 8e-6}[kind]}


# ------------------------------------------------------------- the same in 64 bits ----
def norm64(x, w):
    return x / (x.square().mean(-1, keepdim=True) + EPS).sqrt() * w.double()


def rotate64(x, row):
    """Interleaved pairs turned by the angles of position(s) `row` ([..., tokens, heads, hd])."""
    hd = x.shape[-1]
    inv = 10000.0 ** (-torch.arange(0, hd, 2, device="cuda", dtype=torch.float64) / hd)
    ang = row.double()[:, None, None] * inv
    a, b = x[..., 0::2], x[..., 1::2]
    return torch.stack([a * ang.cos() - b * ang.sin(), a * ang.sin() + b * ang.cos()], dim=-1).flatten(-2)


def attend64(q, k, v, scale, mask=None):
    """q [.., sq, d] over k, v [.., sk, d]; mask true where a key is seen."""
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * scale
    if mask is not None:
        s = s.masked_fill(~mask, -math.inf)
    return torch.matmul(s.softmax(-1), v.double())


def layer64(x, w, norms, past_k, past_v, past):
    n = x.shape[0]
    h = norm64(x, norms[0])
    q, k, v = (h @ w(i).T for i in ("attn_q", "attn_k", "attn_v"))
    row = torch.full((n,), past, device="cuda")  # every token by the call's first position, as chatbot.tl has it
    q = rotate64(q.view(n, 32, 64), row).transpose(0, 1)
    k = rotate64(k.view(n, 4, 64), row).transpose(0, 1)
    v = v.view(n, 4, 64).transpose(0, 1)
    if past:
        k, v = torch.cat([past_k[0].double(), k], 1), torch.cat([past_v[0].double(), v], 1)
    mask = torch.ones(n, past + n, device="cuda", dtype=torch.bool).tril(past)
    o = attend64(q, k.repeat_interleave(8, 0), v.repeat_interleave(8, 0), 0.125, mask)
    x = x + o.transpose(0, 1).reshape(n, 2048) @ w("attn_output").T
    h = norm64(x, norms[1])
    g = h @ w("ffn_gate").T
    x = x + (g * torch.sigmoid(g) * (h @ w("ffn_up").T)) @ w("ffn_down").T
    return x, k, v


def exact(case, seed):
    kind = case["kind"]
    if kind == "linear":
        x, raw = linear_inputs(case, seed)
        return x.double() @ values(case["type"], raw).T
    if kind == "decode":
        q, k, v = decode_inputs(case, seed)
        g = case["hq"] // case["hkv"]
        return torch.cat([attend64(q[b][:, None], k[b].repeat_interleave(g, 0), v[b].repeat_interleave(g, 0),
                                   1 / math.sqrt(case["d"])).transpose(0, 1) for b in range(case["batch"])])
    if kind == "prefill":
        q, k, v = prefill_inputs(case, seed)
        g = case["hq"] // case["hkv"]
        mask = torch.ones(case["n"], k.shape[1], device="cuda", dtype=torch.bool).tril(case["pos0"])
        return torch.stack([attend64(q[:, h], k[h // g], v[h // g], 1 / math.sqrt(case["d"]), mask)
                            for h in range(case["hq"])], dim=1)
    if kind == "sdpa":
        q, k, v, mask = sdpa_inputs(case, seed)
        return attend64(q[0], k[0], v[0], 1 / math.sqrt(case["d"]), mask.bool() if mask is not None else None)
    if kind == "rows":
        t = {i: v.double() for i, v in rows_inputs(case, seed).items()}
        x3 = t["x"].view(case["n"], case["heads"], case["hd"])
        return {"norm": norm64(t["x"], t["w"]), "add_norm": norm64(t["x"] + t["r"], t["w"]),
                "rope": rotate64(x3, torch.arange(case["n"], device="cuda")),
                "swiglu": t["gate"] * torch.sigmoid(t["gate"]) * t["up"], "softmax": t["logits"].softmax(-1)}
    if kind == "layer":
        s = layer_inputs(case, seed)
        x, k, v = layer64(s["x"].double(), lambda i: values(case["type"], s[i]), (s["w1"], s["w2"]), s["k"], s["v"], case["past"])
        return {"x": x, "k": k, "v": v}
    ids = torch.from_numpy(model_prompt(case, seed)).long().cuda()
    x = model_embedding(case, seed)[ids].double()
    for l in range(case["layers"]):
        norms = [model_norm(case, seed, l, i) for i in (0, 1)]
        x, _, _ = layer64(x, lambda i, l=l: values(model_type(case, l, i), model_linear(case, seed, l, i)), norms, None, None, 0)
    head = values(model_type(case, -1, "output"), model_linear(case, seed, -1, "output"))
    out = {"prompt": (norm64(x[-1:], model_norm(case, seed, -1, 0)) @ head.T)[0]}
    if case["steps"]:  # what follows a choice of tokens has no value of its own
        out.update(tokens=None, last=None)
    return out
