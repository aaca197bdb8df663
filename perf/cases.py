"""What this library's users have it do, as measurable cases.

speech.cpp's decoders call the device in two ways: prompts in blocks of up to 512 rows (MUL_MAT over many columns,
attention of a block over the cache, the layer's row-wise ops, routed experts), and one token, or a draft of up to
five, at a time (mat-vecs, one-row attention, the whole step replayed from a recording). Kinds of a case:

  product  one to three weights sharing their input (a single weight; gate + up; q + k + v), M columns; with M <= 8
           optionally behind the fused RMS norm of the decode step
  attend   a block's q / k norms, RoPE and KV stores, then attention over the cache (one row: the fused call)
  moe      a MoE FFN: the F32 router over all rows, gate and up experts, SwiGLU, down experts (the top-k pick itself is
           the host program's, as in speech.cpp: the ids are in hand)
  layer    one decoder layer over a prompt block, op after op as a new graph for each block runs it
  decode   a whole decode step, replayed from the recording that a program keeps: embedding row, layers, head, argmax

Weights are N(0, 0.02) quantized to ggml blocks, activations N(0, 1), norm weights N(1, 0.1), cache values N(0, 1) in
f16, masks causal with the cache read to a multiple of 64 positions. The decode step's embedding is N(0, 1): the stream
that the layers add to is then large beside what each adds, as it is in a trained model (with a small one, a last bit
that moves one int8 code of an activation is magnified from layer to layer).

exact() restates each op in 64 bits as ggml defines it: activations are first rounded as the op rounds them (Q8_0
blocks for Q8_0 weights, Q8_K for the K-quants, fp16 for F16 weights, nothing for F32), then everything is summed in
double precision. A chain of such roundings has no one value that all correct orders of summing come near: a last bit
that moves an activation's code by one stands for a difference some 1e5 times as large, so that with few values it is
chance whether a result is 1e-7 or 1e-3 from the chain in 64 bits. exact() gives None there (the decode step's logits;
a layer's output and the down experts' for few rows), and the same ops over many rows, or one by one, in other cases.
"""
import importlib.util
import math
import pathlib
import sys

import numpy as np
import torch

ROOT = pathlib.Path(__file__).resolve().parent.parent
EPS, ROPE_BASE = 1e-6, 1e6
TYPES = {"f32": 0, "f16": 1, "q8_0": 8, "q4_k": 12, "q5_k": 13, "q6_k": 14}
BITS = {"f32": 32.0, "f16": 16.0, "q8_0": 8.5, "q4_k": 4.5, "q5_k": 5.5, "q6_k": 6.5625}
DEV = "cuda"


# ------------------------------------------------------------------------------------------------------------- cases
def listed():
    return [
        # q/k/v of one decode token, norm fused, 0.6B shape: the smallest call, where the launch counts
        {"name": "token_qkv_q8_0", "kind": "product", "type": "q8_0", "k": 1024, "n": 2048, "group": 3, "m": 1,
         "norm": True},
        # q/k/v of a drafted token run (one token and four drafted), norm fused, 1.7B shape
        {"name": "verify_qkv_q8_0", "kind": "product", "type": "q8_0", "k": 2048, "n": 2048, "group": 3, "m": 5,
         "norm": True},
        # a prompt block's gate and up, 1.7B shape
        {"name": "block_gate_up_q8_0", "kind": "product", "type": "q8_0", "k": 2048, "n": 6144, "group": 2, "m": 512,
         "norm": False},
        # a prompt block's q/k/v in a Q4_K file
        {"name": "block_qkv_q4_k", "kind": "product", "type": "q4_k", "k": 2048, "n": 2048, "group": 3, "m": 512,
         "norm": False},
        # the ragged last block of a prompt, the down projection of a Q4_K file (Q6_K there)
        {"name": "tail_down_q6_k", "kind": "product", "type": "q6_k", "k": 6144, "n": 2048, "group": 1, "m": 133,
         "norm": False},
        # a prompt block's gate and up in a file that was not quantized
        {"name": "block_gate_up_f16", "kind": "product", "type": "f16", "k": 2048, "n": 6144, "group": 2, "m": 512,
         "norm": False},
        # a prompt block's attention with two blocks before it
        {"name": "attend_block", "kind": "attend", "rows": 512, "past": 1024, "heads": 16, "kv_heads": 8,
         "head_dim": 128},
        # attention of a drafted run far into a long transcript
        {"name": "attend_verify", "kind": "attend", "rows": 5, "past": 3001, "heads": 16, "kv_heads": 8,
         "head_dim": 128},
        # a MoE FFN for a few sequences' tokens, and for a prompt
        {"name": "moe_16_q4_k", "kind": "moe", "type": "q4_k", "hidden": 2048, "ffn": 1536, "experts": 64, "top": 4,
         "tokens": 16},
        {"name": "moe_256_q4_k", "kind": "moe", "type": "q4_k", "hidden": 2048, "ffn": 1536, "experts": 64, "top": 4,
         "tokens": 256},
        # one layer of the 1.7B shape over the second block of a prompt
        {"name": "layer_block_q8_0", "kind": "layer", "type": "q8_0", "hidden": 2048, "ffn": 6144, "heads": 16,
         "kv_heads": 8, "rows": 512, "past": 512},
        # the whole decode step of the 0.6B shape at 1024 positions
        {"name": "decode_q8_0", "kind": "decode", "type": "q8_0", "hidden": 1024, "ffn": 3072, "heads": 16,
         "kv_heads": 8, "layers": 28, "vocab": 151936, "past": 1024},
    ]


MAX_MACS = 512 * 12288 * 2048  # of a product: the largest listed


def draw(rng):
    def logint(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["product"] * 5 + ["attend"] * 3 + ["moe"] * 2 + ["layer"] * 2 + ["decode"])
    if kind == "product":
        t = rng.choice(["q8_0", "q8_0", "q8_0", "q4_k", "q4_k", "q6_k", "q6_k", "q5_k", "f16", "f16", "f32"])
        step = 256 if t.endswith("_k") else rng.choice([128, 128, 64, 32])
        k = max(2, round(logint(512, 6144) / step)) * step
        group = rng.choice([1, 1, 2, 3])
        n = logint(64, 1024) if t == "f32" else logint(256, 6144)
        if rng.random() < 0.5:
            n = max(2, n // 128 * 2) * 64  # model widths; the others are ragged
        else:
            n += n % 2  # k and v are half of q
        top = MAX_MACS // (k * n * (2 if group > 1 else 1))
        m = min(logint(1, 1564), max(1, top))
        if m <= 8 and not t.startswith("f"):
            group = max(2, group)  # a decode step's q/k/v, gate/up
        return {"kind": "product", "type": t, "k": k, "n": n, "group": group, "m": m,
                "norm": m <= 8 and not t.startswith("f") and rng.random() < 0.5}
    if kind == "attend":
        d = rng.choice([128, 128, 128, 64])
        heads, kv = rng.choice([(16, 8), (16, 8), (16, 16), (32, 8), (8, 1)])
        rows = logint(1, 512)
        past = logint(1, 4096) if rng.random() < 0.8 else 0
        while rows * (past + rows) * heads * d > 512 * 1536 * 16 * 128:
            past //= 2
            rows = rows if past else rows // 2
        return {"kind": "attend", "rows": rows, "past": past, "heads": heads, "kv_heads": kv, "head_dim": d}
    if kind == "moe":
        t = rng.choice(["q4_k", "q4_k", "q8_0", "q6_k", "q5_k"])
        hidden, ffn = 256 * rng.randint(3, 8), 256 * rng.randint(2, 6)
        top = rng.choice([2, 4, 8])
        experts = min(rng.choice([16, 32, 64, 128]), 64 * 2048 * 1536 // (hidden * ffn))
        tokens = min(logint(1, 512), 256 * 4 * 2048 * 1536 // (top * hidden * ffn))
        return {"kind": "moe", "type": t, "hidden": hidden, "ffn": ffn, "experts": experts, "top": top,
                "tokens": tokens}
    t = rng.choice(["q8_0", "q8_0", "q4_k", "q6_k", "q5_k", "f16"])
    if kind == "layer":
        hidden = rng.choice([1024, 2048])
        return {"kind": "layer", "type": t, "hidden": hidden, "ffn": 3 * hidden, "heads": 16, "kv_heads": 8,
                "rows": logint(9, 512), "past": rng.choice([0, logint(1, 512)])}
    t = rng.choice(["q8_0", "q4_k", "q6_k"])
    return {"kind": "decode", "type": t, "hidden": 1024, "ffn": 3072, "heads": 16, "kv_heads": 8,
            "layers": rng.randint(2, 28 if t == "q8_0" else 10), "vocab": logint(512, 37984) * 4, "past": logint(1, 1024)}


# ----------------------------------------------------------------------------------------------------- work, tolerance
def _sizes(c):
    """Output widths of a product's weights."""
    return {1: [c["n"]], 2: [c["n"], c["n"]], 3: [c["n"], c["n"] // 2, c["n"] // 2]}[c["group"]]


def _product(t, k, ns, m):
    n = sum(ns)
    return {"bytes": n * k * BITS[t] / 8 + 4 * m * (k + n), "flops": 2 * m * n * k}


def _attend_work(rows, past, heads, kv, d):
    seen = rows * past + rows * (rows + 1) // 2  # (row, position) pairs a causal mask leaves
    # cache read once, q / k / v read, new keys and values stored, the result written
    return {"bytes": 4 * (past + rows) * kv * d + rows * (8 * heads + 12 * kv) * d, "flops": 4 * seen * heads * d}


def _layer_work(c, rows, past):
    d, t = 128, c["type"]
    h, f, q, kv = c["hidden"], c["ffn"], c["heads"] * d, c["kv_heads"] * d
    parts = [_product(t, h, [q, kv, kv], rows), _product(t, q, [h], rows), _product(t, h, [f, f], rows),
             _product(t, f, [h], rows), _attend_work(rows, past, c["heads"], c["kv_heads"], d)]
    weights = (h * (q + 2 * kv) + q * h + 3 * h * f) * BITS[t] / 8
    # a layer reads its input and writes its output once; the caches as above
    return {"bytes": weights + 8 * rows * h + 4 * (past + rows) * kv, "flops": sum(p["flops"] for p in parts)}


def work(c):
    if c["kind"] == "product":
        return _product(c["type"], c["k"], _sizes(c), c["m"])
    if c["kind"] == "attend":
        return _attend_work(c["rows"], c["past"], c["heads"], c["kv_heads"], c["head_dim"])
    if c["kind"] == "moe":
        pairs, h, f, e = c["tokens"] * c["top"], c["hidden"], c["ffn"], c["experts"]
        hit = e * (1 - (1 - c["top"] / e) ** c["tokens"])  # experts that any token picks, on average
        return {"bytes": hit * 3 * h * f * BITS[c["type"]] / 8 + 4 * (h * e + c["tokens"] * (h + e) + pairs * (h + 1)),
                "flops": 2 * pairs * 3 * h * f + 2 * c["tokens"] * h * e}
    if c["kind"] == "layer":
        return _layer_work(c, c["rows"], c["past"])
    one = _layer_work(c, 1, c["past"])
    head = _product(c["type"], c["hidden"], [c["vocab"]], 1)
    return {k: c["layers"] * one[k] + head[k] for k in ("bytes", "flops")}


def tolerance(c):
    """About four times what forcing other kernels and sum orders through the library's options changed."""
    if c["kind"] == "product":
        # Q8_0 / Q4_K sum exact integers, F16 / F32 exact products, all in fp32 (1.6e-7); Q5_K / Q6_K (and Q8_0 rows
        # that are no multiple of 128) round each operand to fp16 first over many columns (2.9e-4)
        if c["type"] in ("q5_k", "q6_k") or c["type"] == "q8_0" and c["k"] % 128:
            return {"rel": 1.2e-3}
        return {"rel": 2e-6}
    if c["kind"] == "attend":
        # fp32 sums, but the turned q and k are stored in fp16: a last bit before that moves some of them (6.5e-6)
        return {"rel": 3e-5, "max": 4e-3}
    # Products round their activations to int8 codes: a last bit upstream moves some codes by one.
    if c["kind"] == "moe":  # 8.2e-5; 2.8e-3 where the gate and up products round to fp16
        return {"rel": 4e-4, "max": 2e-2} if c["type"] == "q4_k" else {"rel": 1e-2, "max": 8e-2}
    if c["kind"] == "layer":  # 1.4e-3, 5.7e-3
        return {"rel": 6e-3 if c["type"] in ("q8_0", "q4_k", "f16") else 2e-2, "max": 0.1}
    # Over 28 layers those moves grow to the activations' own rounding noise: 1.1e-2 .. 1.8e-2 of the logits, whatever
    # small thing set them off (2.7e-2 for the K-quants, which are therefore drawn with fewer layers)
    return {"rel": 3e-2, "max": 0.3}


# ------------------------------------------------------------------------------------------------------- the library
_mx = _be = None


def mx():
    global _mx
    if _mx is None:
        _mx = sys.modules.get("speech_cpp_amd")
    if _mx is None:
        pkg = ROOT / "speech.cpp_amd"
        spec = importlib.util.spec_from_file_location("speech_cpp_amd", pkg / "__init__.py",
                                                      submodule_search_locations=[str(pkg)])
        _mx = importlib.util.module_from_spec(spec)
        sys.modules["speech_cpp_amd"] = _mx
        spec.loader.exec_module(_mx)
    return _mx


def backend():
    """The one backend that a program keeps."""
    global _be
    if _be is None:
        _be = mx().Backend(0)
    return _be


class On:
    """A ggml descriptor over a torch tensor's memory; ne / nb may be those of a view of it."""

    def __init__(self, t, ne=None, nb=None, kind=None):
        self.t = t
        self.desc = mx().MxTensor()
        self.desc.type = {torch.float32: 0, torch.float16: 1, torch.int32: 26}[t.dtype] if kind is None else kind
        ne = list(t.shape[::-1]) if ne is None else list(ne)
        size = t.element_size()
        if nb is None:
            nb = [size]
            for v in ne[:-1]:
                nb.append(nb[-1] * v)
        nb = list(nb)
        while len(ne) < 4:
            nb.append(nb[-1] * ne[-1])
            ne.append(1)
        for i in range(4):
            self.desc.ne[i], self.desc.nb[i] = ne[i], nb[i]
        self.desc.data = t.data_ptr()

    def ref(self):
        return mx().ctypes.byref(self.desc)


class State:
    """What a program keeps between calls; frees its recording with itself."""

    def __init__(self):
        self.graph = None

    def __del__(self):
        if self.graph:
            backend().graph_free(self.graph)


# ------------------------------------------------------------------------------------------------------------ weights
def _half(x):
    return x.half().float()


def _bytes16(x):
    return x.half().view(torch.uint8).reshape(x.shape + (2,))


def _k4(sub, top):
    """Scales and mins of 32-element sub-blocks [..., 8, 32] with codes 0..top, each 6 bits of the block's d / dmin."""
    lo = sub.amin(-1).clamp(max=0)
    scale = (sub.amax(-1) - lo) / top
    d, dmin = _half(scale.amax(-1, keepdim=True) / 63), _half((-lo).amax(-1, keepdim=True) / 63)
    sc = torch.round(scale / d.clamp(min=1e-12)).clamp(0, 63)
    m = torch.round(-lo / dmin.clamp(min=1e-12)).clamp(0, 63)
    q = torch.round((sub + (dmin * m)[..., None]) / (d * sc).clamp(min=1e-12)[..., None]).clamp(0, top)
    return d, dmin, sc, m, q


def weight(t, rows, k, g, std=0.02):
    """`rows` x `k` weights N(0, std) of a type: ggml's bytes [rows, row bytes] and the values that they stand for."""
    x = torch.randn(rows, k, generator=g, device=DEV) * std
    if t == "f32":
        return x, x
    if t == "f16":
        return x.half(), x.half()
    if t == "q8_0":
        b = x.view(rows, k // 32, 32)
        d = b.abs().amax(-1, keepdim=True) / 127
        q = torch.round(b / d.clamp(min=1e-12)).clamp(-127, 127)
        raw = torch.cat([_bytes16(d[..., 0]), q.to(torch.int8).view(torch.uint8)], -1)
        return raw.reshape(rows, -1), (q * _half(d)).reshape(rows, k)
    if t in ("q4_k", "q5_k"):
        d, dmin, sc, m, q = _k4(x.view(rows, k // 256, 8, 32), 15 if t == "q4_k" else 31)
        val = q * (d * sc)[..., None] - (dmin * m)[..., None]
        s, mi, qi = sc.to(torch.uint8), m.to(torch.uint8), q.to(torch.uint8)
        packed = torch.cat([s[..., :4] | (s[..., 4:] >> 4 << 6), mi[..., :4] | (mi[..., 4:] >> 4 << 6),
                            (s[..., 4:] & 15) | ((mi[..., 4:] & 15) << 4)], -1)
        low = qi & 15
        qs = (low[..., 0::2, :] | (low[..., 1::2, :] << 4)).reshape(rows, k // 256, 128)
        parts = [_bytes16(d[..., 0]), _bytes16(dmin[..., 0]), packed]
        if t == "q5_k":
            parts.append(sum((qi[..., j, :] >> 4) << j for j in range(8)))
        return torch.cat(parts + [qs], -1).reshape(rows, -1), val.reshape(rows, k)
    b = x.view(rows, k // 256, 16, 16)  # q6_k
    scale = b.abs().amax(-1) / 31
    d = _half(scale.amax(-1, keepdim=True) / 127)
    sc = torch.round(scale / d.clamp(min=1e-12)).clamp(-127, 127)
    q = torch.round(b / (d * sc).clamp(min=1e-12)[..., None]).clamp(-32, 31)
    val = q * (d * sc)[..., None]
    u = (q + 32).to(torch.uint8).reshape(rows, k // 256, 2, 4, 32)  # [half, element / 32 of the half, element]
    ql = torch.cat([(u[..., 0, :] & 15) | ((u[..., 2, :] & 15) << 4),
                    (u[..., 1, :] & 15) | ((u[..., 3, :] & 15) << 4)], -1)
    qh = (u[..., 0, :] >> 4) | (u[..., 1, :] >> 4 << 2) | (u[..., 2, :] >> 4 << 4) | (u[..., 3, :] >> 4 << 6)
    raw = torch.cat([ql.reshape(rows, -1, 128), qh.reshape(rows, -1, 64), sc.to(torch.int8).view(torch.uint8),
                     _bytes16(d[..., 0])], -1)
    return raw.reshape(rows, -1), val.reshape(rows, k)


def upload(t, ne, raw):
    """A weight in the library's own buffer type, as a model file's loader sets it."""
    return backend().tensor(TYPES[t], ne, raw.cpu().numpy())


# ---------------------------------------------------------------------------------------------- inputs, from the seed
def _gen(seed):
    return torch.Generator(DEV).manual_seed(int(seed))


def _weights(c, g, shapes):
    """[(bytes, values)] in the order that prepare and exact share."""
    return [weight(c["type"], n, k, g) for k, n in shapes]


def _mask(rows, past, n_kv):
    j, i = torch.arange(n_kv, device=DEV)[None], torch.arange(rows, device=DEV)[:, None]
    return torch.where(j <= past + i, 0.0, float("-inf")).half()


def _spans(rows, past):
    n_kv = (past + rows + 63) // 64 * 64
    return n_kv, (n_kv + 255) // 256 * 256  # positions read, rows of the cache


def _layer_shapes(c):
    h, f, q, kv = c["hidden"], c["ffn"], c["heads"] * 128, c["kv_heads"] * 128
    return [(h, q), (h, kv), (h, kv), (q, h), (h, f), (h, f), (f, h)]


def _layer_norms(c, g):
    return [1 + 0.1 * torch.randn(n, generator=g, device=DEV) for n in (c["hidden"], c["hidden"], 128, 128)]


def _caches(cap, past, width, g):
    out = torch.zeros(2, cap, width, device=DEV, dtype=torch.float16)
    out[:, :past] = torch.randn(2, past, width, generator=g, device=DEV).half()
    return out


def _expert_ids(c, g):
    return torch.randn(c["tokens"], c["experts"], generator=g, device=DEV).topk(c["top"], -1).indices.int()


# ------------------------------------------------------------------------------------------------------------ prepare
def prepare(c, seed):
    g, s = _gen(seed), State()
    {"product": _prepare_product, "attend": _prepare_attend, "moe": _prepare_moe, "layer": _prepare_layer,
     "decode": _prepare_decode}[c["kind"]](c, g, s)
    torch.cuda.synchronize()  # the inputs are there before the library's own stream reads them
    if c["kind"] == "decode":  # once as it is, so that the recording finds its scratch; then recorded
        be = backend()
        s.step()
        be.sync()
        be.graph_begin()
        s.step()
        s.graph = be.graph_end()
    return s


def run(s):
    if s.graph:
        backend().graph_launch(s.graph)
    else:
        s.step()
    return s.out


def _zeros(*shape):
    return torch.zeros(*shape, device=DEV)


def _prepare_product(c, g, s):
    be, m = backend(), c["m"]
    ws = [upload(c["type"], (c["k"], n), weight(c["type"], n, c["k"], g)[0]) for n in _sizes(c)]
    x = On(torch.randn(m, c["k"], generator=g, device=DEV))
    norm = On(1 + 0.1 * torch.randn(c["k"], generator=g, device=DEV))
    ys = [On(_zeros(m, n)) for n in _sizes(c)]
    s.out = [y.t for y in ys]
    if c["norm"]:
        s.step = lambda: be.mul_mat_fused(ws, x, ys, norm_w=norm, eps=EPS)
    elif len(ws) == 1:
        s.step = lambda: be.mul_mat(ws[0], x, ys[0])
    else:
        s.step = lambda: be.mul_mat_group(ws, x, ys)


def _heads(t, heads, rows, d):
    return On(t, (d, heads, rows), (4, 4 * d, 4 * d * heads))


def _attend_views(c, d, q_rot, cache, n_kv):
    """What FLASH_ATTN_EXT reads: [d, rows, heads] of q and [d, n_kv, kv heads] of the caches."""
    rows, heads, kv = c["rows"], c["heads"], c["kv_heads"]
    qv = On(q_rot, (d, rows, heads), (4, 4 * d * heads, 4 * d))
    return [qv] + [On(cache[i], (d, n_kv, kv), (2, 2 * d * kv, 2 * d)) for i in (0, 1)]


def _prepare_attend(c, g, s):
    be, rows, past, heads, kv, d = backend(), c["rows"], c["past"], c["heads"], c["kv_heads"], c["head_dim"]
    n_kv, cap = _spans(rows, past)
    q, k, v = (torch.randn(rows, n * d, generator=g, device=DEV) for n in (heads, kv, kv))
    qw, kw = (On(1 + 0.1 * torch.randn(d, generator=g, device=DEV)) for _ in range(2))
    cache = _caches(cap, past, kv * d, g)
    pos = On(torch.arange(past, past + rows, device=DEV, dtype=torch.int32))
    mask = On(_mask(rows, past, n_kv))
    q_rot, out = _zeros(rows, heads * d), On(_zeros(rows, heads, d))
    qv, kview, vview = _attend_views(c, d, q_rot, cache, n_kv)
    q3, k3, v3, qr3 = _heads(q, heads, rows, d), _heads(k, kv, rows, d), _heads(v, kv, rows, d), _heads(q_rot, heads, rows, d)
    kc, vc = On(cache[0]), On(cache[1])
    scale = 1 / math.sqrt(d)
    s.out = {"out": out.t, "cache": cache}
    s.keep = (q, k, v)
    if d == 128 and rows == 1 and heads // kv in (1, 2, 4):
        s.step = lambda: be.attn_decode(q3, k3, v3, qw, kw, pos, kc, vc, kview, vview, mask, out, EPS, ROPE_BASE, scale)
        return
    if d == 128:
        def step():
            be.qk_norm_rope_kv(q3, k3, v3, qw, kw, pos, qr3, kc, vc, EPS, ROPE_BASE)
            be.flash_attn_ext(qv, kview, vview, mask, out, scale)
    else:  # other head sizes: op after op
        qn, kn, k_rot = _zeros(rows, heads * d), _zeros(rows, kv * d), _zeros(rows, kv * d)
        qn3, kn3, kr3 = _heads(qn, heads, rows, d), _heads(kn, kv, rows, d), _heads(k_rot, kv, rows, d)
        kr2, v2 = On(k_rot), On(v)

        def step():
            be.rms_norm(q3, qn3, EPS, qw)
            be.rms_norm(k3, kn3, EPS, kw)
            be.rope(qn3, pos, qr3, d, ROPE_BASE)
            be.rope(kn3, pos, kr3, d, ROPE_BASE)
            be.set_rows(kr2, pos, kc)
            be.set_rows(v2, pos, vc)
            be.flash_attn_ext(qv, kview, vview, mask, out, scale)
    s.step = step


def _prepare_moe(c, g, s):
    be, h, f, e, top, n = backend(), c["hidden"], c["ffn"], c["experts"], c["top"], c["tokens"]
    gate, up = (upload(c["type"], (h, f, e), weight(c["type"], e * f, h, g)[0]) for _ in range(2))
    down = upload(c["type"], (f, h, e), weight(c["type"], e * h, f, g)[0])
    router = upload("f32", (h, e), weight("f32", e, h, g)[0])
    xt = torch.randn(n, h, generator=g, device=DEV)
    ids = On(_expert_ids(c, g))
    x, x3, logits = On(xt), On(xt, (h, 1, n)), On(_zeros(n, e))
    yg, yu, ya, yd = _zeros(n, top, f), _zeros(n, top, f), _zeros(n, top, f), On(_zeros(n, top, h))
    rows = [On(t, (f, top * n)) for t in (yg, yu, ya)]
    yg, yu, ya = On(yg), On(yu), On(ya)
    s.out = {"logits": logits.t, "gate": yg.t, "up": yu.t, "out": yd.t}

    def step():
        be.mul_mat(router, x, logits)
        be.mul_mat_id_group([gate, up], x3, ids, [yg, yu])
        be.swiglu(*rows)
        be.mul_mat_id(down, ya, ids, yd)
    s.step = step


def _prepare_layer(c, g, s):
    be, rows, past, h, f, heads, kv, d = (backend(), c["rows"], c["past"], c["hidden"], c["ffn"], c["heads"],
                                          c["kv_heads"], 128)
    n_kv, cap = _spans(rows, past)
    wq, wk, wv, wo, wg, wu, wd = (upload(c["type"], (k, n), weight(c["type"], n, k, g)[0]) for k, n in _layer_shapes(c))
    an, fn, qw, kw = (On(w) for w in _layer_norms(c, g))
    x = On(torch.randn(rows, h, generator=g, device=DEV))
    cache = _caches(cap, past, kv * d, g)
    pos = On(torch.arange(past, past + rows, device=DEV, dtype=torch.int32))
    mask = On(_mask(rows, past, n_kv))
    hn, x2, out = On(_zeros(rows, h)), On(_zeros(rows, h)), On(_zeros(rows, h))
    q, k, v = (_zeros(rows, n * d) for n in (heads, kv, kv))
    q_rot, att = _zeros(rows, heads * d), _zeros(rows, heads, d)
    o, gate, up, act, down = (On(_zeros(rows, n)) for n in (h, f, f, f, h))
    qv, kview, vview = _attend_views(c, d, q_rot, cache, n_kv)
    q3, k3, v3, qr3 = _heads(q, heads, rows, d), _heads(k, kv, rows, d), _heads(v, kv, rows, d), _heads(q_rot, heads, rows, d)
    qo, ko, vo, kc, vc = On(q), On(k), On(v), On(cache[0]), On(cache[1])
    att3, att2 = On(att), On(att, (heads * d, rows))
    scale = 1 / math.sqrt(d)
    s.out = {"out": out.t, "cache": cache}

    def step():
        be.rms_norm(x, hn, EPS, an)
        be.mul_mat_group([wq, wk, wv], hn, [qo, ko, vo])
        be.qk_norm_rope_kv(q3, k3, v3, qw, kw, pos, qr3, kc, vc, EPS, ROPE_BASE)
        be.flash_attn_ext(qv, kview, vview, mask, att3, scale)
        be.mul_mat(wo, att2, o)
        be.add(x, o, x2)
        be.rms_norm(x2, hn, EPS, fn)
        be.mul_mat_group([wg, wu], hn, [gate, up])
        be.swiglu(gate, up, act)
        be.mul_mat(wd, act, down)
        be.add(x2, down, out)
    s.step = step


def _prepare_decode(c, g, s):
    be, past, h, f, heads, kv, d, n_layers = (backend(), c["past"], c["hidden"], c["ffn"], c["heads"], c["kv_heads"],
                                              128, c["layers"])
    n_kv, cap = _spans(1, past)
    embd = upload(c["type"], (h, c["vocab"]), weight(c["type"], c["vocab"], h, g, 1.0)[0])
    final = On(1 + 0.1 * torch.randn(h, generator=g, device=DEV))
    token = On(torch.randint(0, c["vocab"], (1,), generator=g, device=DEV).int())
    pos, mask = On(torch.full((1,), past, device=DEV, dtype=torch.int32)), On(_mask(1, past, n_kv))
    x, hn, q, k, v = (_zeros(1, n) for n in (h, h, heads * d, kv * d, kv * d))
    att, gate, up = _zeros(1, heads, d), On(_zeros(1, f)), On(_zeros(1, f))
    x, hn, att3, att2 = On(x), On(hn), On(att), On(att, (heads * d, 1))
    qo, ko, vo = On(q), On(k), On(v)
    q3, k3, v3 = _heads(q, heads, 1, d), _heads(k, kv, 1, d), _heads(v, kv, 1, d)
    logits, pick = On(_zeros(1, c["vocab"])), On(torch.zeros(1, device=DEV, dtype=torch.int32))
    caches = torch.zeros(n_layers, 2, cap, kv * d, device=DEV, dtype=torch.float16)
    layers = []
    for i in range(n_layers):
        ws = [upload(c["type"], (a, b), weight(c["type"], b, a, g)[0]) for a, b in _layer_shapes(c)]
        norms = [On(w) for w in _layer_norms(c, g)]
        caches[i] = _caches(cap, past, kv * d, g)
        kc, vc = On(caches[i, 0]), On(caches[i, 1])
        views = [On(caches[i, j], (d, n_kv, kv), (2, 2 * d * kv, 2 * d)) for j in (0, 1)]
        layers.append((ws, norms, kc, vc, views))
    scale = 1 / math.sqrt(d)
    s.pick = pick.t  # not compared: two correct steps may pick either of two logits that are nearly equal
    s.out = {"logits": logits.t, "caches": caches}

    def step():
        be.get_rows(embd, token, x)
        for (wq, wk, wv, wo, wg, wu, wd), (an, fn, qw, kw), kc, vc, (kview, vview) in layers:
            be.mul_mat_fused([wq, wk, wv], x, [qo, ko, vo], norm_w=an, eps=EPS)
            be.attn_decode(q3, k3, v3, qw, kw, pos, kc, vc, kview, vview, mask, att3, EPS, ROPE_BASE, scale)
            be.mul_mat_fused([wo], att2, [x], residual=[x])
            be.mul_mat_fused([wg, wu], x, [gate, up], norm_w=fn, eps=EPS)
            be.mul_mat_fused([wd], gate, [x], glu_b=up, residual=[x])
        be.rms_norm(x, hn, EPS, final)
        be.mul_mat(embd, hn, logits)
        be.argmax(logits, pick)
    s.step = step


# -------------------------------------------------------------------------------------------------------------- exact
def _rounded(t, x):
    """Activations as a product of this weight type rounds them (x in any precision, rounded from 32 bits)."""
    x = x.float()
    if t == "f32":
        return x.double()
    if t == "f16":
        return x.half().double()
    if t == "q8_0":
        b = x.reshape(-1, 32)
        d = b.abs().amax(-1, keepdim=True)
        d = d / torch.full_like(d, 127)  # (by a plain number torch multiplies with its reciprocal)
        v = b * torch.where(d > 0, 1 / d, 0.0)
        q = torch.sign(v) * torch.floor(v.abs().double() + 0.5)  # halves away from zero
        return (q * d.half().double()).reshape(x.shape)
    b = x.reshape(-1, 256)
    big = b.gather(-1, b.abs().argmax(-1, keepdim=True))
    inv = torch.where(big != 0, torch.full_like(big, -127) / big, 0.0)
    q = torch.round(inv * b).clamp(max=127).double()
    return (q * torch.where(inv != 0, 1 / inv, 0.0).double()).reshape(x.shape)


def _mm(t, val, x):
    return _rounded(t, x) @ val.double().T


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, past, d):
    """x [rows, heads, d]; the angles are the 32-bit chain of products that defines them."""
    scale = np.float32(math.pow(ROPE_BASE, -2.0 / d))
    theta = torch.arange(past, past + x.shape[0], device=DEV).float()
    angles = []
    for _ in range(d // 2):
        angles.append(theta)
        theta = theta * float(scale)
    a = torch.stack(angles, -1).double()[:, None]
    x0, x1 = x[..., : d // 2], x[..., d // 2:]
    return torch.cat([x0 * a.cos() - x1 * a.sin(), x0 * a.sin() + x1 * a.cos()], -1)


def _attend_exact(q, k, v, qw, kw, cache, past, heads, kv, d):
    """[rows, heads, d] of the result; the new keys and values go into the cache."""
    rows = q.shape[0]
    q = _rope(_rms(q.double().reshape(rows, heads, d), qw), past, d).float().half().double()
    k = _rope(_rms(k.double().reshape(rows, kv, d), kw), past, d)
    cache[0, past:past + rows] = k.reshape(rows, -1).float().half()
    cache[1, past:past + rows] = v.reshape(rows, -1).float().half()
    kk, vv = (cache[i, :past + rows].double().reshape(-1, kv, d) for i in (0, 1))
    seen = torch.arange(past + rows, device=DEV)[None] <= past + torch.arange(rows, device=DEV)[:, None]
    out = torch.zeros(rows, heads, d, device=DEV, dtype=torch.float64)
    for h in range(heads):
        j = h // (heads // kv)
        s = (q[:, h] @ kk[:, j].T / math.sqrt(d)).masked_fill(~seen, float("-inf"))
        out[:, h] = torch.softmax(s, -1) @ vv[:, j]
    return out


def _silu(x):
    return x / (1 + torch.exp(-x))


def _layer_exact(c, vals, norms, x, cache, past):
    t = c["type"]
    wq, wk, wv, wo, wg, wu, wd = vals
    an, fn, qw, kw = norms
    hn = _rms(x, an)
    q, k, v = (_mm(t, w, hn) for w in (wq, wk, wv))
    att = _attend_exact(q, k, v, qw, kw, cache, past, c["heads"], c["kv_heads"], 128)
    x = x + _mm(t, wo, att.reshape(x.shape[0], -1))
    hn = _rms(x, fn)
    return x + _mm(t, wd, _silu(_mm(t, wg, hn)) * _mm(t, wu, hn))


def exact(c, seed):
    g = _gen(seed)
    if c["kind"] == "product":
        vals = [weight(c["type"], n, c["k"], g)[1] for n in _sizes(c)]
        x = torch.randn(c["m"], c["k"], generator=g, device=DEV)
        norm = 1 + 0.1 * torch.randn(c["k"], generator=g, device=DEV)
        return [_mm(c["type"], v, _rms(x.double(), norm) if c["norm"] else x) for v in vals]
    if c["kind"] == "attend":
        rows, past, heads, kv, d = c["rows"], c["past"], c["heads"], c["kv_heads"], c["head_dim"]
        q, k, v = (torch.randn(rows, n * d, generator=g, device=DEV) for n in (heads, kv, kv))
        qw, kw = (1 + 0.1 * torch.randn(d, generator=g, device=DEV) for _ in range(2))
        cache = _caches(_spans(rows, past)[1], past, kv * d, g)
        return {"out": _attend_exact(q, k, v, qw, kw, cache, past, heads, kv, d), "cache": None}
    if c["kind"] == "moe":
        h, f, e, top, n, t = c["hidden"], c["ffn"], c["experts"], c["top"], c["tokens"], c["type"]
        wg, wu = (weight(t, e * f, h, g)[1].view(e, f, h) for _ in range(2))
        wd = weight(t, e * h, f, g)[1].view(e, h, f)
        router = weight("f32", e, h, g)[1]
        x = torch.randn(n, h, generator=g, device=DEV)
        ids = _expert_ids(c, g).long()
        yg, yu = (torch.zeros(n, top, f, device=DEV, dtype=torch.float64) for _ in range(2))
        yd = torch.zeros(n, top, h, device=DEV, dtype=torch.float64)
        for i in range(e):
            row, slot = torch.nonzero(ids == i, as_tuple=True)
            if not row.numel():
                continue
            a, b = _mm(t, wg[i], x[row]), _mm(t, wu[i], x[row])
            yg[row, slot], yu[row, slot] = a, b
            yd[row, slot] = _mm(t, wd[i], _silu(a) * b)
        return {"logits": x.double() @ router.double().T, "gate": yg, "up": yu, "out": yd if n * top >= 512 else None}
    if c["kind"] == "layer":
        if c["rows"] < 64:
            return None
        vals = [weight(c["type"], n, k, g)[1] for k, n in _layer_shapes(c)]
        norms = _layer_norms(c, g)
        x = torch.randn(c["rows"], c["hidden"], generator=g, device=DEV)
        cache = _caches(_spans(c["rows"], c["past"])[1], c["past"], c["kv_heads"] * 128, g)
        return {"out": _layer_exact(c, vals, norms, x.double(), cache, c["past"]), "cache": None}
    return None
