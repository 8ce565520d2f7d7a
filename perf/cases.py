"""The work that is timed: what a program that serves a draft and a target from GGUF
blocks asks of this library, through its public entry points (laguna_hip).

A case is one pass of one kind:

  matvec   an M = 1 projection, once per layer of a stack: every layer's own weights
           and activations, as a token passes through a model (weights are not read
           twice within the memory-side cache's reach unless there is one layer)
  silu     the FFN's fused silu(gate) * up + down projection at M = 1, likewise
  block    a block of m tokens through one projection per layer (block verify, the
           draft's projections; f32 weights are what F16 / BF16 tensors become at load)
  verify   the LM head over a block's hidden states and the argmax of every row
  attn     attention of a block (or one token) over cached keys and values, per layer
  dequant  a whole tensor to f32, as loaders do with the types that are not served raw
  draft    the draft's block forward over its context
  target   one token through the dense target over its K/V cache, with the LM head

Weights have the magnitude of trained ones (N(0, 0.02), quantized by the formats' own
rules), activations and cached keys and values are N(0, 1), and norm weights lie around 1.
"""
import math
import os
import sys

import numpy as np
import torch

# the package of the tree that is the working folder
sys.path.insert(0, os.path.join(os.getcwd(), "laguna-raw-halo-strix_amd"))

import laguna_hip as lh  # noqa: E402

HD = 128  # head size of the draft and the target
TYPES = {"q4k": lh.Q4_K, "q8_0": lh.Q8_0, "f32": lh.F32, "f16": lh.F16, "q4k_t16": lh.Q4_K, "q8_0_t16": lh.Q8_0}
EPS, QK_EPS, ROPE_BASE = 1e-5, 1e-6, 500000.0


def listed():
    return [
        # One attention output projection by itself: the smallest call of a decode step,
        # where the launch and the host path count as much as the kernel.
        {"name": "matvec_q8_0_single", "kind": "matvec", "type": "q8_0", "k": 4096, "n": 4096, "layers": 1},
        # The FFN's gate or up projection of every layer of a 16-layer stack.
        {"name": "matvec_q4k_up", "kind": "matvec", "type": "q4k", "k": 4096, "n": 14336, "layers": 16},
        # The FFN's down projection with its activation, of every layer of such a stack.
        {"name": "silu_q4k_down", "kind": "silu", "type": "q4k", "k": 14336, "n": 4096, "layers": 16},
        # Block verify of 16 tokens straight over the file's blocks.
        {"name": "block_q4k_m16", "kind": "block", "type": "q4k", "x": "f32", "k": 4096, "n": 14336, "m": 16,
         "layers": 16},
        # A long, ragged verify block in bf16 over repacked weights, an odd number of rows.
        {"name": "block_q8_0_t16_m61", "kind": "block", "type": "q8_0_t16", "x": "bf16", "k": 4096, "n": 4099, "m": 61,
         "layers": 16},
        # A projection whose tensor was F16 or BF16 in the file: held in f32 since its load.
        {"name": "block_f32_m16", "kind": "block", "type": "f32", "x": "f32", "k": 4096, "n": 4096, "m": 16,
         "layers": 8},
        # The target's verdict on a block: logits of 16 tokens over the vocabulary, their argmax.
        {"name": "verify_head_m16", "kind": "verify", "type": "q4k", "k": 4096, "n": 151936, "m": 16},
        # A 32-token block over 4096 cached positions, grouped heads, four layers.
        {"name": "attn_r32_s4096", "kind": "attn", "heads": 32, "kv": 8, "hd": 128, "rows": 32, "seq": 4096,
         "layers": 4},
        # A whole FFN tensor decoded at load.
        {"name": "dequant_q8_0", "kind": "dequant", "type": "q8_0", "n": 4096 * 14336},
        # The draft at the length it usually runs, and at its longest block over a longer context.
        {"name": "draft_m16_c2048", "kind": "draft", "embd": 4096, "layers": 6, "m": 16, "ctx": 2048},
        {"name": "draft_m32_c4096", "kind": "draft", "embd": 4096, "layers": 6, "m": 32, "ctx": 4096},
        # The target's decode step.
        {"name": "target_c2048", "kind": "target", "embd": 4096, "layers": 6, "vocab": 151936, "ctx": 2048},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["matvec", "matvec", "silu", "block", "block", "verify", "attn", "dequant", "draft", "target"])
    c = {"kind": kind}
    if kind in ("matvec", "silu", "block"):
        c["type"] = rng.choice(["q4k", "q8_0"] if kind != "block" else ["q4k", "q8_0", "q4k_t16", "q8_0_t16", "f32"])
        k = 256 * _log(rng, 2, 80)
        if c["type"] == "q8_0" and rng.random() < 0.2:
            k += 32 * rng.randrange(1, 8)  # a hidden size of whole blocks that is no multiple of 256 (2880, 5152)
        c["k"], c["n"] = k, _log(rng, 64, 30000)
        while k * c["n"] > 80_000_000:
            c["n"] //= 2
        if kind == "block":
            c["x"] = rng.choice(["f32", "bf16"])
            c["m"] = rng.randrange(2, 65)
            if c["type"] == "f32":
                c["n"] = min(c["n"], 20_000_000 // k)
        c["layers"] = rng.choice([1, 2, 4, 8])
    elif kind == "verify":
        c.update(type=rng.choice(["q4k", "q8_0"]), k=256 * rng.randrange(4, 17), n=_log(rng, 8000, 152000),
                 m=rng.randrange(1, 17))
    elif kind == "attn":
        c["kv"] = rng.choice([1, 2, 4, 8])
        c["heads"] = c["kv"] * rng.choice([1, 2, 4])
        c["hd"] = rng.choice([64, 128, 128, 128, 256])
        c["rows"], c["seq"] = rng.randrange(1, 33), _log(rng, 64, 4096)
        c["seq"] = max(c["seq"], c["rows"])
        c["layers"] = rng.choice([1, 2, 4])
    elif kind == "dequant":
        c.update(type=rng.choice(["q4k", "q8_0", "f16"]), n=_log(rng, 200_000, 60_000_000))
        c["n"] = -(-c["n"] // 256) * 256
    elif kind == "draft":
        c.update(embd=rng.choice([1024, 2048, 4096]), layers=rng.randrange(1, 7), m=rng.randrange(1, 33),
                 ctx=rng.choice([0, _log(rng, 16, 4096), _log(rng, 16, 4096)]))
    else:
        c.update(embd=rng.choice([1024, 2048, 4096]), layers=rng.randrange(1, 7), vocab=_log(rng, 8000, 152000),
                 ctx=_log(rng, 1, 4096))
    return c


# ---- inputs


class _Memory:
    """A GpuBuffer's device memory as torch sees it (and what keeps it allocated)."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (buf.ptr, False),
                                         "strides": None, "version": 2}


def _view(buf, shape, typestr="<f4"):
    return torch.as_tensor(_Memory(buf, shape, typestr), device="cuda")


def _buffer(ctx, t):
    """A device buffer of the framework holding the tensor's bytes."""
    t = t.contiguous()
    b = lh.GpuBuffer(ctx, t.numel() * t.element_size())
    lh.check(lh.lib().lg_buf_copy(b.ptr, t.data_ptr(), b.size, ctx.stream))
    return b


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda") * std


def _half_bytes(t):
    return t.to(torch.float16).view(torch.uint8).reshape(*t.shape[:-1], 2 * t.shape[-1])


def _q4k(w):
    """f32 [blocks][256] -> raw Q4_K bytes [blocks][144]: per 32-element sub-block a
    6-bit scale and minimum of the super-block's f16 d and dmin, 4-bit quants."""
    s = w.view(-1, 8, 32)
    lo, hi = s.amin(-1).clamp(max=0.0), s.amax(-1)
    scale, mn = (hi - lo) / 15.0, -lo
    d = (scale.amax(-1, keepdim=True) / 63.0).clamp(min=2.0 ** -14).half().float()
    dm = (mn.amax(-1, keepdim=True) / 63.0).clamp(min=2.0 ** -14).half().float()
    sc = (scale / d).round().clamp(1, 63)
    m = (mn / dm).round().clamp(0, 63)
    q = ((s + (dm * m).unsqueeze(-1)) / (d * sc).unsqueeze(-1)).round().clamp(0, 15).to(torch.uint8)
    sc, m = sc.to(torch.uint8), m.to(torch.uint8)
    out = torch.empty(s.shape[0], 144, dtype=torch.uint8, device=w.device)
    out[:, 0:2], out[:, 2:4] = _half_bytes(d), _half_bytes(dm)
    out[:, 4:8] = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    out[:, 8:12] = m[:, :4] | ((m[:, 4:] >> 4) << 6)
    out[:, 12:16] = (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)
    q = q.view(-1, 4, 2, 32)
    out[:, 16:] = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)
    return out


def _q80(w):
    """f32 [blocks][32] -> raw Q8_0 bytes [blocks][34]."""
    d = w.abs().amax(-1, keepdim=True) / 127.0
    q = (w / d).round().clamp(-127, 127).to(torch.int8)
    return torch.cat([_half_bytes(d), q.view(torch.uint8)], 1)


PART = 1 << 25  # elements quantized or decoded at a time


def _weight(g, typ, k, n):
    """Raw bytes of a [k, n] tensor of trained magnitude (row i: elements i k ..)."""
    base = TYPES[typ]
    if base == lh.F32:
        return _normal(g, n * k, std=0.02).view(torch.uint8)
    if base == lh.F16:
        return _normal(g, n * k, std=0.02).half().view(torch.uint8)
    parts, block, quant = [], 256 if base == lh.Q4_K else 32, _q4k if base == lh.Q4_K else _q80
    for e in range(0, n * k, PART):
        parts.append(quant(_normal(g, min(PART, n * k - e), std=0.02).view(-1, block)).reshape(-1))
    return torch.cat(parts)


def _draft_shape(c):
    E = c["embd"]
    H = E // HD
    return E, H, max(1, H // 4), E * 7 // 2


DRAFT_PROJ = ("attn_q", "attn_k", "attn_v", "attn_gate", "attn_output", "ffn_gate", "ffn_up", "ffn_down")


def _layer_shapes(c):
    E, H, KV, FF = _draft_shape(c)
    return dict(zip(DRAFT_PROJ, ((E, H * HD), (E, KV * HD), (E, KV * HD), (E, H), (H * HD, E), (E, FF), (E, FF),
                                 (FF, E))))


def _layer_type(p):
    return "q8_0" if p == "attn_output" else "q4k"


def _layer(c, g):
    """One decoder layer: norm weights and raw projections (draft and target alike)."""
    E = c["embd"]
    t = {n: 1.0 + _normal(g, HD if n in ("attn_q_norm", "attn_k_norm") else E, std=0.1) for n in lh.DFLASH_NORMS}
    for p, (k, n) in _layer_shapes(c).items():
        t[p] = _weight(g, _layer_type(p), k, n)
    return t


def _inputs(c, seed):
    """The case's input tensors (torch, on the GPU), from the seed alone."""
    g, kind = _gen(seed), c["kind"]
    L, k, n = c.get("layers", 1), c.get("k"), c.get("n")
    if kind in ("matvec", "silu", "block", "verify"):
        m = c.get("m", 1)
        t = {"w": [_weight(g, c["type"], k, n) for _ in range(L)], "x": [_normal(g, m, k) for _ in range(L)]}
        if kind == "silu":
            t["up"] = [_normal(g, m, k) for _ in range(L)]
        if c.get("x") == "bf16":
            t["x"] = [x.to(torch.bfloat16) for x in t["x"]]
        return t
    if kind == "attn":
        q, kv = c["heads"] * c["hd"], c["kv"] * c["hd"]
        return {"q": [_normal(g, c["rows"], q) for _ in range(L)], "k": [_normal(g, c["seq"], kv) for _ in range(L)],
                "v": [_normal(g, c["seq"], kv) for _ in range(L)]}
    if kind == "dequant":
        return {"w": _weight(g, c["type"], n, 1)}
    E, H, KV, FF = _draft_shape(c)
    t = {"layers": [_layer(c, g) for _ in range(L)], "output_norm": 1.0 + _normal(g, E, std=0.1),
         "k": [_normal(g, c["ctx"], KV * HD) for _ in range(L)], "v": [_normal(g, c["ctx"], KV * HD) for _ in range(L)]}
    if kind == "draft":
        t.update(enc_aux_norm=1.0 + _normal(g, 3 * E, std=0.1), enc_output_norm=1.0 + _normal(g, E, std=0.1),
                 fc=_weight(g, "q4k", 3 * E, E), feat=_normal(g, c["m"], 3 * E), tok=_normal(g, c["m"], E))
    else:
        t.update(x=_normal(g, E), output=_weight(g, "q4k", E, c["vocab"]))
    return t


def _capture_layers(c):
    return [l for l in (1, 3, 5) if l < c["layers"]] or [0]


def prepare(case, seed):
    c, ctx, t = case, lh.VulkanContext(0), _inputs(case, seed)
    kind, s = c["kind"], {"case": case, "ctx": ctx}

    def buffers(ts):
        return [_buffer(ctx, x) for x in ts]

    def outputs(count, *shape):
        s["out"] = [lh.GpuBuffer(ctx, 4 * math.prod(shape)) for _ in range(count)]
        s["view"] = [_view(b, shape) for b in s["out"]]

    if kind in ("matvec", "silu", "block", "verify"):
        w = buffers(t["w"])
        s["type"] = TYPES[c["type"]]
        if c["type"].endswith("_t16"):
            w = [lh.repack_tiled(ctx, b, s["type"], c["k"], c["n"]) for b in w]
            s["type"] = lh.TILED[s["type"]]
        s["w"], s["x"], s["up"] = w, buffers(t["x"]), buffers(t.get("up", []))
        s["x_type"] = lh.BF16 if c.get("x") == "bf16" else lh.F32
        outputs(len(w), c.get("m", 1), c["n"])
        if kind == "verify":
            s["tokens"] = lh.GpuBuffer(ctx, 4 * c["m"])
            s["tokens_view"] = _view(s["tokens"], (c["m"],), "<i4")
    elif kind == "attn":
        s["q"], s["k"], s["v"] = buffers(t["q"]), buffers(t["k"]), buffers(t["v"])
        outputs(c["layers"], c["rows"], c["heads"] * c["hd"])
    elif kind == "dequant":
        s["w"] = _buffer(ctx, t["w"])
        outputs(1, c["n"])
    else:
        E, H, KV, FF = _draft_shape(c)
        layers = [{n: (_buffer(ctx, v)) for n, v in lay.items()} for lay in t["layers"]]
        for lay in layers:
            lay.update({p + "_dtype": TYPES[_layer_type(p)] for p in DRAFT_PROJ})
        norm = _buffer(ctx, t["output_norm"])
        if kind == "draft":
            cfg = lh.DFlashConfig(n_embd=E, n_heads=H, n_kv=KV, head_dim=HD, rope_dim=HD, n_ff=FF, n_aux=3,
                                  n_layers=c["layers"], rope_base=ROPE_BASE)
            s["model"] = lh.DFlashModel(ctx, cfg, {"enc_aux_norm": _buffer(ctx, t["enc_aux_norm"]),
                                                   "fc": _buffer(ctx, t["fc"]), "fc_dtype": lh.Q4_K,
                                                   "enc_output_norm": _buffer(ctx, t["enc_output_norm"]),
                                                   "output_norm": norm}, layers)
            s["model"].set_context([x.cpu().numpy() for x in t["k"]], [x.cpu().numpy() for x in t["v"]])
            s["feat"], s["tok"] = _buffer(ctx, t["feat"]), _buffer(ctx, t["tok"])
            outputs(1, c["m"], E)
        else:
            cfg = lh.TargetConfig(n_embd=E, n_heads=H, n_kv=KV, head_dim=HD, n_ff=FF, n_layers=c["layers"],
                                  n_vocab=c["vocab"], rope_dim=HD, rope_base=ROPE_BASE)
            s["model"] = lh.TargetModel(ctx, cfg, layers, output_norm=norm, output=_buffer(ctx, t["output"]),
                                        output_dtype=lh.Q4_K)
            s["x"], s["cache"] = _buffer(ctx, t["x"]), lh.TargetKvCache(s["model"], c["ctx"] + 1)
            s["kv"] = [_view(b, (c["layers"], c["ctx"] + 1, KV * HD)) for b in (s["cache"].k, s["cache"].v)]
            for l in range(c["layers"]):
                s["kv"][0][l, :-1], s["kv"][1][l, :-1] = t["k"][l], t["v"][l]
            s["capture"] = _capture_layers(c)
            shapes = {"logits": (c["vocab"],), "captured": (len(s["capture"]), E), "hidden": (E,)}
            s["out"] = {n: lh.GpuBuffer(ctx, 4 * math.prod(sh)) for n, sh in shapes.items()}
            s["view"] = {n: _view(s["out"][n], sh) for n, sh in shapes.items()}
    torch.cuda.synchronize()
    return s


def run(state):
    s = state
    c, ctx = s["case"], s["ctx"]
    kind = c["kind"]
    if kind == "matvec":
        for x, w, o in zip(s["x"], s["w"], s["out"]):
            lh.dispatch_proj_quant(ctx, x, w, o, c["k"], c["n"], s["type"])
    elif kind == "silu":
        for g, u, w, o in zip(s["x"], s["up"], s["w"], s["out"]):
            lh.dispatch_silu_mul_proj_quant(ctx, g, u, w, o, c["k"], c["n"], s["type"])
    elif kind in ("block", "verify"):
        for x, w, o in zip(s["x"], s["w"], s["out"]):
            lh.dispatch_proj_quant_batch(ctx, x, s["x_type"], w, o, c["k"], c["n"], c["m"], s["type"])
        if kind == "verify":
            lh.check(lh.lib().lg_dispatch_argmax(s["out"][0].ptr, c["n"], c["m"], c["n"], s["tokens"].ptr, ctx.stream))
            return [s["view"][0], s["tokens_view"]]
    elif kind == "attn":
        for q, k, v, o in zip(s["q"], s["k"], s["v"], s["out"]):
            lh.dispatch_mha_attn_seq(ctx, q, k, v, o, c["heads"], c["kv"], c["hd"], c["seq"], c["seq"] - c["rows"],
                                     rows=c["rows"])
    elif kind == "dequant":
        lh.dequant_to_f32_device(ctx, s["w"], s["w"].size, TYPES[c["type"]], c["n"], s["out"][0])
    elif kind == "draft":
        s["model"].forward_block_device(s["feat"], s["tok"], c["m"], s["out"][0])
    else:
        # the verify loop's rollback: the token's position again
        s["cache"]._c.len = c["ctx"]
        s["model"].forward_token_device(s["x"], s["capture"], s["out"]["captured"], s["out"]["logits"],
                                        hidden=s["out"]["hidden"], cache=s["cache"])
        return [s["view"]["logits"], s["view"]["captured"], s["view"]["hidden"], s["kv"][0], s["kv"][1]]
    return s["view"]


# ---- what a pass cannot do without


def _bytes(typ, k, n):
    base = TYPES[typ]
    return n * k * {lh.Q4_K: 144 / 256, lh.Q8_0: 34 / 32, lh.F32: 4, lh.F16: 2}[base]


def work(case):
    c = case
    kind, L, k, n, m = c["kind"], c.get("layers", 1), c.get("k"), c.get("n"), c.get("m", 1)
    if kind in ("matvec", "silu", "block", "verify"):
        x = m * k * (2 if c.get("x") == "bf16" else 4) * (2 if kind == "silu" else 1)
        return {"bytes": L * (_bytes(c["type"], k, n) + x + 4 * m * n) + (4 * m if kind == "verify" else 0),
                "flops": 2 * L * m * n * k}
    if kind == "attn":
        kv, q = c["seq"] * c["kv"] * c["hd"] * 4, c["rows"] * c["heads"] * c["hd"] * 4
        pairs = c["rows"] * c["seq"] - c["rows"] * (c["rows"] - 1) // 2  # causal
        return {"bytes": L * (2 * kv + 2 * q), "flops": 4 * L * pairs * c["heads"] * c["hd"]}
    if kind == "dequant":
        return {"bytes": _bytes(c["type"], n, 1) + 4 * n, "flops": 2 * n}
    E, H, KV, FF = _draft_shape(c)
    S = c["ctx"] + (2 * m if kind == "draft" else 1)
    b = sum(_bytes(_layer_type(p), *sh) for p, sh in _layer_shapes(c).items()) + 2 * c["ctx"] * KV * HD * 4
    rows = {"attn_k": 2 * m, "attn_v": 2 * m} if kind == "draft" else {}
    f = sum(2 * rows.get(p, m) * sh[0] * sh[1] for p, sh in _layer_shapes(c).items()) + 4 * m * S * H * HD
    b, f = L * b, L * f
    if kind == "draft":
        return {"bytes": b + _bytes("q4k", 3 * E, E) + 4 * m * 5 * E, "flops": f + 2 * m * 3 * E * E}
    return {"bytes": b + _bytes("q4k", E, c["vocab"]) + 4 * (c["vocab"] + 2 * E), "flops": f + 2 * E * c["vocab"]}


def tolerance(case):
    kind = case["kind"]
    if kind == "dequant":
        return "exact"
    return TOL[kind]


# About four times the largest error against 64 bits seen over the listed and drawn cases.
# The Q4_K products lie above the others: their f16 (or byte digit) parts of x meet the
# nibbles before the minimum is taken off, and the draft and the target carry that
# through every layer.
TOL = {"matvec": {"rel": 1.2e-5, "max": 2.1e-5}, "silu": {"rel": 2.8e-5, "max": 5.5e-5},
       "block": {"rel": 2.4e-5, "max": 5.5e-5}, "verify": {"rel": 1.5e-5, "max": 4.5e-5},
       "attn": {"rel": 6e-6, "max": 3.5e-5}, "draft": {"rel": 4e-4, "max": 2.5e-3},
       "target": {"rel": 6e-5, "max": 2.2e-3}}


# ---- the same in 64 bits, plain torch


def _decode(raw, typ):
    """f64 values of a tensor's raw bytes."""
    base = TYPES[typ]
    if base in (lh.F32, lh.F16):
        return raw.view(torch.float32 if base == lh.F32 else torch.float16).double()
    if base == lh.Q8_0:
        b = raw.view(-1, 34)
        return (b[:, :2].contiguous().view(torch.float16).double() * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1)
    b = raw.view(-1, 144)
    d, dm = (b[:, o:o + 2].contiguous().view(torch.float16).double() for o in (0, 2))
    s0, s1, s2 = b[:, 4:8], b[:, 8:12], b[:, 12:16]
    sc = torch.cat([s0 & 63, (s2 & 15) | ((s0 >> 6) << 4)], 1).double()
    mn = torch.cat([s1 & 63, (s2 >> 4) | ((s1 >> 6) << 4)], 1).double()
    q = b[:, 16:].reshape(-1, 4, 32)
    q = torch.stack([q & 15, q >> 4], 2).reshape(-1, 8, 32).double()
    return ((d * sc).unsqueeze(-1) * q - (dm * mn).unsqueeze(-1)).reshape(-1)


def _proj(x, raw, typ, k, n):
    """x W^T in f64, W decoded a part at a time."""
    per, row, parts = max(1, PART // k), raw.numel() // n, []
    for i in range(0, n, per):
        j = min(n, i + per)
        parts.append(x @ _decode(raw[i * row:j * row], typ).view(j - i, k).t())
    return torch.cat(parts, -1)


def _silu(g, u):
    return g / (1.0 + torch.exp(-g)) * u


def _rms(x, w, eps=EPS):
    return x * w.double() / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _rope(x, w, pos):
    """Per-head RMSNorm and NeoX rotation of rows [r][heads * HD] at positions pos[r];
    the angle is the f32 product of the f32 frequency table and the position."""
    i = np.arange(HD // 2, dtype=np.float32)
    freq = (np.float32(1.0) / np.power(np.float32(ROPE_BASE), (np.float32(2.0) * i) / np.float32(HD))).astype(np.float32)
    ang = torch.from_numpy((freq[None, :] * np.asarray(pos, np.float32)[:, None]).astype(np.float64)).to(x.device)
    cos, sin = ang.cos().unsqueeze(1), ang.sin().unsqueeze(1)
    y = _rms(x.view(x.shape[0], -1, HD), w, QK_EPS)
    a, b = y[..., :HD // 2], y[..., HD // 2:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1).reshape(x.shape[0], -1)


def _attention(q, k, v, heads, kv, hd, pos):
    """Causal attention of rows at positions pos over [S][kv * hd]."""
    R, S, G = q.shape[0], k.shape[0], heads // kv
    qh = q.double().view(R, kv, G, hd).permute(1, 0, 2, 3).reshape(kv, R * G, hd).contiguous()
    kh, vh = (t.double().view(S, kv, hd).permute(1, 0, 2).contiguous() for t in (k, v))
    s = torch.matmul(qh, kh.transpose(1, 2).contiguous()) / math.sqrt(hd)
    mask = torch.arange(S, device=q.device)[None, :] > torch.as_tensor(pos, device=q.device)[:, None]
    s = s.view(kv, R, G, S).masked_fill(mask[None, :, None, :], -math.inf).view(kv, R * G, S)
    o = torch.matmul(torch.softmax(s, -1), vh)
    return o.view(kv, R, G, hd).permute(1, 0, 2, 3).reshape(R, heads * hd)


def exact(case, seed):
    c, t = case, _inputs(case, seed)
    kind, k, n = c["kind"], c.get("k"), c.get("n")
    if kind == "silu":
        return [_proj(_silu(g.double(), u.double()), w, c["type"], k, n) for g, u, w in zip(t["x"], t["up"], t["w"])]
    if kind in ("matvec", "block", "verify"):
        y = [_proj(x.double(), w, c["type"], k, n) for x, w in zip(t["x"], t["w"])]
        return [y[0], None] if kind == "verify" else y
    if kind == "attn":
        pos = list(range(c["seq"] - c["rows"], c["seq"]))
        return [_attention(*a, c["heads"], c["kv"], c["hd"], pos) for a in zip(t["q"], t["k"], t["v"])]
    if kind == "dequant":
        return [_decode(t["w"], c["type"])]
    E, H, KV, FF = _draft_shape(c)
    sh = _layer_shapes(c)

    def proj(x, lay, p):
        return _proj(x, lay[p], _layer_type(p), *sh[p])

    def ffn(x, lay):
        h = _rms(x, lay["ffn_norm"])
        return x + proj(_silu(proj(h, lay, "ffn_gate"), proj(h, lay, "ffn_up")), lay, "ffn_down")

    C = c["ctx"]
    if kind == "draft":
        m = c["m"]
        inj, own = list(range(C, C + m)), list(range(C + m, C + 2 * m))
        f = t["feat"].double().view(m, 3, E)
        f = _rms(f, t["enc_aux_norm"].view(3, E)).view(m, 3 * E)
        enc = _rms(_proj(f, t["fc"], "q4k", 3 * E, E), t["enc_output_norm"])
        x = t["tok"].double()
        for i, lay in enumerate(t["layers"]):
            en, nx = _rms(enc, lay["attn_norm"]), _rms(x, lay["attn_norm"])
            kk = torch.cat([t["k"][i].double(), _rope(proj(en, lay, "attn_k"), lay["attn_k_norm"], inj),
                            _rope(proj(nx, lay, "attn_k"), lay["attn_k_norm"], own)])
            vv = torch.cat([t["v"][i].double(), proj(en, lay, "attn_v"), proj(nx, lay, "attn_v")])
            a = _attention(_rope(proj(nx, lay, "attn_q"), lay["attn_q_norm"], own), kk, vv, H, KV, HD, own)
            gate = torch.nn.functional.softplus(proj(nx, lay, "attn_gate"), threshold=1e9)
            x = x + proj((a.view(m, H, HD) * gate.unsqueeze(-1)).view(m, H * HD), lay, "attn_output")
            x = ffn(x, lay)
        return [_rms(x, t["output_norm"])]
    x, captured, kc, vc = t["x"].double().view(1, E), [], [], []
    for i, lay in enumerate(t["layers"]):
        if i in _capture_layers(c):
            captured.append(x[0])
        nx = _rms(x, lay["attn_norm"])
        kc.append(torch.cat([t["k"][i].double(), _rope(proj(nx, lay, "attn_k"), lay["attn_k_norm"], [C])]))
        vc.append(torch.cat([t["v"][i].double(), proj(nx, lay, "attn_v")]))
        a = _attention(_rope(proj(nx, lay, "attn_q"), lay["attn_q_norm"], [C]), kc[i], vc[i], H, KV, HD, [C])
        gate = torch.log1p(torch.exp(proj(nx, lay, "attn_gate")))
        x = x + proj((a.view(1, H, HD) * gate.unsqueeze(-1)).view(1, H * HD), lay, "attn_output")
        x = ffn(x, lay)
    h = _rms(x, t["output_norm"])
    return [_proj(h, t["output"], "q4k", E, c["vocab"])[0], torch.stack(captured), h[0], torch.stack(kc), torch.stack(vc)]
