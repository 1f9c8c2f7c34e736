"""Performance cases of the MTP verification round and of the decoder blocks around it.

Every case is one call sequence of the C ABI (include/q38.h) as a serving program makes it,
eager on the current stream, with handles, weights, workspaces and output buffers made
beforehand. Weights are random tensors in the formats the entry points take (packed VQ codes,
MLX affine words, INT8 / INT4 heads); sizes are those of the benchmark and the GPU tests:
hidden 2048, expert intermediate 512, 512 experts, top-10, vocabulary 151,936, 16 + 2 attention
heads of 256, 16 / 32 GatedDeltaNet heads of 128, 4 HyperConnection streams of rank 256.

Kinds (the "kind" of a case):
  chain  q38_verify_chain: the residual stream of 1-4 rows through several MoE layers ("row"
         or "ckpt", as below), each with its own weights, so that a layer's weights come from
         HBM as in a whole model
  hc     q38_verify_chain_hc: the same for the decoder's MLP half with its stream mixers
  moe    q38_moe_forward on one layer: wide verification (several slots, 5-16 rows) and
         prefill (17-2048 rows), in the layouts "row" (one FP16 scale per output row), "ckpt"
         (the reference checkpoints': a scale per 64 inputs and an affine shared expert),
         "u8" (per-dimension INT8 / U8 books) and "mixed" (two geometries side by side)
  head   q38_head_greedy: the Q8 LM head with its exact argmax
  draft  q38_mtp_forward_decode: one step of the MTP draft head
  gdn    q38_gdn_verify over several linear-attention layers
  attn   q38_attn_verify over several full-attention layers with their KV caches
"""
from __future__ import annotations

import ctypes as C
import math
import os
import sys

import torch

sys.path.insert(0, os.path.join(os.getcwd(), "qwen38-flash.cpp_amd"))
import q38  # noqa: E402

H, I, E, K = 2048, 512, 512, 10
VOCAB = 151936
HC, RANK, GROUP = 4, 256, 64
GDN_HK, GDN_HV, GDN_D = 16, 32, 128
ATT_HQ, ATT_HKV, ATT_D, ATT_ROT, ATT_THETA = 16, 2, 256, 64, 1e7
EPS = 1e-6
SHARED_BITS, SHARED_GROUP = 8, 64
ZIPF_S, ZIPF_TAU = 1.1, 0.28
MOE_FORMATS = ("row", "ckpt", "u8", "mixed")

_ctx = None


def ctx():
    global _ctx
    if _ctx is None:
        _ctx = q38.Ctx(torch.cuda.current_device())
    return _ctx


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one token at a time through a stack of layers: serial decode, the smallest call
        {"name": "chain_r1", "kind": "chain", "format": "row", "rows": 1, "layers": 8},
        # the verification of three drafts and the current token
        {"name": "chain_r4", "kind": "chain", "format": "row", "rows": 4, "layers": 8},
        # the same width through the decoder's MLP half with its stream mixers
        {"name": "mlp_half_r4", "kind": "hc", "rows": 4, "layers": 4, "bits": 4},
        # a ragged batch of slots on a layer in the checkpoints' layout
        {"name": "moe_ckpt_r13", "kind": "moe", "format": "ckpt", "rows": 13, "zipf": False},
        # four slots of four rows on a mixed-geometry layer
        {"name": "moe_mixed_r16", "kind": "moe", "format": "mixed", "rows": 16, "zipf": False},
        # a prompt chunk with skewed expert popularity
        {"name": "prefill_row_r512", "kind": "moe", "format": "row", "rows": 512, "zipf": True},
        # the longest prompt chunk, in the checkpoints' layout
        {"name": "prefill_ckpt_r2048", "kind": "moe", "format": "ckpt", "rows": 2048, "zipf": False},
        # the target tokens of a verification
        {"name": "head_r4", "kind": "head", "rows": 4, "vocab": VOCAB},
        # one draft token of one request
        {"name": "draft_r1", "kind": "draft", "rows": 1, "vocab": VOCAB},
        # the linear-attention half of three decoder layers
        {"name": "gdn_r4", "kind": "gdn", "rows": 4, "layers": 3, "bits": 8, "group": 64},
        # the full-attention half of three decoder layers, a short context
        {"name": "attn_r4_t4096", "kind": "attn", "rows": 4, "layers": 3, "tokens": 4096, "bits": 8, "group": 64},
        # a long copied draft (22 tokens) on a long, odd context
        {"name": "attn_r23_t30001", "kind": "attn", "rows": 23, "layers": 3, "tokens": 30001, "bits": 8, "group": 64},
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("chain", "hc", "moe", "moe", "prefill", "prefill", "head", "draft", "gdn", "gdn", "attn",
                       "attn"))
    if kind == "chain":
        return {"kind": "chain", "format": rng.choice(("row", "ckpt")), "rows": rng.randint(1, 4),
                "layers": rng.randint(1, 7)}
    if kind == "hc":
        return {"kind": "hc", "rows": rng.randint(1, 16), "layers": rng.randint(1, 3), "bits": rng.choice((4, 8))}
    if kind == "moe":
        return {"kind": "moe", "format": rng.choice(MOE_FORMATS), "rows": rng.randint(5, 16),
                "zipf": rng.random() < 0.5}
    if kind == "prefill":
        return {"kind": "moe", "format": rng.choice(("row", "ckpt")), "rows": _log_int(rng, 17, 2047),
                "zipf": rng.random() < 0.5}
    if kind == "head":
        return {"kind": "head", "rows": rng.randint(1, 16), "vocab": 16 * rng.randint(2000, VOCAB // 16)}
    if kind == "draft":
        return {"kind": "draft", "rows": rng.randint(1, 4), "vocab": 16 * rng.randint(2000, VOCAB // 16)}
    if kind == "gdn":
        return {"kind": "gdn", "rows": _log_int(rng, 1, 64), "layers": rng.randint(1, 3), "bits": rng.choice((4, 8)),
                "group": rng.choice((32, 64, 128))}
    return {"kind": "attn", "rows": _log_int(rng, 1, 64), "layers": rng.randint(1, 3),
            "tokens": _log_int(rng, 64, 32768), "bits": rng.choice((4, 8)), "group": rng.choice((32, 64, 128))}


# ------------------------------------------------------------------ tensors
class _Handles:
    """Handles of one state, given back with it."""

    def __init__(self):
        self._drop = []

    def add(self, handle, destroy):
        self._drop.append((handle, destroy))
        return handle

    def __del__(self):
        while self._drop:
            handle, destroy = self._drop.pop()
            destroy(handle)


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed & 0x7FFFFFFF)


def _words(g, *shape):
    return torch.randint(-(1 << 31), 1 << 31, shape, generator=g, device="cuda", dtype=torch.int64).to(torch.int32)


def _normal(g, shape, sd, dtype=torch.bfloat16):
    return (torch.randn(shape, generator=g, device="cuda") * sd).to(dtype)


def _uniform(g, shape, lo, hi, dtype):
    return (torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo).to(dtype)


def _affine(g, out, n_in, bits, group, spread=0.02):
    """An MLX affine projection: packed words, bf16 scales and biases, weights centred with
    the given spread."""
    w = _words(g, out, n_in * bits // 32)
    s = _uniform(g, (out, n_in // group), 0.5, 1.5, torch.float32) * (spread * 4 / (1 << bits))
    b = -s * (((1 << bits) - 1) / 2) + torch.randn(s.shape, generator=g, device="cuda") * (0.05 * spread)
    return w, s.to(torch.bfloat16), b.to(torch.bfloat16)


def _p(t):
    return t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _zipf(g):
    rank = torch.randperm(E, generator=g, device="cuda").double() + 1
    return (-ZIPF_S * ZIPF_TAU * torch.log(rank)).float()


# ------------------------------------------------------------------ MoE layers
def _moe_layer(g, handles, fmt, zipf=False):
    """A layer's tensors and handle. Row scales give outputs of about a tenth of the unit
    residual stream."""
    t = {"format": fmt, "router": _normal(g, (E, H), 0.02), "wsg": _normal(g, (H,), 0.02)}
    ins, outs = (H, H, I), (I, I, H)
    h = q38.P()
    if fmt == "mixed":
        d = q38.desc(mixed=1)
        w = q38.MoeMixedWeights()
        w.router, w.shared_gate = _p(t["router"]), _p(t["wsg"])
        for p in range(3):
            for bank, dim, bits, n in (("d4", 4, 8, E // 2 + 1), ("d8", 8, 14, E // 2)):
                t[f"codes_{bank}{p}"] = _words(g, n, outs[p], q38.words_per_row(ins[p], dim, bits))
                t[f"scales_{bank}{p}"] = _uniform(g, (n, outs[p]), 0.012, 0.035, torch.float16)
            t[f"books_d4{p}"] = _normal(g, (256, 4), 1.0, torch.float16)
            t[f"books_d8{p}"] = torch.randint(-127, 128, (16384, 8), generator=g, device="cuda", dtype=torch.int8)
            t[f"book_scale{p}"] = 2.0 ** -6
            w.codes_d4[p], w.scales_d4[p], w.books_d4[p] = (_p(t[f"{n}_d4{p}"]) for n in ("codes", "scales", "books"))
            w.codes_d8[p], w.scales_d8[p], w.books_d8[p] = (_p(t[f"{n}_d8{p}"]) for n in ("codes", "scales", "books"))
            w.book_scales_d8[p] = 0x2400  # 2^-6 as fp16
        q38.check(q38.lib.q38_moe_layer_create_mixed(ctx().h, C.byref(d), C.byref(w), C.byref(h)))
    else:
        ckpt = fmt == "ckpt"
        d = q38.desc(gu_group=GROUP if ckpt else None, down_group=GROUP if ckpt else None,
                     book_format=q38.Q38_CB_U8_PERDIM if fmt == "u8" else q38.Q38_CB_FP16)
        n = E if ckpt else E + 1
        w = q38.MoeWeights()
        w.router, w.shared_gate = _p(t["router"]), _p(t["wsg"])
        for p in range(3):
            t[f"codes{p}"] = _words(g, n, outs[p], q38.words_per_row(ins[p], 8, 14))
            t[f"scales{p}"] = _uniform(g, (n, outs[p], ins[p] // GROUP if ckpt else 1), 0.012, 0.035, torch.float16)
            t[f"books{p}"] = _normal(g, (16384, 8), 1.0, torch.float16)
            w.codes[p], w.scales[p], w.books[p] = (_p(t[f"{k}{p}"]) for k in ("codes", "scales", "books"))
        if ckpt:
            a = q38.AffineShared(bits=SHARED_BITS, group=SHARED_GROUP, inter=I, scale_dtype=0)
            for p in range(3):
                t[f"sw{p}"], t[f"ss{p}"], t[f"sb{p}"] = _affine(g, outs[p], ins[p], SHARED_BITS, SHARED_GROUP)
                a.weight[p], a.scales[p], a.biases[p] = _p(t[f"sw{p}"]), _p(t[f"ss{p}"]), _p(t[f"sb{p}"])
            q38.check(q38.lib.q38_moe_layer_create_affine_shared(ctx().h, C.byref(d), C.byref(w), C.byref(a),
                                                                 C.byref(h)))
        else:
            q38.check(q38.lib.q38_moe_layer_create(ctx().h, C.byref(d), C.byref(w), C.byref(h)))
    handles.add(h, q38.lib.q38_moe_layer_destroy)
    t["desc"], t["h"] = d, h
    if zipf:
        t["bias"] = _zipf(g)
        q38.check(q38.lib.q38_moe_layer_set_router_bias(h, _p(t["bias"])))
    return t


def _unpack(words, dim_bits):
    """[..., words] int32 of 32-code blocks, LSB first -> [..., codes] int64."""
    bits = dim_bits
    w = words.reshape(*words.shape[:-1], -1, bits).long() & 0xFFFFFFFF
    at = torch.arange(32, device=words.device) * bits
    lo, sh = at // 32, at % 32
    hi = torch.clamp(lo + 1, max=bits - 1)
    v = (w[..., lo] >> sh) | torch.where(sh + bits > 32, w[..., hi] << (32 - sh), torch.zeros_like(w[..., hi]))
    return (v & ((1 << bits) - 1)).reshape(*words.shape[:-1], -1)


def _dequant_affine(w, s, b, bits, group):
    sh = torch.arange(32 // bits, device=w.device) * bits
    q = (((w.long() & 0xFFFFFFFF)[..., None] >> sh) & ((1 << bits) - 1)).reshape(w.shape[0], -1).double()
    return q * s.double().repeat_interleave(group, 1) + b.double().repeat_interleave(group, 1)


def _book(t, p):
    """The [2^14, 8] float64 codebook of a uniform layer. Per-dimension books are 8-bit values
    with an FP16 scale per dimension: centred for the gate, with an offset for up and down."""
    b = t[f"books{p}"].double()
    if t["format"] != "u8":
        return b
    lo, hi = b.float().min(0).values, b.float().max(0).values
    scale = (hi - lo) / 255
    v = (b.float() if p == 0 else b.float() - lo) / scale
    q = torch.copysign(torch.floor(v.abs() + 0.5), v)
    q = q.clamp(-128, 127) if p == 0 else q.clamp(0, 255)
    return q.double() * scale.half().double() + (0.0 if p == 0 else lo.half().double())


def _expert(t, e, p):
    """The dequantised [OUT, IN] float64 weights of expert e's projection p."""
    if t["format"] == "mixed":
        bank, bits = ("d4", 8) if e % 2 == 0 else ("d8", 14)
        codes = _unpack(t[f"codes_{bank}{p}"][e // 2], bits)
        book = t[f"books_{bank}{p}"].double() * (1.0 if bank == "d4" else t[f"book_scale{p}"])
        return book[codes].reshape(codes.shape[0], -1) * t[f"scales_{bank}{p}"][e // 2].double()[:, None]
    codes = _unpack(t[f"codes{p}"][e], 14)
    w = _book(t, p)[codes].reshape(codes.shape[0], -1)
    s = t[f"scales{p}"][e].double()
    return w * s.repeat_interleave(w.shape[1] // s.shape[1], 1)


def _swiglu(x, gate, up, down):
    g = x @ gate.T
    return (g * torch.sigmoid(g) * (x @ up.T)) @ down.T


def _moe_exact(t, x):
    """The layer on x [rows, H] float64 (bf16 values): routing by the BF16 router logits, as
    the interface states it."""
    logits = (x @ t["router"].double().T).to(torch.bfloat16).double()
    if "bias" in t:
        logits = (logits.float() + t["bias"]).double()
    order = torch.sort(logits, dim=1, descending=True, stable=True).indices[:, :K]
    prob = torch.softmax(logits, 1).gather(1, order)
    prob = prob / prob.sum(1, keepdim=True)
    y = torch.zeros_like(x)
    for e in torch.unique(order).tolist():
        r, k = (order == e).nonzero(as_tuple=True)
        y.index_add_(0, r, prob[r, k][:, None] * _swiglu(x[r], *(_expert(t, e, p) for p in range(3))))
    if t["format"] == "ckpt":
        shared = [_dequant_affine(t[f"sw{p}"], t[f"ss{p}"], t[f"sb{p}"], SHARED_BITS, SHARED_GROUP) for p in range(3)]
    else:
        shared = [_expert(t, E, p) for p in range(3)]
    gate = torch.sigmoid(x @ t["wsg"].double())
    return y + gate[:, None] * _swiglu(x, *shared)


def _rms(v, eps=EPS):
    return v / torch.sqrt((v * v).mean(-1, keepdim=True) + eps)


def _bf(v):
    return v.to(torch.bfloat16).double()


# ------------------------------------------------------------------ chain: MoE layers with residual
def _chain_prepare(case, g):
    n, rows = case["layers"], case["rows"]
    hs = _Handles()
    layers = [_moe_layer(g, hs, case["format"]) for _ in range(n)]
    ws = torch.empty(q38.lib.q38_moe_workspace_size(C.byref(layers[0]["desc"]), rows), dtype=torch.uint8, device="cuda")
    x = _normal(g, (rows, H), 1.0)
    return {"layers": layers, "array": (q38.P * n)(*[t["h"] for t in layers]), "x": x, "h": torch.empty_like(x),
            "ws": ws, "n": n, "rows": rows, "handles": hs}


def _chain_run(s):
    s["h"].copy_(s["x"])  # the embedding rows, which the layers then update in place
    q38.check(q38.lib.q38_verify_chain(s["array"], s["n"], _p(s["h"]), s["rows"], EPS, None, _p(s["ws"]),
                                       s["ws"].numel(), _stream()))
    return s["h"]


def _chain_exact(s):
    if s["n"] > 1:
        return None  # the next layers' routing is a step function of the 16-bit stream
    h = s["x"].double()
    return h + _moe_exact(s["layers"][0], _bf(_rms(h)))


# ------------------------------------------------------------------ hc: the decoder's MLP half
def _mixer(g, hs, bits):
    t = {"norm": _normal(g, (HC * H,), 0.1)}
    for name, out, n_in in (("down", RANK, HC * H), ("up", HC * H, RANK), ("inj", HC, HC * H)):
        t[f"{name}_w"], t[f"{name}_s"], t[f"{name}_b"] = _affine(g, out, n_in, bits, GROUP)
    m = q38.Hc(ctx(), q38.HcDesc(H, HC, RANK, bits, GROUP, 1, EPS), t)
    hs.add(m.h, q38.lib.q38_hc_destroy)
    return t, m


def _hc_prepare(case, g):
    n, rows = case["layers"], case["rows"]
    hs = _Handles()
    layers = [_moe_layer(g, hs, "row") for _ in range(n)]
    mixers = [_mixer(g, hs, case["bits"]) for _ in range(n)]
    ws = torch.empty(q38.lib.q38_verify_chain_hc_workspace_size(C.byref(layers[0]["desc"]), C.byref(mixers[0][1].desc),
                                                                rows), dtype=torch.uint8, device="cuda")
    x = _normal(g, (rows, HC * H), 1.0)
    return {"layers": layers, "mixers": mixers, "array": (q38.P * n)(*[t["h"] for t in layers]),
            "marray": (q38.P * n)(*[m.h for _, m in mixers]), "x": x, "h": torch.empty_like(x), "ws": ws, "n": n,
            "rows": rows, "bits": case["bits"], "handles": hs}


def _hc_run(s):
    s["h"].copy_(s["x"])
    q38.check(q38.lib.q38_verify_chain_hc(s["array"], s["marray"], s["n"], _p(s["h"]), s["rows"], _p(s["ws"]),
                                          s["ws"].numel(), _stream()))
    return s["h"]


def _hc_exact(s):
    if s["n"] > 1:
        return None  # (as for the chain)
    t, _ = s["mixers"][0]
    h = s["x"].double().reshape(s["rows"], HC, H)
    xn = _rms(h) * (1.0 + t["norm"].double()).reshape(HC, H)
    down, up, inj = (_dequant_affine(t[f"{k}_w"], t[f"{k}_s"], t[f"{k}_b"], s["bits"], GROUP)
                     for k in ("down", "up", "inj"))
    flat = xn.reshape(s["rows"], HC * H)
    v = flat @ down.T / HC
    gate = torch.sigmoid((v * torch.sigmoid(v)) @ up.T).reshape(s["rows"], HC, H)
    mixed = (gate * xn).sum(1) / HC
    y = _moe_exact(s["layers"][0], _bf(mixed))
    weight = 2.0 * torch.sigmoid(flat @ inj.T / HC)
    return (h + y[:, None, :] * weight[:, :, None]).reshape(s["rows"], HC * H)


# ------------------------------------------------------------------ moe: one layer
def _moe_prepare(case, g):
    hs = _Handles()
    t = _moe_layer(g, hs, case["format"], case["zipf"])
    x = _rms(torch.randn((case["rows"], H), generator=g, device="cuda")).to(torch.bfloat16)
    ws = torch.empty(q38.lib.q38_moe_workspace_size(C.byref(t["desc"]), case["rows"]), dtype=torch.uint8, device="cuda")
    return {"layer": t, "x": x, "y": torch.empty_like(x), "ws": ws, "rows": case["rows"], "handles": hs}


def _moe_run(s):
    q38.check(q38.lib.q38_moe_forward(s["layer"]["h"], _p(s["x"]), s["rows"], _p(s["y"]), None, _p(s["ws"]),
                                      s["ws"].numel(), _stream()))
    return s["y"]


def _moe_exact_case(s):
    return _moe_exact(s["layer"], s["x"].double())


# ------------------------------------------------------------------ head: Q8 logits and exact argmax
def _head_prepare(case, g):
    hs = _Handles()
    v = case["vocab"]
    w = torch.randint(-127, 128, (v, H), generator=g, device="cuda", dtype=torch.int8)
    s = _uniform(g, (v,), 0.0002, 0.0004, torch.float16)
    head = q38.Head(ctx(), q38.Q38_HEAD_Q8, v, H, weights=w, scales=s)
    hs.add(head.h, q38.lib.q38_head_destroy)
    rows = case["rows"]
    x = _rms(torch.randn((rows, H), generator=g, device="cuda")).to(torch.bfloat16)
    ws = torch.empty(head.workspace_size(rows), dtype=torch.uint8, device="cuda")
    return {"w": w, "s": s, "head": head.h, "x": x, "rows": rows, "ws": ws, "handles": hs,
            "argmax": torch.empty(rows, dtype=torch.int32, device="cuda"),
            "logit": torch.empty(rows, dtype=torch.float32, device="cuda")}


def _head_run(s):
    q38.check(q38.lib.q38_head_greedy(s["head"], _p(s["x"]), s["rows"], _p(s["argmax"]), _p(s["logit"]), _p(s["ws"]),
                                      s["ws"].numel(), _stream()))
    return {"argmax": s["argmax"], "logit": s["logit"]}


def _head_exact(s):
    x = s["x"].double()
    logits = torch.cat([(x @ s["w"][i:i + 16384].double().T) * s["s"][i:i + 16384].double()
                        for i in range(0, s["w"].shape[0], 16384)], 1)
    best = logits.max(1)
    return {"argmax": best.indices.to(torch.int32), "logit": best.values}


# ------------------------------------------------------------------ draft: one step of the MTP head
def _draft_prepare(case, g):
    hs = _Handles()
    rows, vocab = case["rows"], case["vocab"]
    layer = _moe_layer(g, hs, "row")
    fc = []
    for _ in range(2):
        w = torch.randint(-127, 128, (H, H), generator=g, device="cuda", dtype=torch.int8)
        s = _uniform(g, (H,), 0.0002, 0.0004, torch.float16)
        hd = q38.Head(ctx(), q38.Q38_HEAD_Q8, H, H, weights=w, scales=s)
        hs.add(hd.h, q38.lib.q38_head_destroy)
        fc.append((w, s, hd.h))
    qw = torch.randint(0, 256, (vocab, H // 2), generator=g, device="cuda", dtype=torch.uint8)
    qs = _uniform(g, (vocab, H // 64), 0.003, 0.006, torch.float16)
    q4 = q38.Head(ctx(), q38.Q38_HEAD_Q4G64, vocab, H, weights=qw, scales=qs)
    hs.add(q4.h, q38.lib.q38_head_destroy)
    h = q38.P()
    seed = int(torch.randint(1 << 30, (1,), generator=g, device="cuda"))
    q38.check(q38.lib.q38_mtp_head_create(ctx().h, layer["h"], fc[0][2], fc[1][2], q4.h, seed, EPS, C.byref(h)))
    hs.add(h, q38.lib.q38_mtp_head_destroy)
    x = _normal(g, (rows, H), 1.0)
    return {"layer": layer, "fc": fc, "qw": qw, "qs": qs, "h": h, "x": x, "rows": rows, "handles": hs, "seed": seed,
            "tokens": torch.randint(vocab, (rows,), generator=g, device="cuda", dtype=torch.int32),
            "logits": torch.empty((rows, vocab), dtype=torch.float32, device="cuda"), "out": torch.empty_like(x),
            "ws": torch.empty(q38.lib.q38_mtp_workspace_size(h, rows), dtype=torch.uint8, device="cuda")}


def _draft_run(s):
    q38.check(q38.lib.q38_mtp_forward_decode(s["h"], _p(s["x"]), _p(s["tokens"]), s["rows"], _p(s["logits"]),
                                             _p(s["out"]), None, _p(s["ws"]), s["ws"].numel(), _stream()))
    return {"logits": s["logits"], "stream": s["out"]}


_MASK = (1 << 64) - 1
_GOLDEN, _MUL1, _MUL2 = 0x9E3779B97F4A7C15, 0xBF58476D1CE4E5B9, 0x94D049BB133111EB


def _mix(z):
    z = ((z ^ (z >> 30)) * _MUL1) & _MASK
    z = ((z ^ (z >> 27)) * _MUL2) & _MASK
    return z ^ (z >> 31)


def _embedding(seed, tokens):
    """The seeded token embedding in the place of a table: element i of token t's row is a
    Box-Muller normal of elements 2 (t H + i) and the next of the splitmix64 stream of
    (seed, layer 0xFFFF, tensor 21), rounded to bf16."""
    key = _mix((_mix((_mix(seed) + _GOLDEN * 0x10000) & _MASK) + _GOLDEN * 22) & _MASK)
    rows = []
    for t in tokens:
        row = []
        for i in range(t * H, (t + 1) * H):
            a, b = (_mix((key + _GOLDEN * (2 * i + j + 1)) & _MASK) >> 11 for j in (0, 1))
            r = math.sqrt(-2.0 * math.log((a + 1) * 2.0 ** -53))
            row.append(r * math.cos(6.283185307179586 * (b * 2.0 ** -53)))
        rows.append(row)
    return _bf(torch.tensor(rows, dtype=torch.float64, device="cuda"))


def _draft_exact(s):
    e = _embedding(s["seed"], s["tokens"].tolist())
    pe, ph = (_bf(_rms(v)) @ w.double().T * sc.double() for v, (w, sc, _) in zip((e, s["x"].double()), s["fc"]))
    x = _bf(pe + ph)
    out = x + _moe_exact(s["layer"], _bf(_rms(x)))
    f = _rms(out)
    logits = torch.empty(s["logits"].shape, dtype=torch.float64, device="cuda")
    for i in range(0, logits.shape[1], 16384):
        n = s["qw"][i:i + 16384].long()
        q = torch.stack([n & 15, n >> 4], -1).reshape(n.shape[0], H)
        w = torch.where(q > 7, q - 16, q).double() * s["qs"][i:i + 16384].double().repeat_interleave(64, 1)
        logits[:, i:i + 16384] = f @ w.T
    return {"logits": logits, "stream": out}


# ------------------------------------------------------------------ gdn: linear-attention layers
def _gdn_prepare(case, g):
    hs = _Handles()
    rows, bits, n, group = case["rows"], case["bits"], case["layers"], case["group"]
    kw, vw = GDN_HK * GDN_D, GDN_HV * GDN_D
    c = 2 * kw + vw
    layers = []
    for _ in range(n):
        t = {"proj": [_affine(g, o, i, bits, group) for o, i in ((c, H), (vw, H), (GDN_HV, H), (GDN_HV, H), (H, vw))],
             "conv": _normal(g, (c, 4), 0.5), "a_log": torch.log(_uniform(g, (GDN_HV,), 1.0, 16.0, torch.float32)),
             "dt": _normal(g, (GDN_HV,), 0.5), "norm": _uniform(g, (GDN_D,), 0.5, 1.5, torch.bfloat16)}
        d = q38.GdnDesc(H, GDN_HK, GDN_HV, GDN_D, GDN_D, 4, bits, group, 0, 0, EPS)
        w = q38.GdnWeights()
        for p in range(5):
            w.weight[p], w.scales[p], w.biases[p] = (_p(v) for v in t["proj"][p])
        w.conv, w.a_log, w.dt_bias, w.norm = _p(t["conv"]), _p(t["a_log"]), _p(t["dt"]), _p(t["norm"])
        h = q38.P()
        q38.check(q38.lib.q38_gdn_create(ctx().h, C.byref(d), C.byref(w), C.byref(h)))
        t["h"] = hs.add(h, q38.lib.q38_gdn_destroy)
        elems = q38.lib.q38_gdn_state_bytes(h) // 2
        t["x"] = _normal(g, (rows, H), 1.0)
        t["origin"] = _normal(g, (elems,), 0.05)
        t["ckpt"] = torch.empty((rows, elems), dtype=torch.bfloat16, device="cuda")
        t["out"] = torch.empty_like(t["x"])
        layers.append(t)
    ws = torch.empty(q38.lib.q38_gdn_workspace_size(layers[0]["h"], rows), dtype=torch.uint8, device="cuda")
    return {"layers": layers, "rows": rows, "bits": bits, "group": group, "ws": ws, "handles": hs}


def _gdn_run(s):
    st = _stream()
    for t in s["layers"]:
        q38.check(q38.lib.q38_gdn_verify(t["h"], _p(t["x"]), s["rows"], _p(t["origin"]), _p(t["ckpt"]), _p(t["out"]),
                                         _p(s["ws"]), s["ws"].numel(), st))
    return [(t["out"], t["ckpt"]) for t in s["layers"]]


def _gdn_layer_exact(t, rows, bits, group):
    kw, vw = GDN_HK * GDN_D, GDN_HV * GDN_D
    c = 2 * kw + vw
    w = [_dequant_affine(*p, bits, group) for p in t["proj"]]
    x = t["x"].double()
    qkv, z, b, a = (x @ w[p].T for p in range(4))
    conv0 = t["origin"][:3 * c].double().reshape(3, c)
    state = t["origin"][3 * c:].double().reshape(GDN_HV, GDN_D, GDN_D)
    cin = torch.cat([conv0, qkv])
    taps = t["conv"].double()
    act = sum(taps[:, j] * cin[j:j + rows] for j in range(4))
    act = act * torch.sigmoid(act)
    rep = GDN_HV // GDN_HK
    q = (_rms(act[:, :kw].reshape(rows, GDN_HK, GDN_D)) / GDN_D).repeat_interleave(rep, 1)
    k = (_rms(act[:, kw:2 * kw].reshape(rows, GDN_HK, GDN_D)) / math.sqrt(GDN_D)).repeat_interleave(rep, 1)
    v = act[:, 2 * kw:].reshape(rows, GDN_HV, GDN_D)
    beta = torch.sigmoid(b)
    decay = torch.exp(-torch.exp(t["a_log"].double()) * torch.nn.functional.softplus(a + t["dt"].double()))
    ys, ck = [], torch.empty((rows, t["origin"].numel()), dtype=torch.float64, device=x.device)
    for r in range(rows):
        state = state * decay[r][:, None, None]
        delta = (v[r] - (state * k[r][:, None, :]).sum(-1)) * beta[r][:, None]
        state = state + delta[:, :, None] * k[r][:, None, :]
        ys.append((state * q[r][:, None, :]).sum(-1))
        ck[r, :3 * c] = cin[r + 1:r + 4].reshape(-1)
        ck[r, 3 * c:] = state.reshape(-1)
    y = _rms(torch.stack(ys)) * t["norm"].double() * torch.sigmoid(z.reshape(rows, GDN_HV, GDN_D))
    return y.reshape(rows, vw) @ w[4].T, ck


def _gdn_exact(s):
    return [_gdn_layer_exact(t, s["rows"], s["bits"], s["group"]) for t in s["layers"]]


# ------------------------------------------------------------------ attn: full-attention layers
def _attn_prepare(case, g):
    hs = _Handles()
    rows, bits, n, tokens, group = (case[k] for k in ("rows", "bits", "layers", "tokens", "group"))
    qw, kw = ATT_HQ * ATT_D, ATT_HKV * ATT_D
    cap = -(-(tokens + rows) // 256) * 256
    layers = []
    for _ in range(n):
        t = {"proj": [_affine(g, o, i, bits, group) for o, i in ((2 * qw, H), (kw, H), (kw, H), (H, qw))],
             "qn": _uniform(g, (ATT_D,), 0.5, 1.5, torch.bfloat16),
             "kn": _uniform(g, (ATT_D,), 0.5, 1.5, torch.bfloat16)}
        d = q38.AttnDesc(H, ATT_HQ, ATT_HKV, ATT_D, ATT_ROT, bits, group, 0, 0, EPS, ATT_THETA)
        w = q38.AttnWeights()
        for p in range(4):
            w.weight[p], w.scales[p], w.biases[p] = (_p(v) for v in t["proj"][p])
        w.q_norm, w.k_norm = _p(t["qn"]), _p(t["kn"])
        h = q38.P()
        q38.check(q38.lib.q38_attn_create(ctx().h, C.byref(d), C.byref(w), C.byref(h)))
        t["h"] = hs.add(h, q38.lib.q38_attn_destroy)
        cache = _normal(g, (2, ATT_HKV, cap, ATT_D), 1.0)
        t["cache"] = cache
        t["rows"] = (cache[0, :, tokens:tokens + rows], cache[1, :, tokens:tokens + rows])
        t["x"] = _normal(g, (rows, H), 1.0)
        t["out"] = torch.empty_like(t["x"])
        layers.append(t)
    ws = torch.empty(q38.lib.q38_attn_workspace_size(layers[0]["h"], rows, tokens + rows), dtype=torch.uint8,
                     device="cuda")
    return {"layers": layers, "rows": rows, "tokens": tokens, "cap": cap, "bits": bits, "group": group, "ws": ws,
            "handles": hs}


def _attn_run(s):
    st = _stream()
    for t in s["layers"]:
        q38.check(q38.lib.q38_attn_verify(t["h"], _p(t["x"]), s["rows"], _p(t["cache"]), s["cap"], s["tokens"],
                                          s["tokens"], _p(t["out"]), _p(s["ws"]), s["ws"].numel(), st))
    # the updated cache whole, and the appended rows by themselves
    return [(t["out"], t["cache"], *t["rows"]) for t in s["layers"]]


def _rope(v, pos):
    half = ATT_ROT // 2
    ang = pos[:, None, None].double() * ATT_THETA ** (-2.0 * torch.arange(half, device=v.device).double() / ATT_ROT)
    a, b = v[..., :half], v[..., half:ATT_ROT]
    return torch.cat([a * torch.cos(ang) - b * torch.sin(ang), a * torch.sin(ang) + b * torch.cos(ang),
                      v[..., ATT_ROT:]], -1)


def _attn_layer_exact(t, s):
    rows, tokens = s["rows"], s["tokens"]
    w = [_dequant_affine(*p, s["bits"], s["group"]) for p in t["proj"]]
    x = t["x"].double()
    qg = (x @ w[0].T).reshape(rows, ATT_HQ, 2 * ATT_D)
    pos = torch.arange(rows, device=x.device) + tokens
    q = _rope(_rms(qg[..., :ATT_D]) * t["qn"].double(), pos)
    k = _rope(_rms((x @ w[1].T).reshape(rows, ATT_HKV, ATT_D)) * t["kn"].double(), pos).transpose(0, 1)
    v = (x @ w[2].T).reshape(rows, ATT_HKV, ATT_D).transpose(0, 1)
    cache = t["cache"].double().clone()
    cache[0, :, tokens:tokens + rows], cache[1, :, tokens:tokens + rows] = k, v
    out = torch.empty((rows, ATT_HQ, ATT_D), dtype=torch.float64, device=x.device)
    seen = torch.arange(tokens + rows, device=x.device)[None, :] <= pos[:, None]
    for h in range(ATT_HQ):
        keys, values = (cache[j, h // (ATT_HQ // ATT_HKV), :tokens + rows].contiguous() for j in (0, 1))
        sc = q[:, h].contiguous() @ keys.T / math.sqrt(ATT_D)
        out[:, h] = torch.softmax(sc.masked_fill(~seen, -math.inf), 1) @ values
    gated = (out * torch.sigmoid(qg[..., ATT_D:])).reshape(rows, ATT_HQ * ATT_D)
    return gated @ w[3].T, cache, k, v


def _attn_exact(s):
    return [_attn_layer_exact(t, s) for t in s["layers"]]


# ------------------------------------------------------------------ the interface
_KINDS = {
    "chain": (_chain_prepare, _chain_run, _chain_exact),
    "hc": (_hc_prepare, _hc_run, _hc_exact),
    "moe": (_moe_prepare, _moe_run, _moe_exact_case),
    "head": (_head_prepare, _head_run, _head_exact),
    "draft": (_draft_prepare, _draft_run, _draft_exact),
    "gdn": (_gdn_prepare, _gdn_run, _gdn_exact),
    "attn": (_attn_prepare, _attn_run, _attn_exact),
}


def prepare(case, seed):
    s = _KINDS[case["kind"]][0](case, _gen(seed))
    s["run"] = _KINDS[case["kind"]][1]
    torch.cuda.synchronize()
    return s


def run(state):
    return state["run"](state)


def exact(case, seed):
    s = prepare(case, seed)
    return _KINDS[case["kind"]][2](s)


def _affine_bytes(out, n_in, bits, group=GROUP):
    return out * (n_in * bits // 8 + n_in // group * 4)


def _moe_work(fmt, rows):
    """Bytes and flops of one layer: the weights of the experts that rows x K uniform routes
    touch, the codebooks, the router, the layer's input and output rows."""
    unique = E * (1.0 - (1.0 - K / E) ** rows)
    rowscale = (2 * I + H) * 2
    d8 = (2 * I * q38.words_per_row(H, 8, 14) + H * q38.words_per_row(I, 8, 14)) * 4
    d4 = (2 * I * q38.words_per_row(H, 4, 8) + H * q38.words_per_row(I, 4, 8)) * 4
    if fmt == "mixed":
        b = unique * ((d4 + d8) / 2 + rowscale) + d4 + rowscale + 3 * (256 * 4 * 2 + 16384 * 8)
    elif fmt == "ckpt":
        b = unique * (d8 + (2 * I * H + H * I) // GROUP * 2) + 3 * 16384 * 8 * 2
        b += 2 * _affine_bytes(I, H, SHARED_BITS) + _affine_bytes(H, I, SHARED_BITS)
    else:
        b = (unique + 1) * (d8 + rowscale) + 3 * 16384 * 8 * (1 if fmt == "u8" else 2)
    return b + E * H * 2 + H * 2 + 2 * rows * H * 2, rows * (2 * E * H + (K + 1) * 6 * H * I)


def work(case):
    kind, rows = case["kind"], case["rows"]
    if kind in ("chain", "hc"):
        b, f = _moe_work(case.get("format", "row"), rows)
        if kind == "hc":
            b += (RANK + HC) * HC * H * case["bits"] // 8 + HC * H * RANK * case["bits"] // 8 + HC * H * 2
            b += (RANK + HC + RANK) * HC * H // GROUP * 4 + 2 * rows * (HC - 1) * H * 2
            f += rows * 2 * HC * H * (2 * RANK + HC)
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    if kind == "moe":
        b, f = _moe_work(case["format"], rows)
        return {"bytes": b, "flops": f}
    if kind == "head":
        return {"bytes": case["vocab"] * (H + 2) + rows * H * 2, "flops": 2 * rows * case["vocab"] * H}
    if kind == "draft":
        b, f = _moe_work("row", rows)
        v = case["vocab"]
        b += 2 * H * (H + 2) + v * (H // 2 + H // 64 * 2) + rows * v * 4
        return {"bytes": b, "flops": f + 2 * rows * H * (2 * H + v)}
    if kind == "gdn":
        kw, vw = GDN_HK * GDN_D, GDN_HV * GDN_D
        c, state = 2 * kw + vw, GDN_HV * GDN_D * GDN_D
        b = sum(_affine_bytes(o, i, case["bits"], case["group"]) for o, i in ((c + vw + 2 * GDN_HV, H), (H, vw)))
        b += (1 + rows) * (3 * c + state) * 2 + 2 * rows * H * 2
        f = 2 * rows * (H * (c + vw + 2 * GDN_HV) + vw * H) + rows * 7 * state
        return {"bytes": case["layers"] * b, "flops": case["layers"] * f}
    qw, kw, seen = ATT_HQ * ATT_D, ATT_HKV * ATT_D, case["tokens"] + rows
    b = sum(_affine_bytes(o, i, case["bits"], case["group"]) for o, i in ((2 * qw + 2 * kw, H), (H, qw)))
    b += 2 * seen * kw * 2 + 2 * rows * kw * 2 + 2 * rows * H * 2
    f = 2 * rows * (H * (2 * qw + 2 * kw) + qw * H) + 4 * rows * seen * qw
    return {"bytes": case["layers"] * b, "flops": case["layers"] * f}


def tolerance(case):
    """Twice to four times the distance of the outputs from 64-bit arithmetic (measured: MoE and draft
    step 0.005, GatedDeltaNet 0.009 over its chain of bf16 states, attention 0.0065, head logits
    3e-8): bf16 results of bf16 intermediates, whose roundings another order of the sums moves."""
    if case["kind"] == "head":
        return {"rel": 1e-6, "max": 1e-5}
    return {"rel": {"chain": 1e-2, "hc": 1e-2, "moe": 1.5e-2, "draft": 1.5e-2, "gdn": 2e-2, "attn": 2e-2}[case["kind"]],
            "max": 0.25}
