"""The work that engines have this library do, as cases that can be timed and compared.

A case is one pass of a model's block-quantized linear operators through the public entry points of
gemm_amd.qlinear, in the order in which an engine calls them; what stands between them (attention, norms,
sampling) is the engine's own and not run, so operator inputs that such code would produce are buffers of the
right shape. Kinds:

  decode    one token through all layers and the output projection: embedding lookup, Q/K/V in one launch,
            attention output + residual, gate+up+SiLU, down + residual, output projection with the greedy pick
  chunk     the seven products of a layer on `tokens` bf16 activation rows: a few rows are a batch of decoding
            sequences or a speculative verify, more are a piece of a prompt
  exact     the same seven products on fp32 activations with no rounding to 16 bits
  moe       routing and the expert FFN of a mixture-of-experts model for `tokens` tokens
  host      one token through the host-pointer calls, the weights registered: how a C engine whose activations
            live in host memory calls the library
  unpack    tensors decoded once at load time, to bf16 (weights that a prefill uses most) or fp32

Weights are random blocks in the formats' own layout, with scale fields that give weights of about the size
that a trained model has; activations are N(0, 1).
"""
import ctypes

import torch

from gemm_amd import qlinear

# format -> ggml type id, elements and bytes of a block, fp16 fields as (offset, least, largest)
FORMATS = {
    "q4_0": (2, 32, 18, ((0, 2e-3, 8e-3),)),
    "q8_0": (8, 32, 34, ((0, 2e-4, 5e-4),)),
    "q2_K": (10, 256, 84, ((80, 2e-3, 4e-3), (82, 3e-3, 6e-3))),
    "q3_K": (11, 256, 110, ((108, 3e-4, 8e-4),)),
    "q4_K": (12, 256, 144, ((0, 1e-4, 3e-4), (2, 7.5e-4, 2.2e-3))),
    "q5_K": (13, 256, 176, ((0, 7e-5, 1.5e-4), (2, 1.1e-3, 2.3e-3))),
    "q6_K": (14, 256, 210, ((208, 6.5e-5, 1.5e-4),)),
    "iq2_xxs": (16, 256, 66, ((0, 3e-4, 8e-4),)),
    "iq4_nl": (20, 32, 18, ((0, 2e-4, 6e-4),)),
    "iq3_s": (21, 256, 110, ((0, 1e-4, 4e-4),)),
    "iq4_xs": (23, 256, 136, ((0, 6.5e-5, 1.3e-4),)),
}
# formats whose few-token products leave the codes unrounded (up to 24 rows of activations)
UNROUNDED_FEW = ("q4_K", "q5_K", "q6_K", "q3_K", "q2_K", "q8_0")


def listed():
    return [
        # the usual 4-bit file of an 8B model, one user: V and down projections of half the layers in Q6_K
        {"name": "decode_q4_K_mix", "kind": "decode", "hidden": 4096, "ffn": 14336, "heads": 4096, "kv": 1024, "vocab": 128256,
         "layers": 32, "fmt": "q4_K", "fmt_down": "q4_K", "fmt_more": "q6_K", "fmt_head": "q6_K"},
        # a small 8-bit model (drafting, on-device sizes): the smallest launches, a vocabulary with added tokens
        {"name": "decode_small_q8_0", "kind": "decode", "hidden": 2048, "ffn": 5632, "heads": 2048, "kv": 256, "vocab": 32003,
         "layers": 22, "fmt": "q8_0", "fmt_down": "q8_0", "fmt_more": "q8_0", "fmt_head": "q8_0"},
        # a low-bit i-quant file: 2-bit grid codes, 3-bit in the down projections, a 5-bit output projection
        {"name": "decode_low_bit", "kind": "decode", "hidden": 4096, "ffn": 14336, "heads": 4096, "kv": 1024, "vocab": 151936,
         "layers": 16, "fmt": "iq2_xxs", "fmt_down": "iq3_s", "fmt_more": "iq3_s", "fmt_head": "q5_K"},
        # sixteen sequences decoding together on a 4-bit file
        {"name": "batch_16_q4_K", "kind": "chunk", "tokens": 16, "hidden": 4096, "ffn": 14336, "heads": 4096, "kv": 1024,
         "layers": 6, "fmt": "q4_K", "fmt_down": "q6_K"},
        # a full prefill chunk
        {"name": "prefill_512_q4_K", "kind": "chunk", "tokens": 512, "hidden": 4096, "ffn": 14336, "heads": 4096, "kv": 1024,
         "layers": 4, "fmt": "q4_K", "fmt_down": "q4_K"},
        # a short prompt of no round length on a narrower 6-bit model
        {"name": "prefill_77_q6_K", "kind": "chunk", "tokens": 77, "hidden": 2560, "ffn": 6912, "heads": 2560, "kv": 640,
         "layers": 8, "fmt": "q6_K", "fmt_down": "q6_K"},
        # a long prompt, the largest products
        {"name": "prefill_2048_q5_K", "kind": "chunk", "tokens": 2048, "hidden": 4096, "ffn": 14336, "heads": 4096, "kv": 1024,
         "layers": 2, "fmt": "q5_K", "fmt_down": "q5_K"},
        # a prompt whose products stay in fp32, as the reference's CPU path computes them
        {"name": "exact_320_q4_K", "kind": "exact", "tokens": 320, "hidden": 4096, "ffn": 14336, "heads": 4096, "kv": 1024,
         "layers": 1, "fmt": "q4_K", "fmt_down": "q6_K"},
        # mixture of experts, one user
        {"name": "moe_1_q4_K", "kind": "moe", "tokens": 1, "experts": 128, "top": 8, "hidden": 2048, "ffn": 768, "layers": 12,
         "fmt": "q4_K", "fmt_down": "q4_K"},
        # mixture of experts, a batch
        {"name": "moe_64_q4_K", "kind": "moe", "tokens": 64, "experts": 128, "top": 8, "hidden": 2048, "ffn": 768, "layers": 3,
         "fmt": "q4_K", "fmt_down": "q4_K"},
        # the C engine's own calls, activations in host memory
        {"name": "host_q4_K", "kind": "host", "hidden": 4096, "ffn": 14336, "heads": 4096, "kv": 1024, "layers": 2, "fmt": "q4_K",
         "fmt_down": "q4_K"},
        # load time: the tensors of a layer to bf16
        {"name": "unpack_q6_K_bf16", "kind": "unpack", "rows": 14336, "cols": 4096, "tensors": 3, "fmt": "q6_K", "to": "bf16"},
    ]


def _spread(rng, lo, hi, step=1):
    """A multiple of `step` between lo and hi, even over the logarithm."""
    return max(lo, min(hi, int(round(lo * (hi / lo) ** rng.random() / step)) * step))


def _fmt(rng):
    """The formats by how often files use them: 4-bit K-quants most, then 6- and 8-bit, then the others."""
    return rng.choice(["q4_K"] * 4 + ["q6_K"] * 2 + ["q8_0"] * 2 + ["q5_K", "q4_0", "q3_K", "q2_K", "iq4_nl", "iq4_xs", "iq3_s", "iq2_xxs"])


def _widths(rng, largest):
    hidden = _spread(rng, 1024, largest, 256)
    return {"hidden": hidden, "ffn": min(14336, int(hidden * rng.uniform(2, 4)) // 256 * 256), "heads": hidden,
            "kv": max(128, hidden // rng.choice([1, 4, 8]) // 64 * 64)}


def draw(rng):
    """Another case of the same kinds: widths of models of 0.3 to 8 billion weights, odd token counts, any of the formats."""
    kind = rng.choice(["decode", "decode", "decode", "chunk", "chunk", "chunk", "chunk", "exact", "moe", "moe", "host", "unpack"])
    fmt = _fmt(rng)
    down = rng.choice([fmt, fmt, "q6_K"])
    if kind == "decode":
        return dict(_widths(rng, 4096), kind=kind, vocab=_spread(rng, 32000, 151936), layers=rng.randint(4, 24), fmt=fmt, fmt_down=down,
                    fmt_more=rng.choice([fmt, "q6_K"]), fmt_head=rng.choice(["q6_K", "q8_0", fmt]))
    if kind == "chunk":
        tokens = _spread(rng, 2, 2048)
        return dict(_widths(rng, 4096), kind=kind, tokens=tokens, layers=rng.randint(4, 8) if tokens <= 256 else rng.randint(1, 2), fmt=fmt,
                    fmt_down=down)
    if kind == "exact":
        return dict(_widths(rng, 4096), kind=kind, tokens=_spread(rng, 8, 512), layers=1, fmt=fmt, fmt_down=down)
    if kind == "moe":
        return {"kind": kind, "tokens": _spread(rng, 1, 128), "experts": rng.choice([32, 64, 128]), "top": rng.choice([2, 4, 8]),
                "hidden": _spread(rng, 1024, 4096, 256), "ffn": _spread(rng, 512, 1536, 256), "layers": rng.randint(2, 4),
                "fmt": rng.choice(["q4_K", "q4_K", "q4_K", "q5_K", "q6_K", "q8_0"]), "fmt_down": rng.choice(["q4_K", "q6_K"])}
    if kind == "host":
        return dict(_widths(rng, 4096), kind=kind, layers=rng.randint(1, 3), fmt=fmt, fmt_down=down)
    return {"kind": kind, "rows": _spread(rng, 1024, 16384), "cols": _spread(rng, 1024, 8192, 256), "tensors": rng.randint(1, 3), "fmt": fmt,
            "to": rng.choice(["bf16", "f32"])}


class Buf:
    """A torch tensor as the binding takes device buffers."""

    def __init__(self, t):
        self.t, self.ptr, self.nbytes = t, t.data_ptr(), t.numel() * t.element_size()


def row_bytes(fmt, cols):
    _, elems, size, _ = FORMATS[fmt]
    return cols // elems * size


def _type(fmt):
    return FORMATS[fmt][0]


def _weights(g, fmt, rows, cols):
    _, elems, size, fields = FORMATS[fmt]
    n = rows * (cols // elems)
    words = torch.randint(-(1 << 63), (1 << 63) - 1, ((n * size + 7) // 8,), dtype=torch.int64, device="cuda", generator=g)
    flat = words.view(torch.uint8)[: n * size]
    blocks = flat.view(n, size)
    for off, lo, hi in fields:
        d = torch.empty(n, 1, dtype=torch.float32, device="cuda").uniform_(lo, hi, generator=g)
        blocks[:, off:off + 2] = d.to(torch.float16).view(torch.uint8)
    if fmt == "q6_K":  # sub-block scales of the size that the format's own quantizer writes most
        sc = blocks[:, 192:208].view(torch.int8)
        sc.bitwise_and_(63).sub_(32)
    return Buf(flat)


def _normal(g, *shape, dtype=torch.float32):
    return torch.randn(*shape, device="cuda", generator=g).to(dtype)


def _out(*shape):
    return torch.empty(*shape, device="cuda", dtype=torch.float32)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _more_bits(i, layers):
    """Layers whose V and down projections the usual K-quant mixes store in more bits: the first and last eighth, every third between."""
    return i < layers // 8 or i >= 7 * layers // 8 or (i - layers // 8) % 3 == 2


def _layer_formats(c, i):
    """The formats of one layer's Q, K, V, attention output, gate, up and down."""
    more = c["kind"] == "decode" and _more_bits(i, c["layers"])
    return [c["fmt"], c["fmt"], c["fmt_more"] if more else c["fmt"], c["fmt"], c["fmt"], c["fmt"], c["fmt_more"] if more else c["fmt_down"]]


def _shapes(c):
    h, f, n, k = c["hidden"], c["ffn"], c["heads"], c["kv"]
    return [(n, h), (k, h), (k, h), (h, n), (f, h), (f, h), (h, f)]


def _layers(g, c):
    return [[(fmt, _weights(g, fmt, r, k)) for fmt, (r, k) in zip(_layer_formats(c, i), _shapes(c))] for i in range(c["layers"])]


# ------------------------------------------------------------------ decode

def _prepare_decode(c, g):
    L, h = c["layers"], c["hidden"]
    s = {"layers": _layers(g, c), "table": _weights(g, c["fmt"], c["vocab"], h), "head": _weights(g, c["fmt_head"], c["vocab"], h)}
    s["token"] = Buf(torch.randint(0, c["vocab"], (1,), dtype=torch.int32, device="cuda", generator=g))
    s["x"], s["att"], s["xf"], s["xo"] = (_normal(g, L, h), _normal(g, L, c["heads"]), _normal(g, L, h), _normal(g, h))
    s["q"], s["k"], s["v"], s["act"] = _out(L, c["heads"]), _out(L, c["kv"]), _out(L, c["kv"]), _out(L, c["ffn"])
    s["res"], s["logits"] = _out(1, h), _out(c["vocab"])
    s["pick"] = torch.zeros(qlinear.ARGMAX_RESULT_BYTES // 4, dtype=torch.int32, device="cuda")
    s["io"] = [[Buf(s[n][i]) for n in ("x", "att", "xf", "q", "k", "v", "act")] for i in range(L)]
    s["ends"] = [Buf(s[n]) for n in ("res", "xo", "logits", "pick")]
    return s


def _run_decode(c, s):
    h, f, nq, kv = c["hidden"], c["ffn"], c["heads"], c["kv"]
    res, xo, logits, pick = s["ends"]
    qlinear.embed_rows_dev(_type(c["fmt"]), s["table"], c["vocab"], s["token"], 1, res, h)
    for W, (x, att, xf, q, k, v, act) in zip(s["layers"], s["io"]):
        (tq, Wq), (_, Wk), (tv, Wv), (to, Wo), (tg, Wg), (_, Wu), (td, Wd) = W
        if tv == tq:
            qlinear.gemv_multi_dev(_type(tq), [Wq, Wk, Wv], [q, k, v], [nq, kv, kv], x, h)
        else:
            qlinear.gemv_multi_dev(_type(tq), [Wq, Wk], [q, k], [nq, kv], x, h)
            qlinear.gemv_dev(_type(tv), Wv, x, v, kv, h)
        qlinear.gemv_add_dev(_type(to), Wo, att, res, h, nq)
        qlinear.gemv_silu_mul_dev(_type(tg), Wg, Wu, xf, act, f, h)
        qlinear.gemv_add_dev(_type(td), Wd, act, res, h, f)
    qlinear.gemv_argmax_dev(_type(c["fmt_head"]), s["head"], xo, logits, pick, c["vocab"], h)
    return {"q": s["q"], "k": s["k"], "v": s["v"], "act": s["act"], "res": s["res"], "logits": s["logits"], "token": s["pick"][:1]}


# ------------------------------------------------------------------ chunk, exact

def _prepare_chunk(c, g):
    L, t = c["layers"], c["tokens"]
    kind = torch.float32 if c["kind"] == "exact" else torch.bfloat16
    s = {"layers": _layers(g, c), "in": [_normal(g, L, t, n, dtype=kind) for n in (c["hidden"], c["heads"], c["hidden"], c["ffn"])]}
    s["out"] = [_out(L, t, r) for r, _ in _shapes(c)]
    size = qlinear.gemm_f32_any_workspace_bytes if c["kind"] == "exact" else qlinear.gemm_bf16_any_workspace_bytes
    s["ws"] = Buf(torch.empty(max(size(r, k) for r, k in _shapes(c)), dtype=torch.uint8, device="cuda"))
    s["io"] = [([Buf(a[i]) for a in s["in"]], [Buf(a[i]) for a in s["out"]]) for i in range(L)]
    return s


def _run_chunk(c, s):
    t, h, f, nq, kv = c["tokens"], c["hidden"], c["ffn"], c["heads"], c["kv"]
    ws = s["ws"]
    for W, ((x, att, xf, act), (q, k, v, o, gate, up, down)) in zip(s["layers"], s["io"]):
        (tq, Wq), (_, Wk), (_, Wv), (to, Wo), (tg, Wg), (_, Wu), (td, Wd) = W
        qlinear.gemm_bf16_multi_dev(_type(tq), [Wq, Wk, Wv], x, [q, k, v], [nq, kv, kv], h, t, h, [nq, kv, kv], ws)
        qlinear.gemm_bf16_any_dev(_type(to), Wo, att, o, h, nq, t, nq, h, ws)
        qlinear.gemm_bf16_multi_dev(_type(tg), [Wg, Wu], xf, [gate, up], [f, f], h, t, h, [f, f], ws)
        qlinear.gemm_bf16_any_dev(_type(td), Wd, act, down, h, f, t, f, h, ws)
    return s["out"]


def _run_exact(c, s):
    t, ws = c["tokens"], s["ws"]
    for W, (ins, outs) in zip(s["layers"], s["io"]):
        for (fmt, w), y, x, (r, k) in zip(W, outs, (ins[0], ins[0], ins[0], ins[1], ins[2], ins[2], ins[3]), _shapes(c)):
            qlinear.gemm_f32_any_dev(_type(fmt), w, x, y, r, k, t, k, r, ws)
    return s["out"]


# ------------------------------------------------------------------ moe

def _prepare_moe(c, g):
    L, t, e, h, f = c["layers"], c["tokens"], c["experts"], c["hidden"], c["ffn"]
    s = {"experts": [[_weights(g, fmt, e * r, k) for fmt, r, k in ((c["fmt"], f, h), (c["fmt"], f, h), (c["fmt_down"], h, f))] for _ in range(L)]}
    s["logits"] = torch.rand(L, t, e, device="cuda", generator=g)
    s["x"] = _normal(g, L, t, h, dtype=torch.bfloat16)
    s["idx"] = torch.zeros(L, t, c["top"], dtype=torch.int32, device="cuda")
    s["w"], s["out"] = _out(L, t, c["top"]), _out(L, t, h)
    s["ws"] = Buf(torch.empty(qlinear.moe_workspace_bytes(t, c["top"], h, f, e), dtype=torch.uint8, device="cuda"))
    s["io"] = [[Buf(s[n][i]) for n in ("logits", "x", "idx", "w", "out")] for i in range(L)]
    return s


def _run_moe(c, s):
    t, e, top, h, f = c["tokens"], c["experts"], c["top"], c["hidden"], c["ffn"]
    types = (_type(c["fmt"]), _type(c["fmt"]), _type(c["fmt_down"]))
    for (gate, up, down), (logits, x, idx, w, out) in zip(s["experts"], s["io"]):
        qlinear.moe_route_dev(logits, t, e, top, idx, w)
        qlinear.moe_ffn_types_dev(types, gate, up, down, x, idx, w, out, t, top, h, f, e, s["ws"])
    return {"experts": s["idx"], "weights": s["w"], "out": s["out"]}


# ------------------------------------------------------------------ host

class Registered:
    """Weights in host memory with their device copy, released with the object."""

    def __init__(self, layers):
        self.layers = [[(fmt, w.t.cpu().numpy()) for fmt, w in W] for W in layers]
        for W in self.layers:
            for _, w in W:
                qlinear.check(qlinear.load().qlin_weight_register(w.ctypes.data, w.nbytes))

    def __del__(self):
        for W in self.layers:
            for _, w in W:
                qlinear.load().qlin_weight_unregister(w.ctypes.data)


def _prepare_host(c, g):
    L = c["layers"]
    s = {"weights": Registered(_layers(g, c))}
    s["in"] = [_normal(g, L, n).cpu().numpy() for n in (c["hidden"], c["heads"], c["hidden"])]
    s["res"] = _normal(g, c["hidden"]).cpu().numpy()
    s["out"] = [torch.empty(L, r, dtype=torch.float32).numpy() for r in (c["heads"], c["kv"], c["kv"], c["ffn"], c["hidden"])]
    return s


def _p(a):
    return ctypes.c_void_p(a.ctypes.data)


def _run_host(c, s):
    lib, h, f, nq, kv = qlinear.load(), c["hidden"], c["ffn"], c["heads"], c["kv"]
    q, k, v, act, res = s["out"]
    for i, W in enumerate(s["weights"].layers):
        (tq, Wq), (tk, Wk), (tv, Wv), (to, Wo), (tg, Wg), (tu, Wu), (td, Wd) = W
        x, att, xf = (a[i] for a in s["in"])
        res[i] = res[i - 1] if i else s["res"]
        qlinear.check(lib.qlin_matvec_qkv(_p(q[i]), _p(Wq), _type(tq), nq, _p(k[i]), _p(Wk), _type(tk), _p(v[i]), _p(Wv), _type(tv), kv, h, _p(x)))
        qlinear.check(lib.qlin_matvec_add(_p(res[i]), _p(Wo), _type(to), nq, _p(att), h))
        qlinear.check(lib.qlin_matvec_silu_mul(_p(act[i]), _p(Wg), _type(tg), _p(Wu), _type(tu), h, _p(xf), f))
        qlinear.check(lib.qlin_matvec_add(_p(res[i]), _p(Wd), _type(td), f, _p(act[i]), h))
    return s["out"]


# ------------------------------------------------------------------ unpack

def _prepare_unpack(c, g):
    n = c["tensors"]
    out = torch.empty(n, c["rows"], c["cols"], device="cuda", dtype=torch.bfloat16 if c["to"] == "bf16" else torch.float32)
    return {"tensors": [_weights(g, c["fmt"], c["rows"], c["cols"]) for _ in range(n)], "out": out, "io": [Buf(o) for o in out]}


def _run_unpack(c, s):
    call = qlinear.dequant_bf16_dev if c["to"] == "bf16" else qlinear.dequant_dev
    for w, o in zip(s["tensors"], s["io"]):
        call(_type(c["fmt"]), w, o, c["rows"], c["cols"])
    return s["out"]


PREPARE = {"decode": _prepare_decode, "chunk": _prepare_chunk, "exact": _prepare_chunk, "moe": _prepare_moe, "host": _prepare_host,
           "unpack": _prepare_unpack}
RUN = {"decode": _run_decode, "chunk": _run_chunk, "exact": _run_exact, "moe": _run_moe, "host": _run_host, "unpack": _run_unpack}


def prepare(case, seed):
    torch.cuda.init()
    return {"case": case, "state": PREPARE[case["kind"]](case, _generator(seed))}


def run(state):
    return RUN[state["case"]["kind"]](state["case"], state["state"])


def work(case):
    c, kind = case, case["kind"]
    if kind == "unpack":
        n = c["tensors"] * c["rows"]
        return {"bytes": n * (row_bytes(c["fmt"], c["cols"]) + c["cols"] * (2 if c["to"] == "bf16" else 4)), "flops": n * c["cols"]}
    t = c.get("tokens", 1)
    if kind == "moe":
        used = c["experts"] * (1 - (1 - c["top"] / c["experts"]) ** t)  # experts that some token is routed to, on average
        one = 2 * c["ffn"] * row_bytes(c["fmt"], c["hidden"]) + c["hidden"] * row_bytes(c["fmt_down"], c["ffn"])
        return {"bytes": c["layers"] * (used * one + t * (6 * c["hidden"] + 4 * c["experts"] + 8 * c["top"])),
                "flops": c["layers"] * 6 * t * c["top"] * c["ffn"] * c["hidden"]}
    wide = 2 if kind == "chunk" else 4
    weights = sum(r * row_bytes(fmt, k) for i in range(c["layers"]) for fmt, (r, k) in zip(_layer_formats(c, i), _shapes(c)))
    acts = c["layers"] * t * (wide * (2 * c["hidden"] + c["heads"] + c["ffn"]) + 4 * sum(r for r, _ in _shapes(c)))
    flops = 2 * t * c["layers"] * sum(r * k for r, k in _shapes(c))
    if kind == "decode":
        weights += c["vocab"] * row_bytes(c["fmt_head"], c["hidden"]) + row_bytes(c["fmt"], c["hidden"])
        acts += 4 * (c["hidden"] + c["vocab"])
        flops += 2 * c["vocab"] * c["hidden"]
    return {"bytes": weights + acts, "flops": flops}


def tolerance(case):
    """About four times what the paths measure against float64 products of the decoded weights: the sums in fp32 in
    any order (matvecs 1.0e-7 to 5.2e-7, products with unrounded codes 1.1e-7 to 2.7e-7, fp32 products 2.1e-6 at the
    longest rows, the expert FFN 2.5e-6), or the weights rounded once to bf16 (1.65e-3) where the path may do so."""
    kind = case["kind"]
    if kind == "unpack":
        return "exact"
    if kind == "moe":  # two router logits can be equal to within the softmax's rounding
        return {"rel": 1e-5, "max": 2e-4, "differ": 1e-3}
    if kind == "exact":
        return {"rel": 8e-6, "max": 1e-4}
    if kind == "chunk" and not (case["tokens"] <= 4 or (case["tokens"] <= 24 and {case["fmt"], case["fmt_down"]} <= set(UNROUNDED_FEW))):
        return {"rel": 7e-3, "max": 0.04}
    return {"rel": 2e-6, "max": 4e-5}
