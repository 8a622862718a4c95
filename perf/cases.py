"""The calls that a program decoding a GGUF Llama on this library makes, as
measurable cases.

A chat program loads a quantised model once and then alternates two things: it
runs a prompt of a handful to a few hundred tokens (batched products, prefill
attention, the whole forward), and it decodes token by token (matrix-vector
products, decode attention over the cache, the whole forward with one token).
The kinds of case below are those calls, from the smallest matrix-vector
product to a 512-token prompt through a 32-layer model:

  matvec   holo_matmul: one matrix times one activation vector
  layer    the four fused products of a decode layer (norm + q/k/v, o + residual,
           norm + gate/up + SwiGLU, down + residual)
  rows     holo_matmul_rows: one matrix times the activation rows of a prompt
  attend   holo_attention_prefill: causal attention of `rows` new positions over
           a cache that already holds `pos0`
  forward  holo_llama_forward: `n` tokens at position `pos0` through a model

Device memory is torch's; the library works on the same device and on the
null stream, which is also torch's default stream.
"""
from __future__ import annotations

import ctypes
import math
import os
import sys

import torch

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, os.path.join(ROOT, "google-classic_amd"))
import holo_mi355x as holo  # noqa: E402

# A decoder's mixes of weight types: (q, k, o, gate, up), (v, down), head, embedding.
MIXES = {
    "q4_0": ("q4_0", "q4_0", "q8_0", "q8_0"),
    "q8_0": ("q8_0", "q8_0", "q8_0", "q8_0"),
    "q4_k_m": ("q4_k", "q6_k", "q6_k", "q4_k"),
}
LLAMA_7B = {"dim": 4096, "ffn": 11008, "heads": 32, "kv_heads": 32, "vocab": 32000}
EPS, ROPE_BASE = 1e-5, 10000.0


def listed():
    return [
        # the smallest call of a decode step: a grouped-query k or v projection
        {"name": "matvec_q4_k_1024x4096", "kind": "matvec", "type": "q4_k", "out": 1024, "in": 4096},
        # a square projection of a Q8_0 file
        {"name": "matvec_q8_0_4096x4096", "kind": "matvec", "type": "q8_0", "out": 4096, "in": 4096},
        # the output head of a Q4_K_M file: the largest matrix of a decode step
        {"name": "matvec_q6_k_32000x4096", "kind": "matvec", "type": "q6_k", "out": 32000, "in": 4096},
        # a decode layer of a 7B Q4_0 model as its four fused calls
        {"name": "layer_q4_0_7b", "kind": "layer", "type": "q4_0", "dim": 4096, "kv_dim": 4096, "ffn": 11008},
        # a short chat message: a gate or up projection of its tokens
        {"name": "rows_16_q4_0_11008x4096", "kind": "rows", "type": "q4_0", "rows": 16, "out": 11008, "in": 4096},
        # a paragraph: the down projection of an 8B Q4_K model
        {"name": "rows_100_q4_k_4096x14336", "kind": "rows", "type": "q4_k", "rows": 100, "out": 4096, "in": 14336},
        # a full prompt batch: a gate or up projection
        {"name": "rows_512_q4_0_11008x4096", "kind": "rows", "type": "q4_0", "rows": 512, "out": 11008, "in": 4096},
        # a decode step's attention with a long conversation in the cache
        {"name": "attend_1_at_2047", "kind": "attend", "rows": 1, "pos0": 2047, "heads": 32, "kv_heads": 32,
         "head_dim": 128},
        # a follow-up message's attention over the conversation before it, grouped-query heads
        {"name": "attend_192_at_1000", "kind": "attend", "rows": 192, "pos0": 1000, "heads": 32, "kv_heads": 8,
         "head_dim": 128},
        # one decode step of a 7B model after a 512-token prompt
        dict(LLAMA_7B, name="forward_1_at_512_7b_q4_0", kind="forward", mix="q4_0", n=1, pos0=512, layers=32),
        # a short question to a 7B model
        dict(LLAMA_7B, name="forward_23_7b_q4_k_m", kind="forward", mix="q4_k_m", n=23, pos0=0, layers=32),
        # a full prompt through a 7B model
        dict(LLAMA_7B, name="forward_512_7b_q4_0", kind="forward", mix="q4_0", n=512, pos0=0, layers=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("matvec", "layer", "rows", "rows", "attend", "forward"))
    if kind in ("matvec", "rows"):
        t = rng.choice(("q4_0", "q8_0", "q4_k", "q6_k"))
        case = {"kind": kind, "type": t}
        if kind == "rows":
            case["rows"] = _log(rng, 2, 1024)
        case["out"] = _log(rng, 256, 32000 if kind == "matvec" else 14336)
        # whole 256-weight blocks; the 32-weight types also in odd block counts
        unit = 256 if t in ("q4_k", "q6_k") or rng.random() < 0.7 else 32
        case["in"] = unit * max(1, _log(rng, 1024, 14336) // unit)
        if kind == "rows":
            most = 512 * 11008 * 4096 // (case["out"] * case["in"])
            case["rows"] = max(2, min(case["rows"], most))
        return case
    if kind == "layer":
        dim = 256 * _log(rng, 8, 32)
        return {"kind": kind, "type": rng.choice(("q4_0", "q4_k")), "dim": dim,
                "kv_dim": dim // rng.choice((1, 4, 8)), "ffn": 256 * int(dim * rng.uniform(2.5, 3.5) / 256)}
    heads = rng.choice((8, 16, 24, 32))
    kv_heads = heads // rng.choice((1, 2, 4))
    if kind == "attend":
        return {"kind": kind, "rows": max(1, _log(rng, 1, 600) - 1), "pos0": _log(rng, 1, 4000), "heads": heads,
                "kv_heads": kv_heads, "head_dim": rng.choice((64, 128, 128))}
    dim = heads * 128
    return {"kind": kind, "mix": rng.choice(sorted(MIXES)), "n": max(1, _log(rng, 1, 600) - 1),
            "pos0": rng.choice((0, _log(rng, 1, 1500))), "layers": rng.randint(1, 4), "dim": dim,
            "ffn": 256 * int(dim * rng.uniform(2.5, 3.5) / 256), "heads": heads, "kv_heads": kv_heads,
            "vocab": _log(rng, 1000, 32000)}


# ---- inputs ---------------------------------------------------------------------

def _blocks(qtype, out, in_dim, gen):
    """A random [out][in_dim] matrix of the type as its file bytes: uniform
    quants, |N(0,1)| block scales, weights of variance about 1/in_dim."""
    dev = gen.device
    if qtype == "f32":
        return torch.randn(out, in_dim, generator=gen, device=dev) / math.sqrt(in_dim)
    qk, bb = holo.BLOCK[holo.TYPE_NAMES[qtype]]
    nb = in_dim // qk
    raw = torch.randint(0, 256, (out, nb, bb), generator=gen, device=dev, dtype=torch.uint8)
    # standard deviation of a weight over its block scale
    spread = {"q4_0": 4.64, "q8_0": 73.3, "q4_k": 256.0, "q6_k": 1366.0}[qtype]
    d = torch.randn(out, nb, generator=gen, device=dev).abs() / (spread * math.sqrt(in_dim))

    def put(at, v):
        raw[:, :, at:at + 2] = v.half().view(torch.uint8).view(out, nb, 2)

    if qtype == "q8_0":
        raw[:, :, 2:] = torch.randint(-127, 128, (out, nb, 32), generator=gen, device=dev,
                                      dtype=torch.int8).view(torch.uint8)
    if qtype == "q4_k":
        put(2, 7.5 * d)  # minima that centre the block
    put(208 if qtype == "q6_k" else 0, d)
    return raw


def _buf(*shape):
    return torch.zeros(*shape, device="cuda", dtype=torch.float32)


def prepare(case, seed):
    holo.init()
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)

    s = {"case": case, "kind": case["kind"], "lib": holo.lib()}
    kind = case["kind"]
    if kind in ("matvec", "rows"):
        m = case.get("rows", 1)
        s["w"] = _blocks(case["type"], case["out"], case["in"], gen)
        s["x"], s["y"] = normal(m, case["in"]), _buf(m, case["out"])
        s["type"] = holo.TYPE_NAMES[case["type"]]
    elif kind == "layer":
        dim, kv, ffn, t = case["dim"], case["kv_dim"], case["ffn"], case["type"]
        shapes = {"wq": (dim, dim), "wk": (kv, dim), "wv": (kv, dim), "wo": (dim, dim), "w1": (ffn, dim),
                  "w3": (ffn, dim), "w2": (dim, ffn)}
        s["w"] = {n: _blocks(t, *shape, gen) for n, shape in shapes.items()}
        s["type"] = holo.TYPE_NAMES[t]
        s["x"], s["att"] = normal(dim), normal(dim)
        s["norms"] = [1 + 0.1 * normal(dim) for _ in range(2)]
        s["out"] = {"q": _buf(dim), "k": _buf(kv), "v": _buf(kv), "x1": _buf(dim), "h": _buf(ffn), "x2": _buf(dim)}
        s["xb"] = _buf(dim)
    elif kind == "attend":
        hd, kv_len = case["head_dim"], case["pos0"] + case["rows"]
        s["q"] = normal(case["rows"], case["heads"] * hd)
        s["k"], s["v"] = normal(kv_len, case["kv_heads"] * hd), normal(kv_len, case["kv_heads"] * hd)
        s["y"] = _buf(case["rows"], case["heads"] * hd)
    else:
        _prepare_model(s, case, gen, normal)
    return s


def _prepare_model(s, case, gen, normal):
    dim, ffn, vocab, n, pos0 = case["dim"], case["ffn"], case["vocab"], case["n"], case["pos0"]
    kv = dim // case["heads"] * case["kv_heads"]
    a, b, head, emb = MIXES[case["mix"]]
    shapes = (("wq", dim, dim, a), ("wk", kv, dim, a), ("wv", kv, dim, b), ("wo", dim, dim, a), ("w1", ffn, dim, a),
              ("w2", dim, ffn, b), ("w3", ffn, dim, a))
    layers = (holo.LlamaLayer * case["layers"])()
    s["layers"] = []
    for i in range(case["layers"]):
        keep = {"attn_norm": 1 + 0.1 * normal(dim), "ffn_norm": 1 + 0.1 * normal(dim)}
        for name, out, in_dim, t in shapes:
            keep[name] = _blocks(t, out, in_dim, gen)
            setattr(layers[i], name + "_type", holo.TYPE_NAMES[t])
        for name, v in keep.items():
            setattr(layers[i], name, v.data_ptr())
        s["layers"].append(keep)
    s["emb"], s["head"], s["out_norm"] = _blocks(emb, vocab, dim, gen), _blocks(head, vocab, dim, gen), 1 + 0.1 * normal(dim)
    max_seq = pos0 + n
    s["kc"], s["vc"] = normal(case["layers"], max_seq, kv), normal(case["layers"], max_seq, kv)
    s["tokens"] = torch.randint(0, vocab, (n,), generator=gen, device="cuda").tolist()
    s["tokens_c"] = (ctypes.c_int * n)(*s["tokens"])
    s["logits"] = _buf(vocab)
    s["layers_c"] = layers
    s["model"] = holo.LlamaModel(
        n_layers=case["layers"], dim=dim, n_heads=case["heads"], n_kv_heads=case["kv_heads"],
        head_dim=dim // case["heads"], ffn_dim=ffn, vocab=vocab, max_seq=max_seq, rms_eps=EPS, rope_base=ROPE_BASE,
        tok_emb=s["emb"].data_ptr(), emb_type=holo.TYPE_NAMES[emb], out_norm=s["out_norm"].data_ptr(),
        output=s["head"].data_ptr(), out_type=holo.TYPE_NAMES[head], key_cache=s["kc"].data_ptr(),
        value_cache=s["vc"].data_ptr(), layers=layers)


# ---- the calls --------------------------------------------------------------------

def run(s):
    case, lib, kind = s["case"], s["lib"], s["kind"]
    if kind == "matvec":
        lib.holo_matmul(s["y"].data_ptr(), s["w"].data_ptr(), s["x"].data_ptr(), case["out"], case["in"], s["type"])
        return s["y"]
    if kind == "rows":
        lib.holo_matmul_rows(s["y"].data_ptr(), s["w"].data_ptr(), s["x"].data_ptr(), case["rows"], case["out"],
                             case["in"], s["type"], 0)
        return s["y"]
    if kind == "layer":
        w, o, t = s["w"], s["out"], s["type"]
        dim, kv, ffn = case["dim"], case["kv_dim"], case["ffn"]
        xb = s["xb"].data_ptr()
        lib.holo_batched_qkv_norm(o["q"].data_ptr(), o["k"].data_ptr(), o["v"].data_ptr(), w["wq"].data_ptr(),
                                  w["wk"].data_ptr(), w["wv"].data_ptr(), s["x"].data_ptr(),
                                  s["norms"][0].data_ptr(), EPS, xb, dim, kv, dim, t)
        lib.holo_matmul_add(o["x1"].data_ptr(), w["wo"].data_ptr(), s["att"].data_ptr(), s["x"].data_ptr(), dim, dim,
                            t)
        lib.holo_batched_ffn_gate_up_norm(o["h"].data_ptr(), w["w1"].data_ptr(), w["w3"].data_ptr(),
                                          o["x1"].data_ptr(), s["norms"][1].data_ptr(), EPS, xb, ffn, dim, t)
        lib.holo_matmul_add(o["x2"].data_ptr(), w["w2"].data_ptr(), o["h"].data_ptr(), o["x1"].data_ptr(), dim, ffn,
                            t)
        return o
    if kind == "attend":
        lib.holo_attention_prefill(s["y"].data_ptr(), s["q"].data_ptr(), s["k"].data_ptr(), s["v"].data_ptr(),
                                   case["rows"], case["pos0"], case["head_dim"], case["heads"], case["kv_heads"])
        return s["y"]
    if lib.holo_llama_forward(ctypes.byref(s["model"]), s["tokens_c"], case["n"], case["pos0"], s["logits"].data_ptr(),
                              0):
        holo.check("holo_llama_forward")
    pos0 = case["pos0"]
    return {"logits": s["logits"], "k": s["kc"][:, pos0:], "v": s["vc"][:, pos0:]}


# ---- what a pass cannot do without --------------------------------------------------

def _matrix_bytes(qtype, out, in_dim):
    return out * holo.row_bytes(holo.TYPE_NAMES[qtype], in_dim)


def _attention(rows, pos0, heads, kv_heads, hd):
    pairs = rows * pos0 + rows * (rows + 1) // 2
    return 8 * (pos0 + rows) * kv_heads * hd + 8 * rows * heads * hd, 4 * pairs * heads * hd


def work(case):
    kind = case["kind"]
    if kind in ("matvec", "rows"):
        m, out, in_dim = case.get("rows", 1), case["out"], case["in"]
        return {"bytes": _matrix_bytes(case["type"], out, in_dim) + 4 * m * (out + in_dim),
                "flops": 2 * m * out * in_dim}
    if kind == "layer":
        dim, kv, ffn = case["dim"], case["kv_dim"], case["ffn"]
        weights = 2 * dim * dim + 2 * kv * dim + 3 * ffn * dim
        return {"bytes": _matrix_bytes(case["type"], weights // dim, dim) + 4 * (8 * dim + 2 * kv + ffn),
                "flops": 2 * weights}
    if kind == "attend":
        b, f = _attention(case["rows"], case["pos0"], case["heads"], case["kv_heads"], case["head_dim"])
        return {"bytes": b, "flops": f}
    dim, ffn, n, vocab, heads = case["dim"], case["ffn"], case["n"], case["vocab"], case["heads"]
    hd = dim // heads
    kv = hd * case["kv_heads"]
    a, b, head, emb = MIXES[case["mix"]]
    ab, af = _attention(n, case["pos0"], heads, case["kv_heads"], hd)
    layer = (_matrix_bytes(a, 2 * dim + kv + 2 * ffn, dim) + _matrix_bytes(b, kv, dim) + _matrix_bytes(b, dim, ffn) +
             ab - 8 * n * dim)
    return {"bytes": case["layers"] * layer + _matrix_bytes(head, vocab, dim) + _matrix_bytes(emb, n, dim) + 4 * vocab,
            "flops": case["layers"] * (2 * n * (2 * dim * dim + 2 * kv * dim + 3 * ffn * dim) + af) + 2 * vocab * dim}


def tolerance(case):
    # fp32 sums throughout; a forward carries its layers' rounding through the
    # rotary angles (fp32: up to 1e-4 rad at position 2000) and the layers above
    if case["kind"] == "forward":
        return {"rel": 5e-5, "max": 2e-3}
    return {"rel": 1e-5, "max": 2e-4}


# ---- the same in 64 bits, in plain torch ----------------------------------------------

def _weights64(qtype, raw):
    """float64 [out][in] of a matrix's file bytes."""
    if qtype == "f32":
        return raw.double()
    out, nb = raw.shape[:2]

    def f16(at):
        return raw[:, :, at:at + 2].contiguous().view(torch.float16).double()  # [out][nb][1]

    def signed(a, b):
        return raw[:, :, a:b].contiguous().view(torch.int8).double()

    if qtype == "q8_0":
        return (f16(0) * signed(2, 34)).view(out, -1)
    if qtype == "q4_0":
        q = raw[:, :, 2:]
        return (f16(0) * (torch.cat((q & 15, q >> 4), 2).double() - 8)).view(out, -1)
    if qtype == "q4_k":
        a, b, c = raw[:, :, 4:8].int(), raw[:, :, 8:12].int(), raw[:, :, 12:16].int()
        sc = torch.cat((a & 63, ((c & 15) << 2) | (a >> 6)), 2).double()
        mn = torch.cat((b & 63, ((c >> 4) << 2) | (b >> 6)), 2).double()
        q = raw[:, :, 16:].view(out, nb, 8, 16)
        q = torch.cat((q & 15, q >> 4), 3).double()
        return ((f16(0) * sc)[..., None] * q - (f16(2) * mn)[..., None]).view(out, -1)
    ql, qh = raw[:, :, :128].view(out, nb, 2, 2, 32), raw[:, :, 128:192].view(out, nb, 2, 32)
    q = torch.stack([((ql[:, :, :, j & 1] >> (4 * (j >> 1))) & 15) | (((qh >> (2 * j)) & 3) << 4) for j in range(4)], 3)
    sc = (f16(208) * signed(192, 208)).view(out, nb, 2, 4, 2, 1)
    return (sc * (q.view(out, nb, 2, 4, 2, 16).double() - 32)).view(out, -1)


def _times(x, qtype, raw):
    return x @ _weights64(qtype, raw).t()


def _norm64(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _silu64(x):
    return x * torch.sigmoid(x)


def _rope64(x, pos, heads):
    n, hd = x.shape[0], x.shape[1] // heads
    freq = ROPE_BASE ** (-2.0 * torch.arange(hd // 2, device=x.device, dtype=torch.float64) / hd)
    th = pos.double()[:, None, None] * freq
    x = x.view(n, heads, 2, hd // 2)
    a, b, c, s = x[:, :, 0], x[:, :, 1], th.cos(), th.sin()
    return torch.cat((a * c - b * s, a * s + b * c), 2).view(n, -1)


def _attend64(q, k, v, heads, kv_heads, pos0):
    rows, kv_len = q.shape[0], k.shape[0]
    hd = q.shape[1] // heads
    hidden = torch.arange(kv_len, device=q.device)[None, :] > pos0 + torch.arange(rows, device=q.device)[:, None]
    out = torch.empty(rows, heads, hd, device=q.device, dtype=torch.float64)
    for h in range(heads):
        g = h // (heads // kv_heads)
        kh, vh = (t[:, g * hd:(g + 1) * hd].contiguous() for t in (k, v))
        p = q[:, h * hd:(h + 1) * hd].contiguous() @ kh.t() / math.sqrt(hd)
        out[:, h] = p.masked_fill(hidden, -math.inf).softmax(1) @ vh
    return out.view(rows, -1)


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind in ("matvec", "rows"):
        return _times(s["x"].double(), case["type"], s["w"])
    if kind == "attend":
        return _attend64(s["q"].double(), s["k"].double(), s["v"].double(), case["heads"], case["kv_heads"],
                         case["pos0"])
    if kind == "layer":
        t, w = case["type"], s["w"]
        x = s["x"].double()[None]
        xb = _norm64(x, s["norms"][0])
        x1 = x + _times(s["att"].double()[None], t, w["wo"])
        xf = _norm64(x1, s["norms"][1])
        h = _silu64(_times(xf, t, w["w1"])) * _times(xf, t, w["w3"])
        out = {"q": _times(xb, t, w["wq"]), "k": _times(xb, t, w["wk"]), "v": _times(xb, t, w["wv"]), "x1": x1,
               "h": h, "x2": x1 + _times(h, t, w["w2"])}
        return {n: v[0] for n, v in out.items()}
    a, b, head, emb = MIXES[case["mix"]]
    heads, kv_heads, n, pos0 = case["heads"], case["kv_heads"], case["n"], case["pos0"]
    pos = pos0 + torch.arange(n, device="cuda")
    kc, vc = s["kc"], s["vc"]
    x = _weights64(emb, s["emb"][s["tokens"]])
    ks, vs = [], []
    for i, w in enumerate(s["layers"]):
        xb = _norm64(x, w["attn_norm"])
        q = _rope64(_times(xb, a, w["wq"]), pos, heads)
        ks.append(_rope64(_times(xb, a, w["wk"]), pos, kv_heads))
        vs.append(_times(xb, b, w["wv"]))
        k, v = (torch.cat((c[i, :pos0].double(), new[-1])) for c, new in ((kc, ks), (vc, vs)))
        x = x + _times(_attend64(q, k, v, heads, kv_heads, pos0), a, w["wo"])
        xb = _norm64(x, w["ffn_norm"])
        x = x + _times(_silu64(_times(xb, a, w["w1"])) * _times(xb, a, w["w3"]), b, w["w2"])
    logits = _times(_norm64(x[-1:], s["out_norm"]), head, s["head"])[0]
    return {"logits": logits, "k": torch.stack(ks), "v": torch.stack(vs)}
