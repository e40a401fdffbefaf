"""The work that the quantized linear path is timed and compared on.

Sizes are those of the repository's own configurations and tests: the
Llama-3-8B projections (hidden 4096, key/value 1024, intermediate 14336,
vocabulary 128256) in the Q4_K_M mix (Q6_K for v, down and the output head),
the Gemma4 token table [2560, 262144] in Q4_K, Q8_0 at 4096 x 4096, and ragged
shapes between them.  Weights are GGUF blocks with normally distributed codes,
activations are normal, optionally with a few large channels as the residual
stream of a trained model has them.

Kinds of work, each through the library's entry points:

  gather     okq_get_rows_q: the token embedding of a prompt
  dequant    okq_dequantize: a whole tensor expanded to f32
  norm_proj  okq_rmsnorm_linear_q_multi: q, k and v of one normalised hidden state
  linear     okq_linear_out_by_in_q and its bf16 form: one projection
  mlp        okq_mlp_gated_silu_q: the gated MLP of a layer
  decode     the quantized calls of several layers of one decode step, captured
             once into a HIP graph and replayed, as a serving loop keeps them
"""
import ctypes
import math

import torch

from ocelotl_amd import okq

Q4_0, Q8_0, Q4_K, Q5_K, Q6_K = 2, 8, 12, 13, 14
TYPES = {"Q4_0": Q4_0, "Q8_0": Q8_0, "Q4_K": Q4_K, "Q5_K": Q5_K, "Q6_K": Q6_K}
ELEMS = {Q4_0: 32, Q8_0: 32, Q4_K: 256, Q5_K: 256, Q6_K: 256}
BYTES = {Q4_0: 18, Q8_0: 34, Q4_K: 144, Q5_K: 176, Q6_K: 210}
EPS = 1e-5


def listed():
    return [
        # one attention block's q, k, v of one new token, launched by itself: the
        # smallest call of a chat turn; large channels as before a first norm
        dict(name="qkv_token", kind="norm_proj", type="Q4_K", rows=1, hidden=4096, n0=4096, n1=1024, n2=1024,
             outliers=True),
        # embedding of a 777-token prompt from the Gemma4-sized table
        dict(name="embed_prompt", kind="gather", type="Q4_K", ne0=2560, ne1=262144, n=777),
        # the output head for one token, a plain call
        dict(name="head_token", kind="linear", type="Q6_K", rows=1, k=4096, n=128256, x="f32", bias=False,
             outliers=False),
        # one token through eight layers (single stream generation)
        dict(name="decode_b1", kind="decode", rows=1, hidden=4096, kv=1024, inter=14336, layers=8),
        # eight and thirty-two sequences decoded together (a serving batch)
        dict(name="decode_b8", kind="decode", rows=8, hidden=4096, kv=1024, inter=14336, layers=8),
        dict(name="decode_b32", kind="decode", rows=32, hidden=4096, kv=1024, inter=14336, layers=8),
        # five drafted tokens verified at once, a Q5_K_M file's gate, with bias
        dict(name="verify_5", kind="linear", type="Q5_K", rows=5, k=4096, n=14336, x="f32", bias=True,
             outliers=False),
        # prompt of 333 tokens: norm and q, k, v of a Q8_0 file, f32 activations
        dict(name="qkv_prompt", kind="norm_proj", type="Q8_0", rows=333, hidden=4096, n0=4096, n1=1024, n2=1024,
             outliers=False),
        # prompt chunk of 512 tokens: a layer's MLP, f32 activations (the
        # reference's own element type)
        dict(name="mlp_prompt", kind="mlp", type="Q4_K", down="Q6_K", rows=512, hidden=4096, inter=14336),
        # 512 tokens through a square Q8_0 projection, bf16 activations
        dict(name="proj_bf16_512", kind="linear", type="Q8_0", rows=512, k=4096, n=4096, x="bf16", bias=False,
             outliers=False),
        # 2048 tokens through a gate projection, bf16 activations: a long prompt
        dict(name="gate_bf16_2048", kind="linear", type="Q4_K", rows=2048, k=4096, n=14336, x="bf16", bias=False,
             outliers=False),
        # a down projection's tensor expanded to f32 (the loader's dequantise policy)
        dict(name="expand_q6k", kind="dequant", type="Q6_K", ne0=14336, ne1=4096),
    ]


MOST = 2048 * 14336 * 4096  # multiply-adds of the largest listed projection


def draw(rng):
    def spread(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def blocks(lo, hi, e=256):
        return e * max(1, round(spread(lo, hi) / e))

    kind = rng.choice(["gather", "dequant", "norm_proj", "linear", "linear", "linear", "mlp", "mlp", "decode"])
    linear = ["Q8_0", "Q4_K", "Q5_K", "Q6_K"]
    if kind == "gather":
        return dict(kind=kind, type=rng.choice(sorted(TYPES)), ne0=blocks(256, 8192), ne1=spread(4000, 150000),
                    n=spread(1, 2048))
    if kind == "dequant":
        t = rng.choice(sorted(TYPES))
        return dict(kind=kind, type=t, ne0=blocks(256, 14336, ELEMS[TYPES[t]]), ne1=spread(64, 4096))
    if kind == "norm_proj":
        kv = 32 * spread(4, 64)
        return dict(kind=kind, type=rng.choice(linear), rows=spread(1, 1024), hidden=blocks(768, 5120),
                    n0=64 * spread(8, 80), n1=kv, n2=kv, outliers=rng.random() < 0.5)
    if kind == "mlp":
        t = rng.choice(["Q4_K", "Q4_K", "Q5_K", "Q8_0", "Q6_K"])
        h, i = blocks(768, 5120), blocks(1024, 14336)
        rows = min(rng.choice([spread(1, 32), spread(33, 700)]), (MOST if t == "Q4_K" else MOST // 2) // (4 * h * i))
        return dict(kind=kind, type=t, down=rng.choice(["Q6_K", t]), rows=rows, hidden=h, inter=i)
    if kind == "decode":
        return dict(kind=kind, rows=spread(1, 32), hidden=blocks(1024, 4096), kv=128 * spread(1, 8),
                    inter=blocks(2816, 14336), layers=rng.randint(2, 8))
    rows, n = spread(1, 2048), spread(256, 20000)
    t = rng.choice(linear)
    k = blocks(512, 14336) if t != "Q8_0" or rows > 8 else blocks(512, 14336, 32)
    x = rng.choice(["f32", "bf16"])
    n = max(256, min(n, (MOST if x == "bf16" else MOST // 3) // (rows * k)))
    return dict(kind=kind, type=t, rows=rows, k=k, n=n, x=x, bias=rng.random() < 0.5, outliers=rng.random() < 0.25)


# ---- inputs -----------------------------------------------------------------

def _normal(gen, *shape):
    return torch.randn(*shape, generator=gen, device="cuda", dtype=torch.float32)


def _codes(gen, shape, mean, sd, lo, hi):
    """Normally distributed integer codes in [lo, hi]."""
    return _normal(gen, *shape).mul_(sd).add_(mean).round_().clamp_(lo, hi).to(torch.int16)


def _ints(gen, shape, lo, hi):
    return torch.randint(lo, hi + 1, shape, generator=gen, device="cuda", dtype=torch.int16)


def _half_bytes(v):
    return v.to(torch.float16).contiguous().view(torch.uint8).view(v.shape[0], 2)


def _u8(v):
    return (v & 255).to(torch.uint8)


def _scale_bytes(ls, lm):
    """The 12 packed 6-bit scale and min bytes of Q4_K and Q5_K."""
    return torch.cat([_u8(ls[:, :4] | ((ls[:, 4:] >> 4) << 6)), _u8(lm[:, :4] | ((lm[:, 4:] >> 4) << 6)),
                      _u8((ls[:, 4:] & 15) | ((lm[:, 4:] & 15) << 4))], 1)


def _some_blocks(gen, t, nb):
    """nb GGUF blocks of type t [nb, bytes], weights of about N(0, 0.02)."""
    spread = _normal(gen, nb).mul_(0.1).add_(1.0).clamp_(0.6, 1.4)
    if t == Q8_0:
        q = _codes(gen, (nb, 32), 0, 40, -127, 127)
        return torch.cat([_half_bytes(spread * (0.02 / 40)), _u8(q)], 1)
    if t == Q4_0:
        q = _codes(gen, (nb, 32), 8, 2.7, 0, 15)
        return torch.cat([_half_bytes(spread * (0.02 / 2.7)), _u8(q[:, :16] | (q[:, 16:] << 4))], 1)
    if t == Q6_K:
        q = _codes(gen, (nb, 2, 4, 32), 32, 11, 0, 63)
        sign = _ints(gen, (nb, 16), 0, 1) * 2 - 1
        sc = _ints(gen, (nb, 16), 70, 127) * sign
        ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
        h = q >> 4
        qh = h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)
        return torch.cat([_u8(ql.reshape(nb, 128)), _u8(qh.reshape(nb, 64)), _u8(sc),
                          _half_bytes(spread * (0.02 / 1100))], 1)
    top = 15 if t == Q4_K else 31
    q = _codes(gen, (nb, 4, 2, 32), top / 2, top / 5.6, 0, top)
    ls, lm = _ints(gen, (nb, 8), 36, 63), _ints(gen, (nb, 8), 40, 60)
    d = 0.02 / (50 * top / 5.6)
    head = [_half_bytes(spread * d), _half_bytes(spread * (d * top / 2)), _scale_bytes(ls, lm)]
    if t == Q5_K:
        bit = torch.arange(4, device="cuda", dtype=torch.int16).view(1, 4, 1) * 2
        head.append(_u8((((q[:, :, 0] >> 4) << bit) | ((q[:, :, 1] >> 4) << (bit + 1))).sum(1)))
    return torch.cat(head + [_u8((q[:, :, 0] & 15) | ((q[:, :, 1] & 15) << 4)).reshape(nb, 128)], 1)


def _blocks(gen, t, k, n):
    """A GGUF tensor [k, n] as n rows of block bytes."""
    nb = k // ELEMS[t] * n
    out = torch.empty(nb, BYTES[t], dtype=torch.uint8, device="cuda")
    step = (1 << 26) // ELEMS[t]
    for i in range(0, nb, step):
        out[i:i + step] = _some_blocks(gen, t, min(step, nb - i))
    return out.view(n, -1)


def _activations(gen, rows, k, outliers):
    x = _normal(gen, rows, k)
    if outliers:
        x[:, torch.randint(0, k, (4,), generator=gen, device="cuda")] *= 50.0
    return x


def _inputs(case, seed):
    """Named tensors of a case, from the seed alone."""
    gen = torch.Generator(device="cuda")
    gen.manual_seed(int(seed))
    kind = case["kind"]
    t = TYPES[case["type"]] if "type" in case else None
    if kind == "gather":
        ids = torch.randint(0, case["ne1"], (case["n"],), generator=gen, device="cuda").cpu()
        return {"w": _blocks(gen, t, case["ne0"], case["ne1"]), "ids": ids}
    if kind == "dequant":
        return {"w": _blocks(gen, t, case["ne0"], case["ne1"])}
    if kind == "norm_proj":
        d = {"x": _activations(gen, case["rows"], case["hidden"], case["outliers"]),
             "g": _normal(gen, case["hidden"]).mul_(0.2).add_(1.0)}
        return d | {"w%d" % i: _blocks(gen, t, case["hidden"], case["n%d" % i]) for i in range(3)}
    if kind == "linear":
        x = _activations(gen, case["rows"], case["k"], case["outliers"])
        return {"x": x if case["x"] == "f32" else x.to(torch.bfloat16), "w": _blocks(gen, t, case["k"], case["n"]),
                "bias": _normal(gen, case["n"]) if case["bias"] else None}
    if kind == "mlp":
        h, i = case["hidden"], case["inter"]
        return {"x": _normal(gen, case["rows"], h), "gate": _blocks(gen, t, h, i), "up": _blocks(gen, t, h, i),
                "down": _blocks(gen, TYPES[case["down"]], i, h)}
    return {"layers": [_layer_inputs(gen, case) for _ in range(case["layers"])]}


def _layer_inputs(gen, case):
    h, i, r = case["hidden"], case["inter"], case["rows"]
    return {"h": _normal(gen, r, h), "attn": _normal(gen, r, h), "h2": _normal(gen, r, h),
            "g1": _normal(gen, h).mul_(0.2).add_(1.0), "g2": _normal(gen, h).mul_(0.2).add_(1.0),
            "q": _blocks(gen, Q4_K, h, h), "k": _blocks(gen, Q4_K, h, case["kv"]), "v": _blocks(gen, Q6_K, h, case["kv"]),
            "o": _blocks(gen, Q4_K, h, h), "gate": _blocks(gen, Q4_K, h, i), "up": _blocks(gen, Q4_K, h, i),
            "down": _blocks(gen, Q6_K, i, h)}


# ---- the calls --------------------------------------------------------------

def _array(kind, values):
    return (kind * len(values))(*values)


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _f32(*shape):
    return torch.empty(*shape, dtype=torch.float32, device="cuda")


def _ptrs(ts):
    return _array(ctypes.c_void_p, [t.data_ptr() for t in ts])


def _layer_calls(case, d, keep):
    """The quantized calls of one layer as (entry point, arguments without the
    stream); attention and the residual sums between them are the caller's."""
    r, h, kv, i = case["rows"], case["hidden"], case["kv"], case["inter"]
    n1, n2 = _f32(r, h), _f32(r, h)
    q, k, v, o, m, gb, ub = _f32(r, h), _f32(r, kv), _f32(r, kv), _f32(r, h), _f32(r, h), _f32(r, i), _f32(r, i)
    ws = [d["q"], d["k"], d["v"]]
    keep += [n1, n2, gb, ub]
    return [
        ("okq_rmsnorm", (d["h"].data_ptr(), r, h, d["g1"].data_ptr(), EPS, n1.data_ptr())),
        ("okq_linear_multi_q", (n1.data_ptr(), r, h, 3, _array(ctypes.c_uint32, [Q4_K, Q4_K, Q6_K]), _ptrs(ws),
                                _array(ctypes.c_uint64, [w.numel() for w in ws]),
                                _array(ctypes.c_int64, [h, kv, kv]), None, _ptrs([q, k, v]))),
        ("okq_linear_out_by_in_q", (d["attn"].data_ptr(), r, h, Q4_K, d["o"].data_ptr(), d["o"].numel(), h, None,
                                    o.data_ptr())),
        ("okq_rmsnorm", (d["h2"].data_ptr(), r, h, d["g2"].data_ptr(), EPS, n2.data_ptr())),
        ("okq_mlp_gated_silu_q", (n2.data_ptr(), r, h, i, Q4_K, d["gate"].data_ptr(), d["gate"].numel(), Q4_K,
                                  d["up"].data_ptr(), d["up"].numel(), Q6_K, d["down"].data_ptr(), d["down"].numel(),
                                  gb.data_ptr(), ub.data_ptr(), m.data_ptr())),
    ], {"q": q, "k": k, "v": v, "o": o, "mlp": m}


_side = []  # the stream that decode graphs are captured on


def prepare(case, seed):
    okq.call("okq_init", 0)
    d, kind = _inputs(case, seed), case["kind"]
    t = TYPES[case["type"]] if "type" in case else None
    if kind == "decode":
        calls, outs, keep = [], [], []
        for layer in d["layers"]:
            c, o = _layer_calls(case, layer, keep)
            calls += c
            outs.append(o)
        if not _side:
            _side.append(torch.cuda.Stream())
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.stream(_side[0]):
            for name, args in calls:  # sizes the stream's workspace
                okq.call(name, *args, _stream())
        _side[0].synchronize()
        with torch.cuda.graph(graph, stream=_side[0]):
            for name, args in calls:
                okq.call(name, *args, _stream())
        return {"graph": graph, "out": outs, "keep": [d, calls, keep]}
    if kind == "gather":
        out = _f32(case["n"], case["ne0"])
        ids = _array(ctypes.c_uint32, d["ids"].tolist())
        args = (t, d["w"].data_ptr(), d["w"].numel(), case["ne0"], case["ne1"], ids, case["n"], out.data_ptr())
        return {"call": ("okq_get_rows_q", args), "out": out, "keep": d}
    if kind == "dequant":
        out = _f32(case["ne1"], case["ne0"])
        args = (t, d["w"].data_ptr(), case["ne1"] * case["ne0"], out.data_ptr())
        return {"call": ("okq_dequantize", args), "out": out, "keep": d}
    if kind == "norm_proj":
        ws, ns = [d["w0"], d["w1"], d["w2"]], [case["n0"], case["n1"], case["n2"]]
        out = [_f32(case["rows"], n) for n in ns]
        args = (d["x"].data_ptr(), case["rows"], case["hidden"], d["g"].data_ptr(), EPS, t, 3, _ptrs(ws),
                _array(ctypes.c_uint64, [w.numel() for w in ws]), _array(ctypes.c_int64, ns), None, _ptrs(out))
        return {"call": ("okq_rmsnorm_linear_q_multi", args), "out": out, "keep": d}
    if kind == "mlp":
        r, h, i, dt = case["rows"], case["hidden"], case["inter"], TYPES[case["down"]]
        out, gb, ub = _f32(r, h), _f32(r, i), _f32(r, i)
        args = (d["x"].data_ptr(), r, h, i, t, d["gate"].data_ptr(), d["gate"].numel(), t, d["up"].data_ptr(),
                d["up"].numel(), dt, d["down"].data_ptr(), d["down"].numel(), gb.data_ptr(), ub.data_ptr(),
                out.data_ptr())
        return {"call": ("okq_mlp_gated_silu_q", args), "out": out, "keep": [d, gb, ub]}
    out = _f32(case["rows"], case["n"])
    name = "okq_linear_out_by_in_q" + ("_bf16" if case["x"] == "bf16" else "")
    args = (d["x"].data_ptr(), case["rows"], case["k"], t, d["w"].data_ptr(), d["w"].numel(), case["n"],
            d["bias"].data_ptr() if case["bias"] else None, out.data_ptr())
    return {"call": (name, args), "out": out, "keep": d}


def run(state):
    if "graph" in state:
        state["graph"].replay()
    else:
        name, args = state["call"]
        okq.call(name, *args, _stream())
    return state["out"]


# ---- what a pass cannot do without ---------------------------------------------

def _tensor_bytes(t, k, n):
    return k // ELEMS[t] * BYTES[t] * n


def work(case):
    kind = case["kind"]
    t = TYPES[case["type"]] if "type" in case else None
    if kind == "gather":
        rows = case["n"]
        return {"bytes": rows * (4 + _tensor_bytes(t, case["ne0"], 1) + 4 * case["ne0"]), "flops": 0}
    if kind == "dequant":
        n = case["ne0"] * case["ne1"]
        return {"bytes": _tensor_bytes(t, case["ne0"], case["ne1"]) + 4 * n, "flops": 0}
    r = case["rows"]
    if kind == "norm_proj":
        h, n = case["hidden"], case["n0"] + case["n1"] + case["n2"]
        return {"bytes": _tensor_bytes(t, h, n) + 4 * (r * h + h + r * n), "flops": 2 * r * h * n}
    if kind == "linear":
        k, n = case["k"], case["n"]
        xb = 4 if case["x"] == "f32" else 2
        return {"bytes": _tensor_bytes(t, k, n) + xb * r * k + 4 * r * n + (4 * n if case["bias"] else 0),
                "flops": 2 * r * k * n}
    h, i = case["hidden"], case["inter"]
    if kind == "mlp":
        return {"bytes": 2 * _tensor_bytes(t, h, i) + _tensor_bytes(TYPES[case["down"]], i, h) + 8 * r * h,
                "flops": 6 * r * h * i}
    kv = case["kv"]
    b = (_tensor_bytes(Q4_K, h, 2 * h + kv + 2 * i) + _tensor_bytes(Q6_K, h, kv) + _tensor_bytes(Q6_K, i, h)
         + 4 * (r * (3 * h) + 2 * h + r * (3 * h + 2 * kv)))
    return {"bytes": case["layers"] * b, "flops": case["layers"] * 2 * r * h * (2 * h + 2 * kv + 3 * i)}


def tolerance(case):
    if case["kind"] in ("gather", "dequant"):
        return "exact"
    if case["rows"] <= 8:
        # up to eight rows may contract activations rounded to 16 bits of
        # their run's largest value: 1e-4 against float64, 3e-4 through an MLP
        return {"rel": 4e-4 if case["kind"] in ("norm_proj", "linear") else 1.3e-3}
    # f32 sums of exact products: up to 7e-7 against float64
    return {"rel": 3e-6}


# ---- the same in 64 bits ----------------------------------------------------------

def _half(b):
    return b.contiguous().view(torch.float16).to(torch.float64)


def _weights(w, t, k):
    """Block bytes [n, row bytes] -> float64 [n, k], from the GGUF block layout."""
    n = w.shape[0]
    b = w.reshape(-1, BYTES[t])
    nb = b.shape[0]
    if t == Q8_0:
        v = _half(b[:, :2]) * b[:, 2:].contiguous().view(torch.int8).to(torch.float64)
    elif t == Q4_0:
        q = torch.cat([b[:, 2:] & 15, b[:, 2:] >> 4], 1).to(torch.float64)
        v = _half(b[:, :2]) * (q - 8)
    elif t == Q6_K:
        ql, qh = b[:, :128].reshape(nb, 2, 2, 32), b[:, 128:192].reshape(nb, 2, 32)
        lo = torch.stack([ql[:, :, 0] & 15, ql[:, :, 1] & 15, ql[:, :, 0] >> 4, ql[:, :, 1] >> 4], 2)
        hi = torch.stack([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (lo | (hi << 4)).reshape(nb, 16, 16).to(torch.float64) - 32
        sc = b[:, 192:208].contiguous().view(torch.int8).to(torch.float64)
        v = _half(b[:, 208:])[:, :, None] * sc[:, :, None] * q
    else:
        s = b[:, 4:16].to(torch.int16)
        lo, mid, top = s[:, :4], s[:, 4:8], s[:, 8:]
        sc = torch.cat([lo & 63, (top & 15) | ((lo >> 6) << 4)], 1).to(torch.float64)
        m = torch.cat([mid & 63, (top >> 4) | ((mid >> 6) << 4)], 1).to(torch.float64)
        qs = b[:, BYTES[t] - 128:].reshape(nb, 4, 32)
        q = torch.stack([qs & 15, qs >> 4], 2).reshape(nb, 8, 32)
        if t == Q5_K:
            q = q | (torch.stack([(b[:, 16:48] >> j) & 1 for j in range(8)], 1) << 4)
        d, dmin = _half(b[:, :2])[:, :, None], _half(b[:, 2:4])[:, :, None]
        v = d * sc[:, :, None] * q.to(torch.float64) - dmin * m[:, :, None]
    return v.reshape(n, k)


def _linear(x, w, t, k, bias=None):
    step = max(1, (1 << 27) // k)
    y = torch.cat([x @ _weights(w[i:i + step], t, k).t() for i in range(0, w.shape[0], step)], 1)
    return y if bias is None else y + bias.to(torch.float64)


def _norm(x, g):
    x = x.to(torch.float64)
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * g.to(torch.float64)


def _mlp(x, gate, up, t, down, dt):
    h, i = x.shape[1], gate.shape[0]
    g, u = _linear(x, gate, t, h), _linear(x, up, t, h)
    return _linear(g * torch.sigmoid(g) * u, down, dt, i)


def exact(case, seed):
    d, kind = _inputs(case, seed), case["kind"]
    t = TYPES[case["type"]] if "type" in case else None
    if kind == "gather":
        return _weights(d["w"][d["ids"].cuda()], t, case["ne0"])
    if kind == "dequant":
        return _weights(d["w"], t, case["ne0"])
    if kind == "norm_proj":
        xn = _norm(d["x"], d["g"])
        return [_linear(xn, d["w%d" % i], t, case["hidden"]) for i in range(3)]
    if kind == "linear":
        return _linear(d["x"].to(torch.float64), d["w"], t, case["k"], d["bias"])
    if kind == "mlp":
        return _mlp(d["x"].to(torch.float64), d["gate"], d["up"], t, d["down"], TYPES[case["down"]])
    out, h = [], case["hidden"]
    for c in d["layers"]:
        n1, n2 = _norm(c["h"], c["g1"]), _norm(c["h2"], c["g2"])
        out.append({"q": _linear(n1, c["q"], Q4_K, h), "k": _linear(n1, c["k"], Q4_K, h),
                    "v": _linear(n1, c["v"], Q6_K, h), "o": _linear(c["attn"].to(torch.float64), c["o"], Q4_K, h),
                    "mlp": _mlp(n2, c["gate"], c["up"], Q4_K, c["down"], Q6_K)})
    return out
