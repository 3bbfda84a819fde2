"""The work that the library's speed is judged by: its quantized GEMV at the token counts of decoding
and speculative verification, the multi-row product of prompts, the MoE layer from one token to a
512-token batch, and the whole model calls (one decode step, one prompt) of a MoE and a dense model.

Weights, activations and caches are synthetic and made on the GPU from the seed: block-quantized
weights of N(0, 0.03)-like spread in the block layouts of include/qr_hip.h, N(0, 1) activations, and a
router whose experts' popularity follows a Zipf law.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "quantr-in-c_amd"))
import quantr_amd as Q  # noqa: E402

TYPES = {"q8_0": Q.TYPE_Q8_0, "q4k": Q.TYPE_Q4_K, "q5k": Q.TYPE_Q5_K, "q6k": Q.TYPE_Q6_K}
BLOCK = {"q8_0": (32, 34), "q4k": (256, 144), "q5k": (256, 176), "q6k": (256, 210)}
ORDERS = {"seq": Q.ORDER_SEQ, "avx2": Q.ORDER_AVX2, "avx512": Q.ORDER_AVX512}
KV = {"f32": Q.KV_F32, "f16": Q.KV_F16, "q8_0": Q.KV_Q8_0}

# Layer shapes that the benchmark and the tests use.
MOE = {
    "qwen3": dict(dim=2048, hidden=768, E=128, K=8, up="q4k", down="q6k", shared=0),
    "qwen15": dict(dim=2048, hidden=1408, E=60, K=4, up="q4k", down="q8_0", shared=5632),
}
MODEL = {
    "moe": dict(dim=2048, heads=32, kv_heads=4, hd=128, vocab=151936, base=1e6, page=256),
    "dense": dict(dim=2048, heads=32, kv_heads=4, hd=64, vocab=32000, base=10000.0, page=256,
                  hidden=5632, up="q4k", down="q6k"),
}


def listed():
    return [
        # one attention projection of one decoded token: the smallest call, launch and latency
        dict(name="gemv_q4k_2048x2048_t1", kind="gemv", type="q4k", layout="tiled", n=2048, d=2048,
             nt=1, order="seq"),
        # the 32000-row output matrix of one decoded token: the benchmark's headline
        dict(name="gemv_q4k_32000x2048_t1", kind="gemv", type="q4k", layout="tiled", n=32000, d=2048,
             nt=1, order="seq"),
        # the same matrix for four tokens of a speculative verification
        dict(name="gemv_q4k_32000x2048_t4", kind="gemv", type="q4k", layout="tiled", n=32000, d=2048,
             nt=4, order="seq"),
        # an FFN up projection as the file stores it, eight tokens, the AVX2 build's dot
        dict(name="gemv_q8_0_5632x2048_t8", kind="gemv", type="q8_0", layout="rows", n=5632, d=2048,
             nt=8, order="avx2"),
        # a llama.cpp checkpoint's FFN matrix for three tokens
        dict(name="gemv_q6k_ggml_5632x2048_t3", kind="gemv", type="q6k", layout="ggml", n=5632,
             d=2048, nt=3, order="seq"),
        # the stacked q / k projection of a short prompt, an odd number of tokens
        dict(name="rows_q4k_4608x2048_T131", kind="rows", type="q4k", layout="tiled", n=4608, d=2048,
             T=131, order="seq"),
        # the MoE layer of one decoded token, of a small batch, and of a prompt chunk
        dict(name="moe_qwen3_T1", kind="moe", shape="qwen3", T=1, order="avx2"),
        dict(name="moe_qwen3_T16", kind="moe", shape="qwen3", T=16, order="avx2"),
        dict(name="moe_qwen3_T512", kind="moe", shape="qwen3", T=512, order="avx2"),
        # a decoded token late in a long conversation (Q8_0 cache)
        dict(name="decode_moe_pos4095", kind="decode", model="moe", layers=8, pos=4095, kv="q8_0",
             order="avx2"),
        # a decoded token of a dense model with the reference's fp16 cache, mid-conversation
        dict(name="decode_dense_pos701", kind="decode", model="dense", layers=8, pos=701, kv="f16",
             order="seq"),
        # a prompt of 512 tokens into an empty cache
        dict(name="prefill_moe_512", kind="prefill", model="moe", layers=4, pos=0, tokens=512,
             kv="q8_0", order="avx2"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "rows", "moe", "decode", "prefill"])
    order = rng.choice(["seq", "avx2"])
    if kind == "gemv":
        layout = rng.choice(["tiled", "tiled", "rows", "ggml"])
        t = rng.choice(["q4k", "q5k", "q6k"] if layout == "ggml" else ["q8_0", "q4k", "q5k", "q6k"])
        n = _log(rng, 256, 32000)
        d = 256 * rng.randint(2, 22)
        if layout == "rows" and t == "q8_0":
            d += 32 * rng.randint(0, 7)
        if layout == "tiled":
            n = max(8, n // 8 * 8)
            order = "seq"
        # eight tokens of a row-major matrix have to fit the call's limit on their length
        nt = rng.choice([1, 1, 2, 3, 4, 8] if layout != "rows" or d <= 2048 else [1, 1, 2, 3, 4])
        return dict(kind=kind, type=t, layout=layout, n=n, d=d, nt=nt, order=order)
    if kind == "rows":
        t = rng.choice(["q8_0", "q4k", "q4k", "q5k", "q6k"])
        layout = rng.choice(["rows", "tiled"]) if t in ("q4k", "q5k") else "rows"
        return dict(kind=kind, type=t, layout=layout, n=_log(rng, 256, 5632),
                    d=256 * rng.randint(2, 22), T=_log(rng, 9, 512), order="seq")
    if kind == "moe":
        shape = rng.choice(["qwen3", "qwen3", "qwen15"])
        return dict(kind=kind, shape=shape, T=_log(rng, 1, 512 if shape == "qwen3" else 64),
                    order=order if shape == "qwen3" else "seq")
    model = rng.choice(["moe", "dense"])
    kv = rng.choice(["q8_0", "f16", "f32"])
    if kind == "decode":
        return dict(kind=kind, model=model, layers=rng.randint(4, 8),
                    pos=_log(rng, 1, 4096 if model == "moe" else 2047), kv=kv, order=order)
    tokens = _log(rng, 16, 320)
    return dict(kind=kind, model=model, layers=rng.randint(2, 4), tokens=tokens,
                pos=rng.choice([0, 0, rng.randint(1, 300)]), kv=kv, order=order)


# ---- synthetic weights ------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _half(g, shape, scale):
    """fp16 block scales around `scale`, as bytes; always normal halves."""
    v = scale * (0.8 + 0.45 * torch.rand(shape, device="cuda", generator=g))
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _blocks(g, t, rows, d, ggml=False):
    """rows x (d / block) random blocks, uint8 [rows, blocks * bytes]."""
    be, bb = BLOCK[t]
    nb = d // be
    w = torch.randint(0, 256, (rows * nb, bb), device="cuda", generator=g, dtype=torch.uint8)
    m = rows * nb
    if t == "q8_0":
        w[:, 0:2] = _half(g, (m,), 4.7e-4)
    elif t == "q6k":
        sc = torch.randint(12, 25, (m, 16), device="cuda", generator=g)
        w[:, 192:208] = (sc if ggml else sc * (torch.arange(16, device="cuda") < 8)).to(torch.uint8)
        w[:, 208:210] = _half(g, (m,), 7.8e-5)
    else:
        top = 15.0 if t == "q4k" else 31.0
        scale = 2.4e-3 / top
        w[:, 0:2] = _half(g, (m,), scale)
        if ggml:  # 12 packed bytes of random 6-bit scales and mins
            w[:, 2:4] = _half(g, (m,), scale * top / 2)
        else:  # 6-bit scale and 2-bit min per 32 elements, 4 unused bytes
            w[:, 2:4] = _half(g, (m,), scale * top / 2 * 16)
            sc = torch.randint(32, 64, (m, 8), device="cuda", generator=g)
            mn = 2 + (torch.rand((m, 8), device="cuda", generator=g) < 0.9).to(sc.dtype)
            w[:, 4:12] = (sc | (mn << 6)).to(torch.uint8)
            w[:, 12:16] = 0
    return w.view(rows, nb * bb)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, device="cuda", generator=g) * std


def _zipf(g, E, dim):
    """Router rows and a direction u: tokens z + 8 u see Zipf(1.1) logits."""
    G = _normal(g, E, dim, std=0.02)
    u = _normal(g, dim)
    u = u / u.norm()
    G = G - torch.outer(G @ u, u)
    p = 1.0 / torch.arange(1, E + 1, device="cuda", dtype=torch.float32) ** 1.1
    b = torch.log(p / p.sum())[torch.randperm(E, device="cuda", generator=g)]
    return (G + torch.outer(b / 8.0, u)).contiguous(), u


def _zipf_tokens(g, T, dim, u):
    z = _normal(g, T, dim)
    return (z - torch.outer(z @ u, u) + 8.0 * u).contiguous()


_DEV = []


def _dev():
    if not _DEV:
        _DEV.append(Q.Device(0))
    return _DEV[0]


def _tile(t, w, n, d):
    """The tiled copy of a matrix, as the GGUF loader stores it."""
    out = torch.empty_like(w)
    torch.cuda.synchronize()
    _dev().tile(TYPES[t], w.data_ptr(), out.data_ptr(), n, d)
    _dev().sync()
    return out


def _matrix(case, seed):
    g = _gen(seed)
    w = _blocks(g, case["type"], case["n"], case["d"], case["layout"] == "ggml")
    x = _normal(g, case["nt"] if case["kind"] == "gemv" else case["T"], case["d"])
    return w, x


def _moe_tensors(g, s):
    E, dim, hid = s["E"], s["dim"], s["hidden"]
    router, u = _zipf(g, E, dim)
    w = dict(router=router, up=_blocks(g, s["up"], E * hid, dim),
             gate=_blocks(g, s["up"], E * hid, dim), down=_blocks(g, s["down"], E * dim, hid))
    if s["shared"]:
        w["shared"] = dict(gate_inp=_normal(g, dim, std=0.02),
                           up=_blocks(g, "q4k", s["shared"], dim),
                           gate=_blocks(g, "q4k", s["shared"], dim),
                           down=_blocks(g, "q4k", dim, s["shared"]))
    return w, u


def _moe_inputs(case, seed):
    s = MOE[case["shape"]]
    g = _gen(seed)
    w, u = _moe_tensors(g, s)
    return s, w, _normal(g, case["T"], s["dim"]), _zipf_tokens(g, case["T"], s["dim"], u)


def _model_tensors(case, seed):
    """A model's tensors, row-major, and the tokens and cached K / V values of a call."""
    m = MODEL[case["model"]]
    g = _gen(seed)
    dim, qd, kvd = m["dim"], m["heads"] * m["hd"], m["kv_heads"] * m["hd"]
    layers = []
    for _ in range(case["layers"]):
        w = dict(rms_att=1 + _normal(g, dim, std=0.1), rms_ffn=1 + _normal(g, dim, std=0.1),
                 wqk=_blocks(g, "q4k", qd + kvd, dim), wv=_blocks(g, "q6k", kvd, dim),
                 wo=_blocks(g, "q4k", dim, qd))
        if case["model"] == "moe":
            w["moe"], _ = _moe_tensors(g, MOE["qwen3"])
        else:
            w["up"] = _blocks(g, m["up"], m["hidden"], dim)
            w["gate"] = _blocks(g, m["up"], m["hidden"], dim)
            w["down"] = _blocks(g, m["down"], dim, m["hidden"])
        n = case["pos"]
        w["k"], w["v"] = _normal(g, n, kvd), _normal(g, n, kvd)
        layers.append(w)
    top = dict(embd=_blocks(g, "q4k", m["vocab"], dim), rms=1 + _normal(g, dim, std=0.1),
               wcls=_blocks(g, "q6k", m["vocab"], dim))
    tokens = torch.randint(0, m["vocab"], (case.get("tokens", 1),), device="cuda", generator=g)
    return m, layers, top, tokens.cpu().numpy().astype(np.int32)


def _prepare_model(case, seed):
    m, layers, top, tokens = _model_tensors(case, seed)
    dim, qd, kvd = m["dim"], m["heads"] * m["hd"], m["kv_heads"] * m["hd"]
    keep, lay = [], []
    dense = case["model"] == "dense"

    def hold(t):
        keep.append(t)
        return t.data_ptr()

    qbytes = qd * Q_row("q4k", dim)
    for w in layers:
        # wq and wk tiled one after the other, as the GGUF loader stores them
        qk = torch.cat([_tile("q4k", w["wqk"][:qd].contiguous(), qd, dim).view(-1),
                        _tile("q4k", w["wqk"][qd:].contiguous(), kvd, dim).view(-1)])
        q = hold(qk)
        y = dict(rms_att=hold(w["rms_att"]), rms_ffn=hold(w["rms_ffn"]), wq=q, wk=q + qbytes,
                 wv=hold(w["wv"]), wo=hold(_tile("q4k", w["wo"], dim, qd)))
        if dense:
            y.update(router=0, up=hold(_tile("q4k", w["up"], m["hidden"], dim)),
                     gate=hold(_tile("q4k", w["gate"], m["hidden"], dim)), down=hold(w["down"]))
        else:
            y.update({k: hold(w["moe"][k]) for k in ("router", "up", "gate", "down")})
        lay.append(y)
    T4 = Q.TYPE_Q4_K | Q.TILED
    seq = case["pos"] + case.get("tokens", 1)
    s = MOE["qwen3"]
    spec = dict(dim=dim, n_heads=m["heads"], n_kv_heads=m["kv_heads"], head_dim=m["hd"],
                n_layers=case["layers"], vocab=m["vocab"], seq_len=max(16, seq), rope_base=m["base"],
                tok_embd=hold(top["embd"]), tok_type=Q.TYPE_Q4_K, rms_final=hold(top["rms"]),
                wcls=hold(_tile("q6k", top["wcls"], m["vocab"], dim)),
                wcls_type=Q.TYPE_Q6_K | Q.TILED, wtype=(T4, T4, Q.TYPE_Q6_K, T4),
                E=0 if dense else s["E"], K=0 if dense else s["K"],
                hidden=m["hidden"] if dense else s["hidden"],
                up_type=T4 if dense else Q.TYPE_Q4_K, down_type=Q.TYPE_Q6_K, layers=lay)
    dev = _dev()
    model, larr, refs = Q.upload_decode_model(dev, spec)
    torch.cuda.synchronize()
    dec = Q.Decoder(dev, model, larr, kv_type=KV[case["kv"]], order=ORDERS[case["order"]],
                    page=m["page"], flags=Q.DEC_GRAPH)
    for i, w in enumerate(layers):
        if case["pos"]:
            dec.kv_write(i, 0, case["pos"], w["k"].data_ptr(), w["v"].data_ptr())
    dev.sync()
    return dict(case=case, dec=dec, keep=(keep, refs, model, larr), tokens=tokens,
                logits=torch.zeros(m["vocab"], device="cuda"), x=torch.zeros(dim, device="cuda"))


def Q_row(t, d):
    return d // BLOCK[t][0] * BLOCK[t][1]


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "rows"):
        w, x = _matrix(case, seed)
        typ = TYPES[case["type"]]
        if case["layout"] == "tiled":
            w, typ = _tile(case["type"], w, case["n"], case["d"]), typ | Q.TILED
        elif case["layout"] == "ggml":
            typ |= Q.GGML
        y = torch.zeros(x.shape[0], case["n"], device="cuda")
        return dict(case=case, w=w, x=x, y=y, typ=typ)
    if kind == "moe":
        s, w, x, xb = _moe_inputs(case, seed)
        T = case["T"]
        L = Q.MoeLayer(s["dim"], s["hidden"], s["E"], s["K"], w["router"].data_ptr(),
                       w["up"].data_ptr(), w["gate"].data_ptr(), w["down"].data_ptr(),
                       TYPES[s["up"]], TYPES[s["up"]], TYPES[s["down"]])
        if s["shared"]:
            sh = w["shared"]
            L.sh_hidden = s["shared"]
            L.sh_gate_inp, L.sh_up = sh["gate_inp"].data_ptr(), sh["up"].data_ptr()
            L.sh_gate, L.sh_down = sh["gate"].data_ptr(), sh["down"].data_ptr()
            L.sh_up_type = L.sh_gate_type = L.sh_down_type = Q.TYPE_Q4_K
        return dict(case=case, L=L, w=w, x=x, xb=xb,
                    idx=torch.zeros(T, s["K"], device="cuda", dtype=torch.int32),
                    wts=torch.zeros(T, s["K"], device="cuda"))
    return _prepare_model(case, seed)


def run(state):
    case, dev = state["case"], _dev()
    kind, order = case["kind"], ORDERS[case["order"]]
    if kind == "gemv":
        dev.gemv(state["typ"], state["w"].data_ptr(), state["x"].data_ptr(), state["y"].data_ptr(),
                 case["n"], case["d"], case["nt"], order=order)
        return state["y"]
    if kind == "rows":
        dev.gemv_rows(state["typ"], state["w"].data_ptr(), state["x"].data_ptr(),
                      state["y"].data_ptr(), case["n"], case["d"], case["T"], order=order)
        return state["y"]
    if kind == "moe":
        dev.moe_forward(state["L"], state["x"].data_ptr(), state["xb"].data_ptr(), case["T"], order,
                        state["idx"].data_ptr(), state["wts"].data_ptr())
        return dict(x=state["x"], idx=state["idx"], wts=state["wts"])
    dec = state["dec"]
    if kind == "decode":
        dec.forward(int(state["tokens"][0]), case["pos"], state["logits"].data_ptr(),
                    state["x"].data_ptr())
    else:
        dec.prefill(state["tokens"], case["pos"], state["logits"].data_ptr(), state["x"].data_ptr())
    return dict(logits=state["logits"], x=state["x"])


# ---- bytes and operations -----------------------------------------------------------------------
def _moe_work(s, T):
    """Weight bytes of the experts that T tokens touch (expected under the Zipf router, at most all)
    and the products' operations."""
    p = [1.0 / i ** 1.1 for i in range(1, s["E"] + 1)]
    tot = sum(p)
    touched = min(s["E"], sum(1 - (1 - min(1.0, s["K"] * q / tot)) ** T for q in p))
    touched = max(touched, float(s["K"]))
    dim, hid = s["dim"], s["hidden"]
    expert = 2 * hid * Q_row(s["up"], dim) + dim * Q_row(s["down"], hid)
    b = 4 * s["E"] * dim + touched * expert
    f = 2.0 * T * (s["E"] * dim + s["K"] * 3 * dim * hid)
    if s["shared"]:
        b += 3 * s["shared"] * Q_row("q4k", dim)
        f += 2.0 * T * 3 * dim * s["shared"]
    return b, f


def work(case):
    kind = case["kind"]
    if kind in ("gemv", "rows"):
        T = case["nt"] if kind == "gemv" else case["T"]
        n, d = case["n"], case["d"]
        return {"bytes": n * Q_row(case["type"], d) + 4 * T * (d + n), "flops": 2.0 * T * n * d}
    if kind == "moe":
        s = MOE[case["shape"]]
        b, f = _moe_work(s, case["T"])
        return {"bytes": b + 4 * case["T"] * (3 * s["dim"] + 2 * s["K"]), "flops": f}
    m, T = MODEL[case["model"]], case.get("tokens", 1)
    dim, qd, kvd = m["dim"], m["heads"] * m["hd"], m["kv_heads"] * m["hd"]
    row = {"f32": 4 * kvd, "f16": 2 * kvd, "q8_0": kvd // 32 * 34}[case["kv"]]
    if case["model"] == "moe":
        b, f = _moe_work(MOE["qwen3"], T)
    else:
        b = 2 * m["hidden"] * Q_row(m["up"], dim) + dim * Q_row(m["down"], m["hidden"])
        f = 2.0 * T * 3 * dim * m["hidden"]
    b += (qd + kvd) * Q_row("q4k", dim) + kvd * Q_row("q6k", dim) + dim * Q_row("q4k", qd) + 8 * dim
    f += 2.0 * T * dim * (2 * qd + 2 * kvd)
    b += 2 * row * (case["pos"] + T)
    f += 4.0 * qd * sum(case["pos"] + t + 1 for t in range(T))
    b = b * case["layers"] + T * Q_row("q4k", dim) + m["vocab"] * (Q_row("q6k", dim) + 4)
    return {"bytes": b, "flops": f * case["layers"] + 2.0 * dim * m["vocab"]}


def tolerance(case):
    """The library promises the reference build's results bit for bit: every float operation in the
    reference's order, rounded once.  Any correct implementation gives the same bits."""
    return "exact"


# ---- the same results in 64 bits, with plain torch ---------------------------------------------
def _h(b):
    """Two bytes -> the (normal) half they hold, float64 [..., 1]."""
    return b.contiguous().view(torch.float16).to(torch.float64)


def _nib(b):
    """[..., k] bytes -> [..., 2k] nibbles, low first."""
    return torch.stack([b & 15, b >> 4], -1).flatten(-2).to(torch.float64)


def _dequant(t, w, ggml=False):
    """uint8 [rows, bytes] -> float64 [rows, d]."""
    be, bb = BLOCK[t]
    rows = w.shape[0]
    b = w.reshape(-1, bb)
    if t == "q8_0":
        v = b[:, 2:].contiguous().view(torch.int8).to(torch.float64) * _h(b[:, 0:2])
    elif t == "q6k" and not ggml:
        hi = torch.stack([(b[:, 128:192] >> s) & 3 for s in (0, 2, 4, 6)], -1).flatten(-2)
        q = _nib(b[:, :128]) + 16.0 * hi.to(torch.float64) - 32.0
        v = q * (b[:, 192:200].to(torch.float64) * _h(b[:, 208:210])).repeat_interleave(32, -1)
    elif t == "q6k":
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        parts = [(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                 (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)]
        q = torch.stack(parts, 2).reshape(-1, 256).to(torch.float64) - 32.0
        v = q * (b[:, 192:208].to(torch.float64) * _h(b[:, 208:210])).repeat_interleave(16, -1)
    else:
        at = 16 if t == "q4k" else 48
        s = b[:, 4:16]
        if ggml:
            sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], -1)
            mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], -1)
            qs = b[:, at:].reshape(-1, 4, 32)
            q = torch.stack([qs & 15, qs >> 4], 2).reshape(-1, 256).to(torch.float64)
            if t == "q5k":
                hi = torch.stack([(b[:, 16:48] >> j) & 1 for j in range(8)], 1).reshape(-1, 256)
                q = q + 16.0 * hi.to(torch.float64)
        else:
            sc, mn = s[:, :8] & 63, s[:, :8] >> 6
            q = _nib(b[:, at:])
            if t == "q5k":
                hi = torch.stack([(b[:, 16:48] >> j) & 1 for j in range(8)], -1).flatten(-2)
                q = q + 16.0 * hi.to(torch.float64)
        sc = (sc.to(torch.float64) * _h(b[:, 0:2])).repeat_interleave(32, -1)
        v = q * sc - (mn.to(torch.float64) * _h(b[:, 2:4])).repeat_interleave(32, -1)
    return v.reshape(rows, -1)


def _cut(f):
    """fp32 -> half with its mantissa cut, as float64 (normal range)."""
    f = (f.contiguous().view(torch.int32) & ~0x1FFF).view(torch.float32)
    return torch.where(f.abs() < 2.0 ** -14, torch.zeros_like(f), f).to(torch.float64)


def _q8(x):
    """The Q8_0 quantization of an activation (blocks of 32 along the last axis), dequantized."""
    v = x.to(torch.float32).reshape(*x.shape[:-1], -1, 32)
    dd = v.abs().amax(-1, keepdim=True) / 127.0
    inv = torch.where(dd != 0, 1.0 / dd, torch.zeros_like(dd))
    return (torch.round(v * inv).to(torch.float64) * _cut(dd)).reshape(x.shape)


def _q8k(x):
    """llama.cpp's Q8_K quantization (blocks of 256), dequantized."""
    v = x.to(torch.float32).reshape(*x.shape[:-1], -1, 256)
    top = torch.gather(v, -1, v.abs().argmax(-1, keepdim=True))
    s = -127.0 / top
    return (torch.round(v * s).clamp(max=127).to(torch.float64) / s.to(torch.float64)).reshape(x.shape)


def _mm(x, t, w):
    return _q8(x) @ _dequant(t, w).T


def _silu(v):
    return v / (1.0 + torch.exp(-v))


def _moe64(s, w, x, xb):
    """x + the layer of the tokens xb, float64 [T, dim]."""
    T, dim, hid, K = xb.shape[0], s["dim"], s["hidden"], s["K"]
    p = torch.softmax(xb.to(torch.float64) @ w["router"].to(torch.float64).T, -1)
    pw, pi = p.topk(K, -1)
    pw = pw / pw.sum(-1, keepdim=True)
    out = x.to(torch.float64).clone()
    xq = _q8(xb)
    for e in torch.unique(pi).tolist():
        tok, slot = (pi == e).nonzero(as_tuple=True)
        rows, drows = slice(e * hid, (e + 1) * hid), slice(e * dim, (e + 1) * dim)
        hb = _silu(xq[tok] @ _dequant(s["up"], w["up"][rows]).T) * (
            xq[tok] @ _dequant(s["up"], w["gate"][rows]).T)
        out.index_add_(0, tok, pw[tok, slot, None] * _mm(hb, s["down"], w["down"][drows]))
    if s["shared"]:
        sh = w["shared"]
        hb = _silu(xq @ _dequant("q4k", sh["up"]).T) * (xq @ _dequant("q4k", sh["gate"]).T)
        g = 1.0 / (1.0 + torch.exp(-(xb.to(torch.float64) @ sh["gate_inp"].to(torch.float64))))
        out = out + g[:, None] * _mm(hb, "q4k", sh["down"])
    return out


def _rms(x, w):
    return w.to(torch.float64) * (x * (1.0 / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)))


def _kv64(kind, v):
    if not v.numel():
        return v.to(torch.float64)
    return _q8(v) if kind == "q8_0" else _cut(v.to(torch.float32)) if kind == "f16" else (
        v.to(torch.float64))


def _model64(case, seed):
    m, layers, top, tokens = _model_tensors(case, seed)
    dim, hd, H, KH = m["dim"], m["hd"], m["heads"], m["kv_heads"]
    qd, kvd, pos, T = H * hd, KH * hd, case["pos"], len(tokens)
    x = _dequant("q4k", top["embd"][torch.from_numpy(tokens).to("cuda").long()])
    i = torch.arange(0, qd, 2, device="cuda", dtype=torch.float32)
    freq = torch.pow(torch.tensor(m["base"], device="cuda", dtype=torch.float32), -(i / float(hd)))
    at = torch.arange(pos, pos + T, device="cuda", dtype=torch.float32)
    theta = (at[:, None] * freq).to(torch.float64)
    cos, sin = torch.cos(theta), torch.sin(theta)

    def rope(v):
        a, b = v[:, 0::2], v[:, 1::2]
        c, s = cos[:, :a.shape[1]], sin[:, :a.shape[1]]
        return torch.stack([a * c - b * s, a * s + b * c], -1).flatten(-2)

    seen = torch.arange(pos + T, device="cuda")[None, :] <= torch.arange(
        pos, pos + T, device="cuda")[:, None]
    for w in layers:
        xb = _rms(x, w["rms_att"])
        qk = _mm(xb, "q4k", w["wqk"])
        q, k, v = rope(qk[:, :qd]), rope(qk[:, qd:]), _mm(xb, "q6k", w["wv"])
        K = torch.cat([_kv64(case["kv"], w["k"]), _kv64(case["kv"], k)])
        V = torch.cat([_kv64(case["kv"], w["v"]), _kv64(case["kv"], v)])
        ao = torch.empty(T, qd, device="cuda", dtype=torch.float64)
        for h in range(H):
            kv = slice(h * KH // H * hd, (h * KH // H + 1) * hd)
            hs = slice(h * hd, (h + 1) * hd)
            a = (q[:, hs] @ K[:, kv].T) / math.sqrt(hd)
            ao[:, hs] = torch.softmax(a.masked_fill(~seen, -math.inf), -1) @ V[:, kv]
        x = x + _mm(ao, "q4k", w["wo"])
        xb = _rms(x, w["rms_ffn"])
        if case["model"] == "moe":
            x = _moe64(MOE["qwen3"], w["moe"], x, xb)
        else:
            hb = _silu(_mm(xb, m["up"], w["up"])) * _mm(xb, m["up"], w["gate"])
            x = x + _mm(hb, m["down"], w["down"])
    x = x[-1]
    return dict(logits=_mm(_rms(x, top["rms"])[None], "q6k", top["wcls"])[0], x=x)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gemv", "rows"):
        w, x = _matrix(case, seed)
        ggml = case["layout"] == "ggml"
        d = case["d"] // BLOCK[case["type"]][0] * BLOCK[case["type"]][0]
        xq = _q8k(x[:, :d]) if ggml else _q8(x[:, :d])
        return xq @ _dequant(case["type"], w, ggml).T
    if kind == "moe":
        s, w, x, xb = _moe_inputs(case, seed)
        return dict(x=_moe64(s, w, x, xb), idx=None, wts=None)
    return _model64(case, seed)
