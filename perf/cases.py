"""The work this package is timed on: one pass of each public path, from a single decode row to whole layers.

A case is a dict of plain values. `listed()` names twelve; `draw(rng)` gives further ones of the same ranges. Three
families, as the package has them:

  12-bit weights, int8 activations   `w12` (one product), `mlp` (a vision MLP), `dec_prefill` / `dec_decode` (the int8
                                     decoder), `moe` (the routed expert layer)
  12-trit weights at the engine's    `ref_ffn` (a vision MLP of QuantLinears), `ref_prefill` / `ref_decode` (the
  own integer semantics              decoder), `ref_moe` (the routed expert layer)
  the LinearBackend seam             `backend` (host codes in, exact host sums out)

Every output is an integer that the semantics fix, so every case is compared exactly. Activations are normal (int8:
sigma 40 clipped to +-127; codes: a quarter of the level), weights normal at a quarter of their range, drawn on the GPU
from the seed. Whole models keep their layers' real shapes and have fewer of them (and a smaller vocabulary, in the
same proportion to the layers), which leaves each launch and its share of the pass as they are in the full model.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import tritify_amd as T
from tritify_amd import backend as B
from tritify_amd import workloads as W
from tritify_amd.decoder import DecoderModel
from tritify_amd.moe import MoeLayer
from tritify_amd.quant import qscale_record
from tritify_amd.refdecoder import RefDecoder
from tritify_amd.refmoe import RefMoeLayer
from tritify_amd.refvision import RefFeedForward

WLEVELS = 265720  # 12 trits: (3^12 - 1) / 2
ACT = 1 << 28  # the level of 12-trit activations
OUT = {"i64": B.OUT_I64, "i32": B.OUT_I32, "i8": B.OUT_I8}
OUT_BYTES = {"i64": 8, "i32": 4, "i8": 1}
TARGET = {"i64": 127, "i32": 16384, "i8": 127}  # what four standard deviations of a channel map to
DEV = "cuda"


def listed():
    return [
        # one decode row against a 4096 x 4096 projection: latency and the weight stream
        dict(name="w12_row", kind="w12", m=1, n=4096, k=4096, out="i8", planes="w12"),
        # a long prompt against the same projection, on the planes kept for it
        dict(name="w12_prompt", kind="w12", m=2048, n=4096, k=4096, out="i8", planes="w12b"),
        # the MLP of one image's stage-3 tokens (GELU as a code table), up and down
        dict(name="mlp_image", kind="mlp", tokens=4096, dim=448, hidden=1792),
        # a prompt of 512 tokens through the int8 decoder's layers and head
        dict(name="dec_prefill", kind="dec_prefill", tokens=512, layers=4, vocab=32768),
        # 8 greedy steps of that decoder behind such a prompt, from the captured step
        dict(name="dec_decode", kind="dec_decode", prompt=512, steps=8, layers=4, vocab=32768),
        # the expert layer on a prompt's tokens: each expert gets a few hundred rows
        dict(name="moe_prompt", kind="moe", tokens=4096, hidden=4096, ffn=1408, experts=128, top_k=8),
        # the same layer on a batch of decode rows: each expert gets a few rows, the weights are the work
        dict(name="moe_batch", kind="moe", tokens=48, hidden=4096, ffn=1408, experts=128, top_k=8),
        # the image MLP at the engine's own semantics: dynamic quantization, exact sums, GELU, twice
        dict(name="ref_ffn_image", kind="ref_ffn", rows=4096, dim=448, hidden=1792),
        # a prompt through the engine-semantics decoder's batched forward
        dict(name="ref_prefill", kind="ref_prefill", tokens=256, layers=2, vocab=8192),
        # 8 greedy steps of that decoder from the captured step, at a cache of 512 positions
        dict(name="ref_decode", kind="ref_decode", pos=512, steps=8, layers=2, vocab=8192),
        # the engine-semantics expert layer (sigmoid router, shared expert) on a batch of decode rows
        dict(name="ref_moe_batch", kind="ref_moe", tokens=64, dim=2048, hidden=1408, experts=16, top_k=4),
        # one projection of 64 rows through the LinearBackend seam, host buffers both ways, weights resident
        dict(name="backend_rows", kind="backend", rows=64, out=4864, k=896),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["w12"] * 3 + ["mlp", "dec_prefill", "dec_decode", "moe", "ref_ffn", "ref_ffn", "ref_prefill",
                                     "ref_decode", "ref_moe", "backend", "backend"])
    if kind == "w12":  # decode rows, batches and prompts; odd rows, channels and inner sizes
        m = _log(rng, 1, 4096)
        planes = "w12b" if m > 512 and rng.random() < 0.4 else "w12"
        return dict(kind=kind, m=m, n=_log(rng, 112, 8192), k=_log(rng, 128, 8192),
                    out=rng.choice(["i8", "i8", "i32", "i64"]), planes=planes)
    if kind == "mlp":  # the stages of an image encoder at several image sizes
        dim = rng.choice([112, 224, 448, 896])
        return dict(kind=kind, tokens=_log(rng, 49, 16384), dim=dim, hidden=4 * dim)
    if kind == "dec_prefill":
        return dict(kind=kind, tokens=_log(rng, 17, 600), layers=rng.choice([2, 3, 4]), vocab=_log(rng, 4096, 32768))
    if kind == "dec_decode":
        return dict(kind=kind, prompt=_log(rng, 16, 900), steps=rng.randint(4, 16), layers=rng.choice([2, 3, 4]),
                    vocab=_log(rng, 4096, 32768))
    if kind == "moe":
        return dict(kind=kind, tokens=_log(rng, 1, 2048), hidden=rng.choice([1024, 2048, 4096]),
                    ffn=rng.choice([512, 768, 1408]), experts=rng.choice([8, 32, 64, 128]), top_k=rng.choice([2, 4, 8]))
    if kind == "ref_ffn":
        dim = rng.choice([112, 224, 448, 896])
        return dict(kind=kind, rows=_log(rng, 1, 4096), dim=dim, hidden=4 * dim)
    if kind == "ref_prefill":
        return dict(kind=kind, tokens=_log(rng, 9, 300), layers=2, vocab=_log(rng, 1024, 8192))
    if kind == "ref_decode":
        return dict(kind=kind, pos=_log(rng, 16, 700), steps=rng.randint(4, 12), layers=2, vocab=_log(rng, 1024, 8192))
    if kind == "ref_moe":
        return dict(kind=kind, tokens=_log(rng, 1, 192), dim=rng.choice([512, 1024, 2048]),
                    hidden=rng.choice([512, 704, 1408]), experts=rng.choice([8, 16]), top_k=rng.choice([2, 4]))
    return dict(kind="backend", rows=_log(rng, 1, 512), out=_log(rng, 64, 4864), k=_log(rng, 64, 4864))


# -- inputs ----------------------------------------------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _codes(g, peak, *shape):
    """Normal i32 codes at a quarter of `peak`, clipped to it (device)."""
    return torch.randn(*shape, generator=g, device=DEV).mul_(peak / 4).round_().clamp_(-peak, peak).to(torch.int32)


def _rows8(g, m, k):
    """Int8 activations of m x k, sigma 40, zero padded to the device layout's row (device)."""
    x = torch.zeros(m, B.kp(k), dtype=torch.int8, device=DEV)
    x[:, :k] = torch.randn(m, k, generator=g, device=DEV).mul_(40).round_().clamp_(-127, 127).to(torch.int8)
    return x


def _scales(codes, sigma, target=127):
    """Per-channel (mant, shift) that map four standard deviations of a channel's accumulator, at an input of
    standard deviation sigma, to target."""
    dev = codes.double().square().sum(dim=1).sqrt().clamp(min=1.0) * (4.0 * sigma)
    mant, exp = torch.frexp(target / dev)  # target / dev = mant * 2^exp, mant in [0.5, 1)
    return (mant * (1 << 31)).round().clamp(max=(1 << 31) - 1).to(torch.int32), (31 - exp).to(torch.int32)


def _w12(codes, planes="w12"):
    n, k = codes.shape
    if planes == "w12b":
        lo = torch.empty(B.w12b_bytes(n, k), dtype=torch.int8, device=DEV)
        hi = torch.empty_like(lo)
        B.w12b_pack(codes, n, k, lo, hi)
        return lo, hi
    nlo, nnib = B.w12_bytes(n, k)
    lo = torch.empty(nlo, dtype=torch.int8, device=DEV)
    nib = torch.empty(nnib, dtype=torch.uint8, device=DEV)
    B.w12_pack(codes, n, k, lo, nib)
    return lo, nib


def _host(t):
    return t.cpu().numpy()


def _np(pair):
    return tuple(_host(t) for t in pair)


QWEN = dict(d=896, ffn=4864, nh=14, nkv=2, hd=64)


def _decoder(case, g, max_pos, max_rows):
    cfg = dict(QWEN, layers=case["layers"], vocab=case["vocab"])
    m = DecoderModel(cfg, max_pos, max_rows)
    d, ffn, nq, qd = m.d, m.ffn, m.nq, m.nh * m.hd
    for l in range(m.L):
        w = [_codes(g, 2047, *s) for s in ((nq, d), (d, qd), (2 * ffn, d), (d, ffn))]
        s = [_scales(c, sig, t) for c, (sig, t) in zip(w, (W.DEC_SCALES[n] for n in ("qkv", "o", "gu", "dn")))]
        m.set_layer(l, *[a for c, p in zip(w, s) for a in (_host(c), _np(p))])
    emb = _codes(g, 2047, m.V, d)
    sig, t = W.DEC_SCALES["lm"]
    m.set_embedding(_host(emb).reshape(-1), _np(_scales(emb, sig, t)))
    m.set_tables(*W.rope_tables(max_pos), W.exp_table(), W.silu_table())
    return m


REF = dict(dim=896, nh=14, nkv=2, hd=64, hidden=4864, eps=1e-6, theta=1.0e6)


def _ref_decoder(case, g, max_seq):
    cfg = dict(REF, layers=case["layers"], vocab=case["vocab"], max_seq=max_seq)
    sc = B.ref_scale_from_f64(1.0 / WLEVELS)
    d, qd, kvd, h, V = cfg["dim"], cfg["nh"] * cfg["hd"], cfg["nkv"] * cfg["hd"], cfg["hidden"], cfg["vocab"]
    shapes = dict(in_norm=(d,), post_norm=(d,), wq=(qd, d), wk=(kvd, d), wv=(kvd, d), wo=(d, qd), gate=(h, d),
                  up=(h, d), down=(d, h))
    c = lambda *s: (_host(_codes(g, WLEVELS, *s)), sc)  # noqa: E731
    layers = [{n: c(*s) for n, s in shapes.items()} for _ in range(cfg["layers"])]
    return RefDecoder(cfg, c(V, d), c(d), c(V, d), layers)


def _act(g, n):
    """n activation codes at the 2^28 level and their scale record."""
    m, s = B.ref_scale_from_f64(4.0 / ACT)
    return _codes(g, ACT, n), qscale_record(m, s)


def prepare(case, seed):
    g, kind = _gen(seed), case["kind"]
    st = dict(case)
    if kind == "w12":
        m, n, k = case["m"], case["n"], case["k"]
        w = _codes(g, 2047, n, k)
        st["x"], st["w"] = _rows8(g, m, k), _w12(w, case["planes"])
        st["mant"], st["shift"] = _scales(w, 40, TARGET[case["out"]])
        st["y"] = torch.empty(m, n, dtype={"i64": torch.int64, "i32": torch.int32, "i8": torch.int8}[case["out"]],
                              device=DEV)
    elif kind == "mlp":
        t, d, h = case["tokens"], case["dim"], case["hidden"]
        wi, wo = _codes(g, 2047, h, d), _codes(g, 2047, d, h)
        st["x"], st["wi"], st["wo"] = _rows8(g, t, d), _w12(wi), _w12(wo)
        st["si"], st["so"] = _scales(wi, 40), _scales(wo, 24)
        st["lut"] = torch.from_numpy(W.gelu_table()).to(DEV)
        st["h"] = torch.zeros(t, B.kp(h), dtype=torch.int8, device=DEV)
        st["y"] = torch.empty(t, d, dtype=torch.int8, device=DEV)
    elif kind == "dec_prefill":
        t = case["tokens"]
        st["model"] = _decoder(case, g, t, t)
        st["tok"] = torch.randint(0, case["vocab"], (t,), generator=g, device=DEV, dtype=torch.int32)
    elif kind == "dec_decode":
        p, s = case["prompt"], case["steps"]
        m = st["model"] = _decoder(case, g, p + s + 1, p)
        m.forward(torch.randint(0, case["vocab"], (p,), generator=g, device=DEV, dtype=torch.int32), p)
        st["from"] = (m.part.clone(), m.pos.clone(), m.step.clone())
        m.decode_step()
        torch.cuda.synchronize()
        st["graph"] = m.capture_decode_step()
    elif kind == "moe":
        t, H, F, E, K = (case[n] for n in ("tokens", "hidden", "ffn", "experts", "top_k"))
        m = st["model"] = MoeLayer(H, F, E, K, W.silu_table(), W.sigmoid_table(), 8, 13)
        for e in range(E + 1):  # as MoeLayer.set_expert lays an expert out, from codes that are on the device already
            gu, dn = _codes(g, 2047, 2 * F, H), _codes(g, 2047, H, F)
            a, b = e * m.gu_lo_bytes, (e + 1) * m.gu_lo_bytes
            B.w12_pack_gate_up(gu, F, H, m.gu_lo[a:b], m.gu_nib[a // 2:b // 2])
            a, b = e * m.d_lo_bytes, (e + 1) * m.d_lo_bytes
            B.w12_pack(dn, H, F, m.d_lo[a:b], m.d_nib[a // 2:b // 2])
            m.gu_mant[e * 2 * F:(e + 1) * 2 * F], m.gu_shift[e * 2 * F:(e + 1) * 2 * F] = _scales(gu, 40)
            m.d_mant[e * H:(e + 1) * H], m.d_shift[e * H:(e + 1) * H] = _scales(dn, 16)
        st["x"] = _rows8(g, t, H)
        st["logits"] = torch.randn(t, E, generator=g, device=DEV).mul_(1024).round_().to(torch.int32)
        st["y"] = torch.empty(t, H, dtype=torch.int8, device=DEV)
    elif kind == "ref_ffn":
        d, h = case["dim"], case["hidden"]
        sc = B.ref_scale_from_f64(1.0 / WLEVELS)

        def layer(o, i):
            return _host(_codes(g, WLEVELS, o, i)), sc, (_host(_codes(g, WLEVELS, o)).astype(np.int64), sc)

        st["model"] = RefFeedForward(d, h, layer(h, d), layer(d, h))
        st["x"], st["xs"] = _act(g, case["rows"] * d)
    elif kind == "ref_prefill":
        st["model"] = _ref_decoder(case, g, case["tokens"])
        st["tok"] = _host(torch.randint(0, case["vocab"], (case["tokens"],), generator=g, device=DEV,
                                        dtype=torch.int32))
    elif kind == "ref_decode":
        p, s = case["pos"], case["steps"]
        m = st["model"] = _ref_decoder(case, g, p + s + 1)
        prompt = torch.randint(0, case["vocab"], (p + 1,), generator=g, device=DEV, dtype=torch.int32)
        m.token.copy_(prompt[0:1])
        m.pos.zero_()
        m.step_launches()
        torch.cuda.synchronize()
        st["graph"] = m.capture_greedy_step()
        m.pos.zero_()
        for i in range(p):  # the prompt through decode_step, as the engine feeds it
            m.token.copy_(prompt[i:i + 1])
            st["graph"].replay()
        st["tok"], st["pos0"] = prompt[p:p + 1].clone(), m.pos.clone()
    elif kind == "ref_moe":
        d, h, E = case["dim"], case["hidden"], case["experts"]
        sc = B.ref_scale_from_f64(1.0 / WLEVELS)
        c = lambda *s: (_host(_codes(g, WLEVELS, *s)), sc)  # noqa: E731
        expert = lambda: {"gate": c(h, d), "up": c(h, d), "down": c(d, h)}  # noqa: E731
        bias = _host(torch.randn(E, generator=g, device=DEV).mul_(0.05 * (1 << 20)).round_().to(torch.int64))
        st["model"] = RefMoeLayer(d, c(E, d), [expert() for _ in range(E)], case["top_k"], True, sigmoid_bias=bias,
                                  shared=expert())
        st["x"], st["xs"] = _act(g, case["tokens"] * d)
    else:
        r, o, k = case["rows"], case["out"], case["k"]
        st["backend"] = T.HipBackend(0)
        st["weights"] = T.Weights(T.weight_id_fresh(), _host(_codes(g, WLEVELS, o * k)))
        st["x"] = _host(_codes(g, WLEVELS, r * k))
        st["backend"].linear_weights(st["x"], st["weights"], r, o, k)  # the weights are resident from here on
    return st


# -- one pass --------------------------------------------------------------------------------------------------------


def run(st):
    kind = st["kind"]
    if kind == "w12":
        f = B.w12b_linear if st["planes"] == "w12b" else B.w12_linear
        f(st["x"], *st["w"], st["m"], st["n"], st["k"], st["y"], OUT[st["out"]], st["mant"], st["shift"])
        return st["y"]
    if kind == "mlp":
        t, d, h = st["tokens"], st["dim"], st["hidden"]
        B.w12_linear_lut(st["x"], *st["wi"], t, h, d, st["h"], *st["si"], st["lut"])
        B.w12_linear(st["h"], *st["wo"], t, d, h, st["y"], B.OUT_I8, *st["so"])
        return st["h"], st["y"]
    if kind == "dec_prefill":
        m = st["model"]
        m.pos.zero_()
        m.forward(st["tok"], st["tokens"])
        return m.logits, m.r, m.kc, m.vc
    if kind == "dec_decode":
        m = st["model"]
        for t, v in zip((m.part, m.pos, m.step), st["from"]):
            t.copy_(v)
        for _ in range(st["steps"]):
            st["graph"].replay()
        return m.logits, m.token, m.kc, m.vc
    if kind == "moe":
        st["model"].forward(st["x"], st["logits"], st["tokens"], st["y"])
        return st["y"]
    if kind == "ref_ffn":
        return st["model"].forward_int(st["x"], st["xs"], st["rows"])
    if kind == "ref_prefill":
        return st["model"].forward(st["tok"])
    if kind == "ref_decode":
        m = st["model"]
        m.token.copy_(st["tok"])
        m.pos.copy_(st["pos0"])
        for _ in range(st["steps"]):
            st["graph"].replay()
        return m.buf["logits"], m.rec["logits"], m.token, m.kc, m.vc
    if kind == "ref_moe":
        return st["model"].forward(st["x"], st["xs"], st["tokens"])
    return st["backend"].linear_weights(st["x"], st["weights"], st["rows"], st["out"], st["k"])


# -- what a pass cannot do without -----------------------------------------------------------------------------------


def _layer_macs(c):
    q, kv = c["nh"] * c["hd"], c["nkv"] * c["hd"]
    d, f = c.get("d", c.get("dim")), c.get("ffn", c.get("hidden"))
    return (q + 2 * kv) * d + d * q + 3 * f * d, q, kv, d


def work(case):
    kind = case["kind"]
    if kind == "w12":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 1.5 * n * k + m * k + m * n * OUT_BYTES[case["out"]] + 8 * n, "flops": 2.0 * m * n * k}
    if kind == "mlp":
        t, d, h = case["tokens"], case["dim"], case["hidden"]
        return {"bytes": 3.0 * d * h + t * (2 * d + 2 * h), "flops": 4.0 * t * d * h}
    if kind in ("dec_prefill", "dec_decode"):
        macs, q, kv, d = _layer_macs(QWEN)
        L, V = case["layers"], case["vocab"]
        weights = 1.5 * (L * macs + V * d)
        if kind == "dec_prefill":
            t = case["tokens"]
            return {"bytes": weights + t * 2 * d + L * t * 2 * kv + 4 * V,
                    "flops": 2.0 * (t * L * macs + V * d) + L * 2.0 * t * t * q}
        s, p = case["steps"], case["prompt"]
        return {"bytes": s * (weights + L * 2 * kv * p + 4 * V), "flops": 2.0 * s * (L * (macs + 2 * p * q) + V * d)}
    if kind == "moe":
        t, H, F, E, K = (case[n] for n in ("tokens", "hidden", "ffn", "experts", "top_k"))
        hit = E * (1 - (1 - K / E) ** t) + 1  # experts that some token chose (as many as are expected), and the shared
        return {"bytes": 4.5 * hit * H * F + t * (2 * H + 4 * E), "flops": 6.0 * t * (K + 1) * H * F}
    if kind == "ref_ffn":
        r, d, h = case["rows"], case["dim"], case["hidden"]
        return {"bytes": 6.0 * d * h + 8.0 * r * d, "flops": 4.0 * r * d * h}
    if kind in ("ref_prefill", "ref_decode"):
        macs, q, kv, d = _layer_macs(REF)
        L, V = case["layers"], case["vocab"]
        weights = 3.0 * (L * macs + V * d)
        if kind == "ref_prefill":
            t = case["tokens"]
            return {"bytes": weights + 4 * t * (d + V), "flops": 2.0 * t * (L * (macs + t * q) + V * d)}
        s, p = case["steps"], case["pos"]
        return {"bytes": s * (weights + L * 8 * kv * p + 4 * V), "flops": 2.0 * s * (L * (macs + 2 * p * q) + V * d)}
    if kind == "ref_moe":
        t, d, h, E, K = (case[n] for n in ("tokens", "dim", "hidden", "experts", "top_k"))
        hit = E * (1 - (1 - K / E) ** t) + 1
        return {"bytes": 9.0 * hit * d * h + 3 * E * d + 8 * t * d, "flops": 2.0 * t * (3 * (K + 1) * d * h + E * d)}
    r, o, k = case["rows"], case["out"], case["k"]
    return {"bytes": 3.0 * o * k + 4 * r * k + 8 * r * o, "flops": 2.0 * r * o * k}


def tolerance(case):
    return "exact"  # every output is an integer that the semantics fix


# -- the same by plain torch, where a page of it says what the integers are ------------------------------------------


def _dot(x, w):
    """x . w^T of integers, exactly: sums below 2^53 in float64, on the host."""
    return torch.matmul(x.double().cpu(), w.double().cpu().t()).to(torch.int64)


def _requant(v, mant, shift, lim):
    """round(v mant / 2^shift), half away from zero, clamped to +-lim; the shifts here are positive."""
    m, s = mant.cpu().to(torch.int64), shift.cpu().to(torch.int64)
    a = (v.abs() * m + (torch.ones_like(s) << (s - 1))) >> s
    return (a.clamp(max=lim) * torch.sign(v)).clamp(min=-lim)


def exact(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind == "w12":
        m, n, k = case["m"], case["n"], case["k"]
        if m * n * k > 4e10:
            return None
        w = _codes(g, 2047, n, k)
        v = _dot(_rows8(g, m, k)[:, :k], w)
        if case["out"] == "i64":
            return v
        v = _requant(v, *_scales(w, 40, TARGET[case["out"]]), 127 if case["out"] == "i8" else (1 << 31) - 1)
        return v.to(torch.int8 if case["out"] == "i8" else torch.int32)
    if kind == "mlp":
        t, d, h = case["tokens"], case["dim"], case["hidden"]
        wi, wo = _codes(g, 2047, h, d), _codes(g, 2047, d, h)
        q = _requant(_dot(_rows8(g, t, d)[:, :d], wi), *_scales(wi, 40), 127)
        hid = torch.zeros(t, B.kp(h), dtype=torch.int8)
        hid[:, :h] = torch.from_numpy(W.gelu_table())[q + 127]
        return hid, _requant(_dot(hid[:, :h], wo), *_scales(wo, 24), 127).to(torch.int8)
    if kind == "backend":
        r, o, k = case["rows"], case["out"], case["k"]
        w = _codes(g, WLEVELS, o * k).view(o, k)
        return _dot(_codes(g, WLEVELS, r * k).view(r, k), w).reshape(-1)
    return None  # the dynamic Scales and the layers around them are defined by the engine's own integer steps
