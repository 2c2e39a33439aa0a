"""The promise a projection relies on when its input is declared closed (KT_QL_X_CLOSED): the whole output of RMSNorm,
SwiGLU, add and the prefill attention has a largest |code| of exactly 2^28, or is all zeros at Scale::ZERO. Each op over
ordinary, tiny, single-valued and zero inputs and zero scales, and every declared input of a decoder's forward and of an
expert layer's shared expert as it reaches its projection."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

ONE = 1 << 28


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def rec(torch, sc):
    w = np.zeros(4, dtype=np.int64)
    w[0] = sc[0]
    w.view(np.int32)[2] = sc[1]
    return torch.from_numpy(w).cuda()


def closed(codes, record):
    c, mant = codes.cpu().numpy().astype(np.int64), int(record.cpu().numpy()[0])
    return int(np.abs(c).max()) == (ONE if mant != 0 else 0)


def inputs(rng, n):
    """Codes of each kind, as (name, codes)."""
    one = np.zeros(n, np.int32)
    one[n // 2] = -3
    return [("ordinary", rng.integers(-ONE, ONE + 1, size=n).astype(np.int32)), ("tiny", rng.integers(-2, 3, size=n)),
            ("one value", one), ("largest", np.full(n, -(2**31))), ("zeros", np.zeros(n))]


@pytest.mark.parametrize("op", ["norm", "add", "swiglu", "attention"])
@pytest.mark.parametrize("scale", [(1509949440, 58), (2**31 - 1, 90), (2**30, 20), (0, 0)])
def test_ops_close(torch_dev, op, scale):
    torch = torch_dev
    from tritify_amd import backend as B

    rng = np.random.default_rng(scale[1])
    rows, dim = 5, 128  # the attention: 2 heads of 64
    n = rows * dim
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32)).cuda()  # noqa: E731
    nws = max(B.ref_seq_workspace(rows), B.ref_attention_prefill_workspace(rows, 2, 2, 64))
    ws = torch.empty(nws, dtype=torch.uint8, device="cuda")
    other = (1318646415, 57)
    silu, slut = B.ref_codelut(B.LUT_SILU, -30.0, 30.0, 16, 20, True)
    exp, elut = B.ref_codelut(B.LUT_EXP, -30.0, 0.0, 16, 20, False)
    cos, sin = B.ref_rope_tables(rows, 64, 10000.0)
    tab = lambda a: torch.from_numpy(a.view(np.uint8) if a.dtype != np.int64 else a).cuda()  # noqa: E731
    silu, exp = torch.from_numpy(silu).cuda(), torch.from_numpy(exp).cuda()
    for name, a in inputs(rng, n):
        for second, b in inputs(rng, n):
            say(f"case: {op} scale={scale} {name} / {second}")
            y, ys = torch.full((n,), 7, dtype=torch.int32, device="cuda"), torch.full((4,), -1, dtype=torch.int64,
                                                                                    device="cuda")
            ar, br = rec(torch, scale), rec(torch, other)
            if op == "norm":
                B.ref_rmsnorm_seq(dev(a), ar, rows, dim, dev(b[:dim]), other, B.ref_scale_from_f64(1e-6), ws, nws, y, ys)
            elif op == "add":
                B.ref_add_seq(dev(a), ar, dev(b), br, n, ws, nws, y, ys)
            elif op == "swiglu":  # up's codes are zeros where its scale is
                u = b if scale[0] else np.zeros(n)
                B.ref_swiglu_seq(dev(a), br, dev(u), ar, n, silu, slut, ws, nws, y, ys)
            else:
                B.ref_attention_prefill(dev(a), br, dev(a), br, dev(b), ar, rows, 2, 2, 64, rows, tab(cos), tab(sin),
                                        B.ref_scale_from_f64(0.125), exp, elut, ws, nws, y, ys)
            assert closed(y, ys), (name, second)


def declared(torch, monkeypatch):
    """Every input that reaches a projection as closed from here on: whether it is."""
    from tritify_amd import backend as B

    seen, plain = [], B.quant_linear_multi

    def checked(x, rows, inp, xs, *args, x_kind=B.X_ANY, **kw):
        if x_kind == B.X_CLOSED:
            seen.append(closed(x[:rows * inp], xs))
        return plain(x, rows, inp, xs, *args, x_kind=x_kind, **kw)

    monkeypatch.setattr(B, "quant_linear_multi", checked)
    return seen


@pytest.mark.parametrize("nkv,grouped", [(2, True), (1, False)])
@pytest.mark.parametrize("zero", ["", "in_norm", "wv", "up"])
def test_a_decoders_projections(torch_dev, monkeypatch, nkv, grouped, zero):
    """zero: a norm's gains, or a projection, that are all zero, so that what follows is zeros at Scale::ZERO."""
    torch = torch_dev
    from tritify_amd import backend as B
    from tritify_amd.refdecoder import RefDecoder

    say(f"case: decoder closed nkv={nkv} zero={zero}")
    rng = np.random.default_rng(nkv)
    dim, hid, V, L, T = 128, 256, 50, 2, 9
    sc = B.ref_scale_from_f64(1.0 / O.WLEVELS)
    c = lambda *s: (rng.integers(-O.WLEVELS, O.WLEVELS + 1, size=s).astype(np.int32), sc)  # noqa: E731
    shapes = dict(in_norm=(dim,), post_norm=(dim,), wq=(128, dim), wk=(64 * nkv, dim), wv=(64 * nkv, dim), wo=(dim, 128),
                  gate=(hid, dim), up=(hid, dim), down=(dim, hid))
    layers = [{n: c(*s) for n, s in shapes.items()} for _ in range(L)]
    if zero:
        layers[0][zero] = (np.zeros_like(layers[0][zero][0]), sc)
    m = RefDecoder(dict(dim=dim, nh=2, nkv=nkv, hd=64, hidden=hid, layers=L, vocab=V, max_seq=16, eps=1e-6, theta=1e4),
                   c(V, dim), c(dim), c(V, dim), layers)
    assert m.grouped == grouped
    seen = declared(torch, monkeypatch)
    m.forward(rng.integers(0, V, size=T).astype(np.int32))
    assert len(seen) == L * (4 if grouped else 7) + 1 and all(seen)


def test_a_shared_experts_down(torch_dev, monkeypatch):
    torch = torch_dev
    from tritify_amd import backend as B
    from tritify_amd.refmoe import RefMoeLayer

    say("case: shared expert closed")
    rng = np.random.default_rng(3)
    d, h, E, T = 64, 128, 4, 5
    sc = B.ref_scale_from_f64(1.0 / O.WLEVELS)
    c = lambda *s: (rng.integers(-O.WLEVELS, O.WLEVELS + 1, size=s).astype(np.int32), sc)  # noqa: E731
    expert = lambda: {"gate": c(h, d), "up": c(h, d), "down": c(d, h)}  # noqa: E731
    layer = RefMoeLayer(d, c(E, d), [expert() for _ in range(E)], 2, True, shared=expert())
    seen = declared(torch, monkeypatch)
    x = torch.from_numpy(rng.integers(-ONE, ONE + 1, size=T * d).astype(np.int32)).cuda()
    layer.forward(x, rec(torch, (1509949440, 58)), T)
    assert seen == [True]
