"""The sequence forms of add, RMSNorm and SwiGLU (kt_hip_ref_*_seq) at the sizes where their grids change: rows that do
not fill a CTA of four, a row longer or shorter than a wave's stride, the last row count every CTA folds itself and
the first that takes the one-CTA fold, and tensors with fewer, as many and more values than the first pass has slots
for. Codes and records equal the oracle's; SwiGLU equals the one-CTA kernel, which its own tests hold to the oracle."""
import sys

import numpy as np
import pytest

from oracle import oracle as O
from test_scale_dev import scale_out, sd  # noqa: F401  (sd: the device's Scale arithmetic on the host)

pytestmark = pytest.mark.gpu


def rec(torch, sc):
    w = np.zeros(4, dtype=np.int64)
    w[0] = sc[0]
    w.view(np.int32)[2] = sc[1]
    return torch.from_numpy(w).cuda()


def rd(r):
    w = r.cpu().numpy()
    return int(w[0]), int(w.view(np.int32)[2])


def dev(torch, a):
    return torch.from_numpy(np.ascontiguousarray(a, dtype=np.int32).reshape(-1)).cuda()


def rand_scale(rng):
    return int(rng.integers(2**30, 2**31)), int(rng.integers(40, 62))


def ws(torch, rows):
    from tritify_amd import backend as B

    n = B.ref_seq_workspace(rows)
    return torch.full((n,), 0xA5, dtype=torch.uint8, device="cuda"), n  # its contents must not matter


@pytest.mark.parametrize("rows,dim", [(1, 1), (2, 63), (3, 65), (5, 512), (7, 513), (130, 896), (1024, 33),
                                      (1025, 33), (2500, 16)])
@pytest.mark.parametrize("mag", [1, 2**28, 2**31 - 1])
def test_rmsnorm_seq_edges(torch_dev, rows, dim, mag):
    torch = torch_dev
    from tritify_amd import backend as B

    print(f"case: rmsnorm_seq rows={rows} dim={dim} mag={mag}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(rows * 131 + dim)
    x = rng.integers(-mag, mag + 1, size=(rows, dim)).astype(np.int32)
    x[rows // 2] = 0  # a row whose factor is the eps alone: the largest, over rows that are all far below it
    if rows > 4:
        x[-1] = x[0]  # equal factors: the fold's later row
        x[1] = np.sign(x[1]) * (np.abs(x[1].astype(np.int64)) >> 9)
    g = rng.integers(-O.WLEVELS, O.WLEVELS + 1, size=dim).astype(np.int32)
    if mag == 2**31 - 1:
        x[0, 0], g[0] = -2**31, -2**31  # the largest product there is
    gs, eps = rand_scale(rng), B.ref_scale_from_f64(1e-6)
    w, n = ws(torch, rows)
    y, ys = torch.zeros(rows * dim, dtype=torch.int32, device="cuda"), rec(torch, (0, 0))
    for xs in (rand_scale(rng), (0, 0)):
        B.ref_rmsnorm_seq(dev(torch, x), rec(torch, xs), rows, dim, dev(torch, g), gs, eps, w, n, y, ys)
        yo, so = O.rd_rmsnorm(x.reshape(-1), rows, dim, xs, g, gs, eps)
        assert np.array_equal(y.cpu().numpy(), yo) and rd(ys) == so, xs


@pytest.mark.parametrize("n", [1, 255, 1024, 1025, 512 * 1024, 512 * 1024 + 3])
def test_add_and_swiglu_seq_edges(torch_dev, n):
    torch = torch_dev
    from tritify_amd import backend as B

    print(f"case: add_seq / swiglu_seq n={n}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(n)
    a = rng.integers(-(2**28), 2**28 + 1, size=n).astype(np.int32)
    b = rng.integers(-(2**28), 2**28 + 1, size=n).astype(np.int32)
    b[-1] = 2**28 + 7  # the largest value is the last one's
    w, nw = ws(torch, 1)
    for sa, sb in ((rand_scale(rng), rand_scale(rng)), (rand_scale(rng), (0, 0)), ((0, 0), (0, 0))):
        yo, so = O.rd_add(a, sa, b, sb)
        ad, ar = dev(torch, a), rec(torch, sa)
        B.ref_add_seq(ad, ar, dev(torch, b), rec(torch, sb), n, w, nw, ad, ar)  # in place, as the residual add
        assert np.array_equal(ad.cpu().numpy(), yo) and rd(ar) == so, (sa, sb)
    codes, lut = B.ref_codelut(B.LUT_SILU, -30.0, 30.0, 16, 20, True)
    cd = torch.from_numpy(codes).cuda()
    for gshift in (53, 60):
        gs, us = (int(rng.integers(2**30, 2**31)), gshift), rand_scale(rng)
        out = []
        for seq in (False, True):
            h, hs = torch.zeros(n, dtype=torch.int32, device="cuda"), rec(torch, (0, 0))
            args = (dev(torch, a), rec(torch, gs), dev(torch, b), rec(torch, us), n, cd, lut)
            B.ref_swiglu_seq(*args, w, nw, h, hs) if seq else B.ref_swiglu(*args, h, hs)
            out.append((h.cpu().numpy(), rd(hs)))
        assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1], gshift


@pytest.mark.parametrize("nh,nkv,hd,T", [(14, 2, 64, 2), (14, 2, 64, 5), (4, 4, 64, 64), (6, 2, 64, 67), (2, 1, 128, 131),
                                         (4, 2, 96, 66), (1, 1, 64, 300), (2, 1, 64, 2050)])
@pytest.mark.parametrize("mag", [2**20, 2**28])
def test_attention_prefill_edges(torch_dev, nh, nkv, hd, T, mag):
    """The prefill attention where its row groups, lane blocks and runs end: rows that do not fill a group of four,
    blocks of 64 cached rows with one more and one less, one row per CTA past 2048, each head dimension's kernel."""
    torch = torch_dev
    from tritify_amd import backend as B

    print(f"case: attention_prefill nh={nh} nkv={nkv} hd={hd} T={T} mag={mag}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(nh * 100 + T + hd)
    model = O.RefModel(3, dict(dim=nh * hd, layers=1, nh=nh, nkv=nkv, hd=hd, hidden=8, vocab=2, eps=1e-6, theta=10000.0,
                               max_seq=T))
    q, k, v = (rng.integers(-mag, mag + 1, size=T * n * hd).astype(np.int32) for n in (nh, nkv, nkv))
    v[:hd] = 0  # row 0 of the first head attends to zeros alone
    # score scales spread so the softmax is neither flat nor one-hot
    qs, ks, vs = (int(rng.integers(2**30, 2**31)), 81 if mag == 2**28 else 65), rand_scale(rng), rand_scale(rng)
    want, wsc = model.attention_prefill(T, q, qs, k, ks, v, vs)
    cos_t, sin_t = B.ref_rope_tables(T, hd, 10000.0)
    ec, lut = B.ref_codelut(B.LUT_EXP, -30.0, 0.0, 16, 20, False)
    n = B.ref_attention_prefill_workspace(T, nh, nkv, hd)
    w = torch.full((n,), 0xA5, dtype=torch.uint8, device="cuda")
    o, os_ = torch.zeros(T * nh * hd, dtype=torch.int32, device="cuda"), rec(torch, (0, 0))
    B.ref_attention_prefill(dev(torch, q), rec(torch, qs), dev(torch, k), rec(torch, ks), dev(torch, v), rec(torch, vs),
                            T, nh, nkv, hd, T, torch.from_numpy(cos_t.view(np.uint8)).cuda(),
                            torch.from_numpy(sin_t.view(np.uint8)).cuda(), B.ref_scale_from_f64(1.0 / np.sqrt(hd)),
                            torch.from_numpy(ec).cuda(), lut, w, n, o, os_)
    assert np.array_equal(o.cpu().numpy(), want) and rd(os_) == wsc


@pytest.mark.parametrize("hd", [64, 96, 128])
def test_attention_prefill_sums_at_the_i64_limit(torch_dev, sd, hd):  # noqa: F811
    """A table of numerators 2^32 and v codes of -2^31: (row, head)s whose sums reach -2^63, alone and beside the largest
    scale, where |sum| wraps. Against the engine's steps in Python on the host's Scales."""
    torch = torch_dev
    from tritify_amd import backend as B

    print(f"case: attention_prefill i64 limit hd={hd}", file=sys.stderr, flush=True)
    T, nh, num, act = 3, 2, 1 << 32, 1 << 28
    rng = np.random.default_rng(hd)
    for spread in (0, 2**20, 2**31 - 1):
        v = rng.integers(-spread, spread + 1, size=(T, nh, hd)).astype(np.int64)
        v[:, 0, 3] = -(2**31), 0, 0  # sums of -2^63 in every row, at factors 1, 1/2 and 1/3
        vs = (1509949440, 58)
        zero = torch.zeros(T * nh * hd, dtype=torch.int32, device="cuda")
        cos_t, sin_t = B.ref_rope_tables(T, hd, 10000.0)
        ec, lut = B.ref_codelut(B.LUT_EXP, -30.0, 0.0, 16, 20, False)
        n = B.ref_attention_prefill_workspace(T, nh, nh, hd)
        w = torch.full((n,), 0xA5, dtype=torch.uint8, device="cuda")
        o, os_ = torch.zeros(T * nh * hd, dtype=torch.int32, device="cuda"), rec(torch, (0, 0))
        one = rec(torch, (2**30, 60))
        B.ref_attention_prefill(zero, one, zero, one, dev(torch, v), rec(torch, vs), T, nh, nh, hd, T,
                                torch.from_numpy(cos_t.view(np.uint8)).cuda(),
                                torch.from_numpy(sin_t.view(np.uint8)).cuda(), B.ref_scale_from_f64(1.0 / np.sqrt(hd)),
                                torch.full((len(ec),), num, dtype=torch.int64, device="cuda"), lut, w, n, o, os_)
        wrap = lambda x: (int(x) + 2**63) % 2**64 - 2**63  # noqa: E731
        ratio = lambda a, b: scale_out(sd.sd_from_ratio, 0, a, 0, b)  # noqa: E731
        sums = np.array([[[wrap(sum(num * int(v[j, h, d]) for j in range(i + 1))) for d in range(hd)] for h in range(nh)]
                         for i in range(T)], dtype=np.int64)
        sc = [scale_out(sd.sd_mul, *vs, *ratio(1, (i + 1) * num)) for i in range(T)]
        cinv = scale_out(sd.sd_recip, *sc[0])  # the largest: one numerator
        at = [[[sd.sd_apply(*scale_out(sd.sd_mul, *sc[i], *cinv), int(x)) for x in sums[i, h]] for h in range(nh)]
              for i in range(T)]
        gmax = max(0, max(wrap(abs(x)) for r in at for h in r for x in h))
        want = [sd.sd_rq_apply(gmax, x) if gmax else 0 for r in at for h in r for x in h]
        assert sums[0, 0, 3] == sums[1, 0, 3] == -(2**63)
        assert o.cpu().numpy().tolist() == want, spread
        assert rd(os_) == (scale_out(sd.sd_mul, *ratio(gmax, act), *sc[0]) if gmax else (0, 0)), spread
