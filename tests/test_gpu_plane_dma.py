"""The DMA-fed 3 x 3 digit-plane product at the sizes where its tiles, rings and splits change: a row or column more and
less than each tile, k of one to a few k-tiles (fewer than the ring's stages), tiles past the matrix, k past the int32
bound (a second launch that adds), and QuantLinear over split k with a bias and over segments. The product's sums are
compared with float64 matrix products of the codes, exact below 2^53; the layer with the oracle."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

WLEVELS = 265720
LO3, HI3 = -128 * (1 + 256 + 65536), 127 * (1 + 256 + 65536)  # the range of three balanced base-256 digits


def gemm(torch, x, w, k):
    import tritify_amd as T

    kp = T.kp(k)
    planes = []
    for a in (x, w):
        d = torch.from_numpy(a).cuda()
        p = torch.empty(3 * a.shape[0] * kp, dtype=torch.int8, device="cuda")
        T.pack_planes(d, a.shape[0], k, 3, p)
        planes.append(p)
    m, n = x.shape[0], w.shape[0]
    guard = 64  # values on both sides of y that must stay as they are
    y = torch.full((m * n + 2 * guard,), -77, dtype=torch.int64, device="cuda")
    T.digit_gemm(planes[0], 3, planes[1], 3, y[guard:], m, n, k)
    torch.cuda.synchronize()
    y = y.cpu().numpy()
    assert (y[:guard] == -77).all() and (y[-guard:] == -77).all()
    return y[guard:-guard].reshape(m, n)


# 32 x 64 tiles, 64 x 64 tiles, 64 x 128 tiles
@pytest.mark.parametrize("m,n", [(5, 1), (31, 63), (32, 64), (33, 65), (255, 500), (513, 900), (1000, 961),
                                 (2049, 2049), (2048, 2113), (65536, 64), (16385, 112)])
@pytest.mark.parametrize("k", [1, 65, 250])
def test_tiles(torch_dev, m, n, k):
    if m * n * k > 10**9:
        k = 64
    print(f"case: plane dma m={m} n={n} k={k}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(m * 7 + n + k)
    x = rng.integers(-WLEVELS, WLEVELS + 1, size=(m, k)).astype(np.int32)
    w = rng.integers(-WLEVELS, WLEVELS + 1, size=(n, k)).astype(np.int32)
    got = gemm(torch_dev, x, w, k)
    assert np.array_equal(got, (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int64))


@pytest.mark.parametrize("m,n,k", [(40, 70, 512), (300, 800, 320), (2049, 2049, 64), (5, 70, 50000)])
def test_largest_sums(torch_dev, m, n, k):
    """Every digit at -128 or 127: the largest plane sums of each sign; k = 50000 takes two launches."""
    print(f"case: plane dma extremes m={m} n={n} k={k}", file=sys.stderr, flush=True)
    x = np.where(np.arange(m)[:, None] % 2, HI3, LO3) * np.ones((1, k), np.int64)
    w = np.where(np.arange(n)[:, None] % 3, LO3, HI3) * np.ones((1, k), np.int64)
    got = gemm(torch_dev, x.astype(np.int32), w.astype(np.int32), k)
    assert np.array_equal(got, x[:, :1] * w[:, 0][None, :] * k)


@pytest.mark.parametrize("rows,inp,out,bias", [(27, 3584, 900, True), (256, 2000, 300, False), (5, 700, 130, True),
                                               (5, 1300, 130, True), (70, 1100, 512, True), (1030, 100, 1030, True),
                                               (2100, 70, 2100, True)])
def test_quant_linear(torch_dev, rows, inp, out, bias):
    """The layer on each tile class, k split over CTAs from 1100 on."""
    from test_gpu_quant import run

    rng = np.random.default_rng(rows + inp + out)
    x = rng.integers(-(2**27), 2**27, size=rows * inp).astype(np.int32)
    w = rng.integers(-WLEVELS, WLEVELS + 1, size=out * inp).astype(np.int32)
    b = rng.integers(-(2**28), 2**28, size=out).astype(np.int64) if bias else None
    run(torch_dev, x, rows, inp, (1509949440, 58), w, out, (1657624235, 49), b, (1318646415, 57))


@pytest.mark.parametrize("rows,outs", [(37, (128, 256, 70)), (1100, (640, 384)), (1100, (576, 512)), (300, (64, 448))])
def test_segments(torch_dev, rows, outs):
    """Several calls on one x: boundaries at multiples of 128 and of 64 alone (no 128-column tile), each call's codes
    and record equal to its own QuantLinear's."""
    torch = torch_dev
    import tritify_amd as T
    from tritify_amd import backend as B

    print(f"case: plane dma segments rows={rows} outs={outs}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(rows + outs[0])
    inp, total, at = 130, sum(outs), 0
    x = torch.from_numpy(rng.integers(-(2**27), 2**27, size=rows * inp).astype(np.int32)).cuda()
    xs = T.qscale_record(1509949440, 58)
    ws = [(1657624235 + 7 * i, 49 + i) for i in range(len(outs))]
    w = rng.integers(-WLEVELS, WLEVELS + 1, size=(total, inp)).astype(np.int32)
    bias = rng.integers(-(2**28), 2**28, size=total).astype(np.int64)
    bs = [(1318646415, 57)] * len(outs)
    planes = torch.empty(3 * total * T.kp(inp), dtype=torch.int8, device="cuda")
    T.pack_planes(torch.from_numpy(w).cuda(), total, inp, 3, planes)
    n, _ = B.quant_linear_workspace(rows, inp, total)
    wsp = torch.full((n,), 0x5A, dtype=torch.uint8, device="cuda")
    ys = [torch.empty(rows * o, dtype=torch.int32, device="cuda") for o in outs]
    rec = torch.empty(4 * len(outs), dtype=torch.int64, device="cuda")
    B.quant_linear_multi(x, rows, inp, xs, outs, planes, 3, ws, torch.from_numpy(bias).cuda(), bs, wsp, n, ys, rec)
    for g, o in enumerate(outs):
        q = T.QuantLinear("t", w[at:at + o], o, inp, ws[g], (bias[at:at + o], bs[g]))
        y, r = q.forward_int(x, xs, rows)
        assert torch.equal(y, ys[g]) and torch.equal(r, rec[4 * g:4 * g + 4]), g
        at += o
