"""kt_hip_ref_moe_experts against the general path it stands for -- kt_hip_quant_linear_rows for gate and for up,
kt_hip_ref_swiglu of the rows, kt_hip_quant_linear_rows for down, each checked against the oracle in
test_gpu_refmoe.py -- codes and records byte for byte over the forms that path accepts: rows by index or in place, one
input record or one per row, every plane count, empty groups, zero rows and zero weight Scales, widths around the
tiles, the threads' spans and the widest row."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LIM = {1: 127, 3: 265720, 5: 2**30}


def say(*a):
    print(*a, file=sys.stderr, flush=True)


def test_workspace_refuses_what_the_row_kernel_does_not_hold(torch_dev):
    from tritify_amd import backend as B

    assert B.ref_moe_experts_workspace(1, 64, 4096, 1) > 0 and B.ref_moe_experts_workspace(1, 64, 4097, 1) == 0


@pytest.mark.parametrize("counts,dim,hidden,pgu,pd,by_index,step", [
    ([1], 64, 1, 3, 3, False, 0),
    ([3, 0, 5, 1], 200, 65, 3, 1, True, 0),
    ([0, 33, 2], 128, 64, 1, 3, True, 1),
    ([7, 0, 32, 1, 40], 300, 1023, 3, 3, True, 0),
    ([2, 2], 65, 1024, 3, 5, False, 1),
    ([4, 1], 2100, 1025, 5, 3, True, 0),
    ([1, 6], 96, 4096, 3, 3, False, 0),
])
def test_experts_equal_the_products_and_the_swiglu(torch_dev, counts, dim, hidden, pgu, pd, by_index, step):
    torch = torch_dev
    from tritify_amd import backend as B

    say(f"case: moe experts counts={counts} dim={dim} hidden={hidden} planes {pgu}/{pd}")
    rng = np.random.default_rng(dim + hidden)
    G, P = len(counts), sum(counts)
    x_rows = 9 if by_index else P
    dev = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    x = rng.integers(-(2**28), 2**28 + 1, size=(x_rows, dim)).astype(np.int32)
    x[x_rows // 2] = 0
    if x_rows > 3:
        x[1] >>= 20  # a row of few levels
    xidx = rng.integers(0, x_rows, size=P).astype(np.int32)
    xidx[P // 3] = x_rows if P > 1 else 0  # outside x: a zero row
    rec = np.zeros((P, 4), dtype=np.int64)
    rec[:, 0] = rng.integers(2**30, 2**31, size=P)
    rec.view(np.int32)[:, 2] = rng.integers(53, 58, size=P)  # products around SiLU's table: inside, below and above
    scale = lambda: (rng.integers(2**30, 2**31, size=G).astype(np.int64),  # noqa: E731
                     rng.integers(44, 52, size=G).astype(np.int32))
    (gm, gs), (um, us), (dm, ds) = scale(), scale(), scale()
    if G > 2:
        um[G - 1], us[G - 1] = 0, 0  # up at Scale::ZERO: zero rows
    w = {n: rng.integers(-LIM[p], LIM[p] + 1, size=(G, o, i)).astype(np.int32)
         for n, p, o, i in (("gate", pgu, hidden, dim), ("up", pgu, hidden, dim), ("down", pd, dim, hidden))}
    w["gu"] = np.concatenate([w["gate"], w["up"]], axis=1)
    planes = {}
    for n, p in (("gate", pgu), ("up", pgu), ("gu", pgu), ("down", pd)):
        _, o, i = w[n].shape
        gb = B.pack_planes_tiled_bytes(o, i, p)
        buf = torch.empty(G * gb, dtype=torch.int8, device="cuda")
        for g in range(G):
            B.pack_planes_tiled(dev(w[n][g].reshape(-1)), o, i, p, buf[g * gb:])
        planes[n] = (buf, gb)
    off = dev(np.concatenate([[0], np.cumsum(counts)]).astype(np.int64))
    xd, xi, xr = dev(x.reshape(-1)), dev(xidx) if by_index else None, dev(rec.reshape(-1))
    sc = {n: (dev(m), dev(s)) for n, m, s in (("gate", gm, gs), ("up", um, us), ("down", dm, ds))}
    codes, lut = B.ref_codelut(B.LUT_SILU, -30.0, 30.0, 16, 20, True)
    codes = dev(np.asarray(codes, np.int64))

    def rows_ql(n, p, src, idx, rows_in, rr, st):
        _, o, i = w[n].shape
        nb = B.quant_linear_rows_workspace(P, i, o, G)
        ws = torch.empty(nb, dtype=torch.uint8, device="cuda")
        y = torch.empty(P * o, dtype=torch.int32, device="cuda")
        ys = torch.empty(P * 4, dtype=torch.int64, device="cuda")
        B.quant_linear_rows(src, idx, rows_in, P, i, rr, st, None, off, *planes[n], p, o, *sc[n], ws, nb, y, ys,
                            groups=G)
        return y, ys

    g, grec = rows_ql("gate", pgu, xd, xi, x_rows, xr, step)
    u, urec = rows_ql("up", pgu, xd, xi, x_rows, xr, step)
    h = torch.empty(P * hidden, dtype=torch.int32, device="cuda")
    hr = torch.empty(P * 4, dtype=torch.int64, device="cuda")
    B.ref_swiglu(g, grec, u, urec, hidden, codes, lut, h, hr, rows=P)
    want, wrec = rows_ql("down", pd, h, None, P, hr, 1)

    ptr = lambda t: t.data_ptr()  # noqa: E731
    mw = B.MoeWeights(ptr(planes["gu"][0]), ptr(planes["down"][0]), planes["gu"][1], planes["down"][1],
                      *(ptr(sc[n][0]) for n in ("gate", "up", "down")),
                      *(ptr(sc[n][1]) for n in ("gate", "up", "down")), pgu, pd)
    nb = B.ref_moe_experts_workspace(P, dim, hidden, G)
    ws = torch.full((nb,), 0x5A, dtype=torch.uint8, device="cuda")  # nothing in it is read before it is written
    y = torch.empty(P * dim, dtype=torch.int32, device="cuda")
    yr = torch.empty(P * 4, dtype=torch.int64, device="cuda")
    B.ref_moe_experts(xd, xi, x_rows, P, dim, hidden, xr, step, G, off, mw, codes, lut, ws, nb, y, yr)
    assert np.array_equal(y.cpu().numpy(), want.cpu().numpy())
    assert np.array_equal(yr.cpu().numpy(), wrec.cpu().numpy())
    if P > 2:
        assert want.any()
