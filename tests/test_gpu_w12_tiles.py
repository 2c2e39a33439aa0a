"""The W12 products where the choice of their tiles changes: the LDS-staged kernel past 128 rows at one CTA per CU and
one more, 256-row tiles that fill their last round and that do not, row lengths that are not multiples of 16 (16-byte
stores at odd addresses), and the dense SwiGLU product on each of its tiles. Against float64 products (exact: sums below
2^53) and the requant in Python's integers."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def inputs(torch, m, n, k, seed):
    import tritify_amd as T

    rng = np.random.default_rng(seed)
    x = rng.integers(-128, 128, size=(m, k)).astype(np.int8)
    w = rng.integers(-2048, 2048, size=(n, k)).astype(np.int32)
    mant = rng.integers(-(2**31), 2**31, size=n).astype(np.int32)
    shift = rng.integers(38, 50, size=n).astype(np.int32)
    kp = T.kp(k)
    xp = np.zeros((m, kp), np.int8)
    xp[:, :k] = x
    return x, w, mant, shift, torch.from_numpy(xp).cuda(), torch.from_numpy(w).cuda()


def pack(torch, wd, n, k, f=None):
    import tritify_amd as T

    nlo, nnib = T.w12_bytes(n, k)
    lo = torch.empty(nlo, dtype=torch.int8, device="cuda")
    nib = torch.empty(nnib, dtype=torch.uint8, device="cuda")
    T.w12_pack(wd, n, k, lo, nib) if f is None else T.w12_pack_gate_up(wd, f, k, lo, nib)
    return lo, nib


def dot(x, w):
    return (x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.int64)


def requant(v, mant, shift, lo, hi):
    """round(v mant / 2^shift), half away from zero, clamped (|v mant| < 2^62, shifts positive)."""
    p = v * mant.astype(np.int64)[None, :]
    q = (np.abs(p) + (np.int64(1) << (shift.astype(np.int64) - 1))) >> shift.astype(np.int64)
    return np.clip(np.sign(p) * q, lo, hi)


@pytest.mark.parametrize("m,n,k", [(129, 1000, 70), (200, 897, 320), (512, 1024, 64), (512, 1025, 64), (513, 1024, 64),
                                   (300, 333, 130), (2048, 2049, 64), (2048, 6001, 64), (4096, 4096, 64), (4000, 111, 64),
                                   (1111, 3000, 192)])
@pytest.mark.parametrize("kind", ["i64", "i32", "i8", "add"])
def test_dense(torch_dev, m, n, k, kind):
    torch = torch_dev
    import tritify_amd as T

    print(f"case: w12 tiles m={m} n={n} k={k} {kind}", file=sys.stderr, flush=True)
    x, w, mant, shift, xd, wd = inputs(torch, m, n, k, m + n + k)
    lo, nib = pack(torch, wd, n, k)
    v = dot(x, w)
    out, dt, lim = {"i64": (T.OUT_I64, np.int64, None), "i32": (T.OUT_I32, np.int32, (-2**31, 2**31 - 1)),
                    "i8": (T.OUT_I8, np.int8, (-127, 127)), "add": (T.OUT_I32_ADD, np.int32, (-2**31, 2**31 - 1))}[kind]
    want = v if lim is None else requant(v, mant, shift, *lim)
    pad = 32
    base = np.full(m * n + 2 * pad, 5, dt)
    if kind == "add":
        base[pad:-pad] = np.random.default_rng(1).integers(-2**31, 2**31, size=m * n).astype(dt)
        want = np.clip(base[pad:-pad].reshape(m, n).astype(np.int64) + want, -2**31, 2**31 - 1)
    y = torch.from_numpy(base.copy()).cuda()
    T.w12_linear(xd, lo, nib, m, n, k, y[pad:], out, torch.from_numpy(mant).cuda(), torch.from_numpy(shift).cuda())
    got = y.cpu().numpy()
    assert (got[:pad] == 5).all() and (got[-pad:] == 5).all()
    assert np.array_equal(got[pad:-pad].reshape(m, n), want.astype(dt))


@pytest.mark.parametrize("m,f,k", [(130, 64, 70), (150, 1024, 64), (300, 2432, 64), (600, 4864, 64), (1025, 1408, 128),
                                   (1500, 2048, 64)])
def test_dense_swiglu(torch_dev, m, f, k):
    torch = torch_dev
    import tritify_amd as T
    from tritify_amd import workloads as W

    print(f"case: w12 swiglu tiles m={m} f={f} k={k}", file=sys.stderr, flush=True)
    x, w, mant, shift, xd, wd = inputs(torch, m, 2 * f, k, m + f + k)
    lo, nib = pack(torch, wd, 2 * f, k, f)
    silu = W.silu_table()
    q = requant(dot(x, w), mant, shift, -127, 127)
    p = silu.astype(np.int64)[q[:, :f] + 127] * q[:, f:]
    want = np.clip(np.sign(p) * ((np.abs(p) + 128) >> 8), -127, 127)
    y = torch.full((m * f + 64,), 99, dtype=torch.int8, device="cuda")
    T.w12_swiglu(xd, lo, nib, m, f, k, torch.from_numpy(mant).cuda(), torch.from_numpy(shift).cuda(),
                 torch.from_numpy(silu).cuda(), 8, y, f)
    got = y.cpu().numpy()
    assert (got[m * f:] == 99).all()
    assert np.array_equal(got[:m * f].reshape(m, f), want.astype(np.int8))


# 64-row tiles in one round and in three (more tiles than CTAs), 128-row tiles, 256-row tiles
@pytest.mark.parametrize("m,n,k", [(300, 1000, 70), (1500, 4096, 64), (2600, 4096, 64), (4096, 4096, 64)])
def test_one_group_i8(torch_dev, m, n, k):
    """The grouped product of one group with the int8 epilogue on each of its tiles."""
    torch = torch_dev
    import tritify_amd as T
    from tritify_amd import backend as B

    print(f"case: w12 one group m={m} n={n} k={k}", file=sys.stderr, flush=True)
    x, w, mant, shift, xd, wd = inputs(torch, m, n, k, m + n + k)
    lo, nib = pack(torch, wd, n, k)
    y = torch.full((m * n + 64,), 99, dtype=torch.int8, device="cuda")
    B.w12_grouped_linear(xd, m, None, 0, None, 1, m, lo, nib, n, k, torch.from_numpy(mant).cuda(),
                         torch.from_numpy(shift).cuda(), B.EPI_I8, y, n)
    got = y.cpu().numpy()
    assert (got[m * n:] == 99).all()
    assert np.array_equal(got[:m * n].reshape(m, n), requant(dot(x, w), mant, shift, -127, 127).astype(np.int8))
