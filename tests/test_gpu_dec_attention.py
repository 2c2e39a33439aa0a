"""The int8 decoder's prefill attention where its kernels and tiles end: one row, the last row count of the short kernel
and the first of the tiled one, a row more and less than a tile of 32, positions that do not fill a block, a cache with
earlier positions, more blocks than waves, scores whose weights fall past the table, and tables whose entries reach and
pass the three digits the products take. Against the oracle per row and head."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,pos,nh,nkv,max_pos", [(1, 0, 4, 2, 8), (40, 1000, 2, 2, 1040), (127, 0, 4, 2, 127),
                                                  (128, 0, 4, 2, 128), (129, 30, 14, 2, 160), (159, 1, 4, 4, 160),
                                                  (160, 600, 7, 1, 760), (300, 0, 4, 2, 300)])
@pytest.mark.parametrize("table", ["exp", "edge", "wide"])
@pytest.mark.parametrize("flat", [False, True])
def test_prefill_attention(torch_dev, T, pos, nh, nkv, max_pos, table, flat):
    torch = torch_dev
    from tritify_amd import backend as B
    from tritify_amd import workloads as W

    print(f"case: dec attention T={T} pos={pos} nh={nh} nkv={nkv} table={table} flat={flat}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(T * 31 + pos + nh)
    hd, nq = 64, (nh + 2 * nkv) * 64
    span = 12 if flat else 128  # flat: every weight counts; else most fall past the table
    qkv = rng.integers(-span, span, size=(T, nq)).astype(np.int8)
    kc = rng.integers(-span, span, size=(max_pos, nkv, hd)).astype(np.int8)
    vc = rng.integers(-128, 128, size=(max_pos, nkv, hd)).astype(np.int8)
    exp = W.exp_table().astype(np.int32)
    if table == "edge":
        exp[:3] = (1 << 20) - 1, (1 << 14) - 1, 1 << 14
    elif table == "wide":
        exp[0], exp[1] = 1 << 20, (1 << 23) + 12345
    o = torch.full((T * nh * hd + 64,), 99, dtype=torch.int8, device="cuda")
    d = [torch.from_numpy(a.reshape(-1)).cuda() for a in (qkv, kc, vc, exp)]
    p = torch.tensor([pos], dtype=torch.int32, device="cuda")
    B.check(B.lib().kt_hip_dec_attention(0, d[0].data_ptr(), T, nq, p.data_ptr(), d[1].data_ptr(), d[2].data_ptr(), nh,
                                         nkv, hd, d[3].data_ptr(), o.data_ptr(), max_pos, 0), "dec attention")
    got = o.cpu().numpy()
    assert (got[T * nh * hd:] == 99).all()
    got = got[:T * nh * hd].reshape(T, nh, hd)
    for t in sorted({0, 1, T // 2, T - 2, T - 1} & set(range(T))):
        for h in range(nh):
            want = O.dec_attend(qkv[t, h * hd:(h + 1) * hd], kc.reshape(-1), vc.reshape(-1), pos + t, nkv, h // (nh // nkv),
                                hd, exp)
            assert np.array_equal(got[t, h], want), (t, h)


@pytest.mark.parametrize("T,pos,max_pos", [(100, -40, 30), (200, -40, 120), (130, -200, 64), (128, 300, 290), (64, 20, 20)])
def test_positions_outside_the_caches(torch_dev, T, pos, max_pos):
    """Rows before position 0 and from max_pos on read no cache row (the caches end where their tensors do) and give
    zeros; the rows between are the oracle's."""
    torch = torch_dev
    from tritify_amd import backend as B
    from tritify_amd import workloads as W

    print(f"case: dec attention outside T={T} pos={pos} max_pos={max_pos}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(T + max_pos)
    nh, nkv, hd = 4, 2, 64
    qkv = rng.integers(-12, 12, size=(T, (nh + 2 * nkv) * hd)).astype(np.int8)
    kc, vc = (rng.integers(-12, 12, size=max_pos * nkv * hd).astype(np.int8) for _ in range(2))
    exp = W.exp_table().astype(np.int32)
    o = torch.full((T * nh * hd,), 99, dtype=torch.int8, device="cuda")
    d = [torch.from_numpy(a.reshape(-1)).cuda() for a in (qkv, kc, vc, exp)]
    p = torch.tensor([pos], dtype=torch.int32, device="cuda")
    B.check(B.lib().kt_hip_dec_attention(0, d[0].data_ptr(), T, qkv.shape[1], p.data_ptr(), d[1].data_ptr(),
                                         d[2].data_ptr(), nh, nkv, hd, d[3].data_ptr(), o.data_ptr(), max_pos, 0),
            "dec attention")
    got = o.cpu().numpy().reshape(T, nh, hd)
    for t in range(T):
        for h in range(nh):
            want = np.zeros(hd, np.int8)
            if 0 <= pos + t < max_pos:
                want = O.dec_attend(qkv[t, h * hd:(h + 1) * hd], kc, vc, pos + t, nkv, h // (nh // nkv), hd, exp)
            assert np.array_equal(got[t, h], want), (t, h)
