"""The engine-semantics attention step on several CTAs per head (kt_hip_ref_attention_step_ws) where its split changes:
four, two or one lane per cached step up to 256, 512 and more steps (one lane where head_dim has no multiple of 16, or
the cache rows no 16-byte alignment); the first v values of a wave, 8 per share of the steps; slices of the P.V that
do not divide the CTA; one head as wide as the CTA. Codes, Scale and the cache rows against the oracle, exactly."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def rec(torch, sc):
    w = np.zeros(4, dtype=np.int64)
    w[0] = sc[0]
    w.view(np.int32)[2] = sc[1]
    return torch.from_numpy(w).cuda()


@pytest.mark.parametrize("nh,nkv,hd,ms", [(2, 1, 64, 1030), (4, 2, 48, 520), (2, 2, 192, 520), (3, 1, 20, 520),
                                          (2, 1, 6, 520), (1, 1, 1024, 9)])
def test_ref_attention_heads_at_the_edges_of_its_split(torch_dev, nh, nkv, hd, ms):
    torch = torch_dev
    from tritify_amd import backend as B

    print(f"case: ref_attention heads nh={nh} nkv={nkv} hd={hd} steps={ms}", file=sys.stderr, flush=True)
    cfg = dict(dim=64, layers=1, nh=nh, nkv=nkv, hd=hd, hidden=64, vocab=8, eps=1e-6, theta=1.0e6, max_seq=ms)
    cache = O.RefCache(O.RefModel(11, cfg))
    qd, kvd = nh * hd, nkv * hd
    cos_d, sin_d = (torch.from_numpy(t.view(np.uint8)).cuda() for t in B.ref_rope_tables(ms, hd, cfg["theta"]))
    exp_codes, exp_lut = B.ref_codelut(B.LUT_EXP, -30.0, 0.0, 16, 20, False)
    exp_d = torch.from_numpy(exp_codes).cuda()
    isq = B.ref_scale_from_f64(1.0 / np.sqrt(hd))
    kc, vc = (torch.zeros(ms * kvd, dtype=torch.int32, device="cuda") for _ in range(2))
    ks_d, vs_d = (torch.zeros(ms * 16, dtype=torch.uint8, device="cuda") for _ in range(2))
    o, os_ = torch.zeros(qd, dtype=torch.int32, device="cuda"), rec(torch, (0, 0))
    pos_d = torch.zeros(1, dtype=torch.int32, device="cuda")
    ws = torch.full((B.ref_attention_step_workspace(ms, nh, hd),), 0x77, dtype=torch.uint8, device="cuda")
    rng = np.random.default_rng(hd + ms)
    sc = lambda lo, hi: (int(rng.integers(2**30, 2**31)), int(rng.integers(lo, hi)))  # noqa: E731
    check = {0, 1, 2, 254, 255, 256, 257, 510, 511, 512, 513, 1022, 1023, 1024, 1025, ms - 1}
    for p in range(ms):
        q, k, v = (rng.integers(-(2**28), 2**28, size=n).astype(np.int32) for n in (qd, kvd, kvd))
        qs, ks, vs = sc(78, 84), sc(40, 62), sc(40, 62)
        if p % 7 == 3:
            ks = (0, 0)
        if p % 11 == 5:
            vs = (0, 0)
        pos_d.fill_(p)
        t = [torch.from_numpy(a).cuda() for a in (q, k, v)]
        B.ref_attention_step(t[0], rec(torch, qs), t[1], rec(torch, ks), t[2], rec(torch, vs), pos_d, nh, nkv, hd, ms,
                             kc, vc, ks_d, vs_d, cos_d, sin_d, isq, exp_d, exp_lut, o, os_, ws_dev=ws)
        if p in check:
            oo, so = O.rd_attention_core(cache, q, qs, k, ks, v, vs, p)
            w = os_.cpu().numpy()
            assert np.array_equal(o.cpu().numpy(), oo), p
            assert (int(w[0]), int(w.view(np.int32)[2])) == tuple(so), p
            assert np.array_equal(vc[p * kvd:(p + 1) * kvd].cpu().numpy(), v), p
        else:
            O.rd_attention_append(cache, k, ks, v, vs, p)
