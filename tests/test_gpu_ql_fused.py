"""QuantLinear with the GELU table behind it and with what is known of its input: the same integers as the plain calls
in sequence, over odd and even widths, outputs that are not 8-byte aligned, fewer and more values than one step of the
grid, a zero input with and without a bias, and a zero scale."""
import sys

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def layer(rng, out, inp, bias):
    import tritify_amd as T

    w = rng.integers(-O.WLEVELS, O.WLEVELS + 1, size=(out, inp)).astype(np.int32)
    b = (rng.integers(-(2**28), 2**28, size=out).astype(np.int64), (1318646415, 57)) if bias else None
    return T.QuantLinear("t", w, out, inp, (1657624235, 49), b)


@pytest.mark.parametrize("rows,inp,out,bias", [(2, 64, 33, True), (5, 70, 128, False), (130, 100, 515, True),
                                               (1100, 64, 1024, True)])
@pytest.mark.parametrize("x_scale", [(1509949440, 58), (1509949440, 45), (0, 0)])
@pytest.mark.parametrize("zero", [False, True])
def test_gelu_behind_the_layer(torch_dev, rows, inp, out, bias, x_scale, zero):
    torch = torch_dev
    import tritify_amd as T
    from tritify_amd import backend as B
    from tritify_amd.refvision import gelu_table

    print(f"case: ql gelu rows={rows} in={inp} out={out} bias={bias} xs={x_scale} zero={zero}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(rows + out)
    ql = layer(rng, out, inp, bias)
    x = torch.from_numpy(rng.integers(-(2**27), 2**27, size=rows * inp).astype(np.int32) * (0 if zero else 1)).cuda()
    xs = T.qscale_record(*x_scale)
    codes, lut = gelu_table()
    h, hs = ql.forward_int(x, xs, rows)
    want, wrec = torch.empty_like(h), torch.full((4,), -1, dtype=torch.int64, device="cuda")
    B.ref_gelu(h, hs, rows * out, codes, lut, want, wrec)
    for shift in (0, 1):  # the second: outputs on odd words
        y = torch.full((rows * out + 2,), 77, dtype=torch.int32, device="cuda")
        rec = torch.full((4,), -1, dtype=torch.int64, device="cuda")
        parts = torch.full((B.QL_PARTS,), -1, dtype=torch.int32, device="cuda")
        ws, n = ql.workspace(rows)
        B.quant_linear_gelu(x, rows, inp, xs, ql.w_planes, ql.pw, out, ql.w_scale, ql.bias, ql.b_scale, ws, n, codes,
                            lut, y[shift:], rec, parts)
        assert torch.equal(y[shift:shift + rows * out], want) and torch.equal(rec, wrec)
        assert (y[:shift] == 77).all() and (y[shift + rows * out:] == 77).all()
        assert int(parts.cpu().numpy().view(np.uint32).max()) == int(want.abs().max())
        # the next layer from those maxima equals the next layer from nothing known
        if shift == 0:
            nxt = layer(rng, 40, out, True)
            a, ar = nxt.forward_int(want, wrec, rows)
            b, br = nxt.forward_int(y[:rows * out], rec, rows, x_kind=B.X_PARTS, xmax_dev=parts)
            assert torch.equal(a, b) and torch.equal(ar, br)


@pytest.mark.parametrize("rows,inp,outs", [(2, 64, (128, 256, 33)), (37, 896, (128, 130)), (3000, 70, (70,))])
@pytest.mark.parametrize("zero", [False, True])
def test_closed_inputs(torch_dev, rows, inp, outs, zero):
    """An input whose largest code is 2^28 (or all zero at a zero scale), declared as closed; outputs on odd words."""
    torch = torch_dev
    import tritify_amd as T
    from tritify_amd import backend as B

    print(f"case: ql closed rows={rows} in={inp} outs={outs} zero={zero}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(rows)
    x = rng.integers(-(2**27), 2**27, size=rows * inp).astype(np.int32)
    x[-1] = -2**28
    x = torch.from_numpy(x * (0 if zero else 1)).cuda()
    xs = T.qscale_record(*((0, 0) if zero else (1509949440, 58)))
    total = sum(outs)
    w = rng.integers(-O.WLEVELS, O.WLEVELS + 1, size=(total, inp)).astype(np.int32)
    planes = torch.empty(3 * total * T.kp(inp), dtype=torch.int8, device="cuda")
    T.pack_planes(torch.from_numpy(w).cuda(), total, inp, 3, planes)
    bias = torch.from_numpy(rng.integers(-(2**28), 2**28, size=total).astype(np.int64)).cuda()
    n, _ = B.quant_linear_workspace(rows, inp, total)
    got = []
    for kind, shift in ((B.X_ANY, 0), (B.X_CLOSED, 0), (B.X_CLOSED, 1)):
        ws = torch.full((n,), 0x5A, dtype=torch.uint8, device="cuda")
        ys = [torch.full((rows * o + 1,), 7, dtype=torch.int32, device="cuda") for o in outs]
        rec = torch.full((4 * len(outs),), -1, dtype=torch.int64, device="cuda")
        B.quant_linear_multi(x, rows, inp, xs, outs, planes, 3, [(1657624235, 49)] * len(outs), bias,
                             [(1318646415, 57)] * len(outs), ws, n, [y[shift:] for y in ys], rec, x_kind=kind)
        got.append([y[shift:shift + rows * o] for y, o in zip(ys, outs)] + [rec])
    for other in got[1:]:
        assert all(torch.equal(a, b) for a, b in zip(got[0], other))
    with pytest.raises(B.HipError):  # partial maxima without any
        B.quant_linear_multi(x, rows, inp, xs, outs, planes, 3, [(1657624235, 49)] * len(outs), bias,
                             [(1318646415, 57)] * len(outs), ws, n, ys, rec, x_kind=B.X_PARTS)
