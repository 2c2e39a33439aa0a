"""The one-row QuantLinear product at the edges of its k slices and of its columns per CTA, against the oracle's
forward_int, codes, Scale and maxima bit for bit: rows just past the short kernel's 1024 values, a partly filled last
chunk round, the longest row, and outputs on both sides of the line between 4 and 8 columns a CTA, with a bias (its
factor is per CTA) and without."""
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

WLEVELS = 265720


@pytest.mark.parametrize("inp,out,with_bias", [
    (1024, 9, True), (1025, 9, False), (1088, 1024, True), (4095, 1025, False), (4097, 3, True), (4864, 896, True),
    (7000, 1032, True), (8192, 5, False), (8192, 1100, False),
])
def test_one_row_against_the_oracle(torch_dev, inp, out, with_bias):
    import tritify_amd as TA
    from oracle import oracle as O

    print(f"case: one row in={inp} out={out} bias={with_bias}", file=sys.stderr, flush=True)
    rng = np.random.default_rng(inp + out)
    x = rng.integers(-(2**28), 2**28 + 1, size=inp).astype(np.int32)
    w = rng.integers(-WLEVELS, WLEVELS + 1, size=out * inp).astype(np.int32)
    w[:inp] = WLEVELS * np.where(x[:inp] < 0, -1, 1)  # the largest sum a row can have
    bias = rng.integers(-(2**28), 2**28, size=out).astype(np.int64) if with_bias else None
    xs, ws, bs = (1509949440, 58), (1657624235, 49), (1318646415, 57) if with_bias else None
    ql = TA.QuantLinear("t", w, out, inp, ws, None if bias is None else (bias, bs))
    y, sc = ql.forward_int_host(x, xs)
    yo, so, xmax, ymax = O.quant_linear_forward(x, 1, inp, xs, w, out, ws, bias=bias, bs=bs or (0, 0))
    assert np.array_equal(y, yo), f"codes differ at {np.argwhere(y != yo)[:5].tolist()}"
    assert (sc["mant"], sc["shift"], sc["xmax"], sc["ymax"]) == (*so, xmax, ymax)
