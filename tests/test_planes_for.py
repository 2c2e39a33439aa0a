"""kt_hip_planes_for on both sides of every bound it decides by: the ends of one, two and three balanced base-256 digits,
the power of two its quick test stops at, and the ends of i32 (host only, no GPU)."""
import numpy as np
import pytest


def digits(lo, hi):
    mn, mx = -128, 127
    for p in range(1, 5):
        if lo >= mn and hi <= mx:
            return p
        mn, mx = 256 * mn - 128, 256 * mx + 127
    return 5


@pytest.mark.parametrize("v", [0, 127, 128, -128, -129, 32639, 32640, -32896, -32897, 2**22 - 1, 2**22, -2**22, -2**22 - 1,
                               8355711, 8355712, -8421504, -8421505, 2**31 - 1, -2**31])
@pytest.mark.parametrize("n", [1, 7, 1000])
def test_planes_for(v, n):
    from tritify_amd import backend as B

    a = np.zeros(n, np.int32)
    a[n // 2] = v
    p = digits(min(0, v), max(0, v))
    assert B.planes_for(a) == (1 if p == 1 else 3 if p <= 3 else 5)
