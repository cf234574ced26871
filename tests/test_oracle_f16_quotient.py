"""The float16 row quantizer's quotient (quant.hip quant_rows_vec): with r = rn(1 / s) and q0 = rn(x r) in
float32, q1 = fma(fma(-q0, s, x), r, q0) rounds to the same float16 as the division x / s that the
reference makes. The device's steps are restated in numpy, each fused multiply-add rounded once, and
compared over every pair of significands and over subnormal values and scales. Without the correction step
the comparison must fail."""

import numpy as np
import pytest

NORMAL = (1024 + np.arange(1024)).astype(np.float64) / 1024  # every significand of a normal float16
SUBNORMAL = np.arange(1, 1024).astype(np.float64) * 2.0 ** -24


def _fma32(a, b, c):
    """float32 of a * b + c, rounded once. a * b of float32 numbers is exact in float64; the sum is rounded to odd
    there, which leaves the second rounding, to float32, as if it were the only one."""
    p = a.astype(np.float64) * b.astype(np.float64)
    c = c.astype(np.float64)
    s = p + c
    t = s - p
    err = (p - (s - t)) + (c - t)  # s + err == p + c exactly
    bits = s.view(np.int64)
    even = (bits & 1) == 0
    toward = np.where((err > 0) == (s > 0), bits + 1, bits - 1)  # the odd neighbour on err's side
    s = np.where((err != 0) & even, toward, bits).view(np.float64)
    return s.astype(np.float32)


def _quotients(x, s, corrected=True):
    """(device's, division's) float16 bits of every x (rows) over every s (columns)."""
    x, s = (np.ascontiguousarray(v) for v in np.broadcast_arrays(x.astype(np.float32)[:, None], s.astype(np.float32)[None, :]))
    r = np.float32(1) / s
    q = x * r
    if corrected:
        q = _fma32(_fma32(-q, s, x), r, q)
    return q.astype(np.float16).view(np.uint16), (x / s).astype(np.float16).view(np.uint16)


# x, s and the exponent by which x is scaled: quotients around 1, up to 127 and beyond, into float16's
# subnormal range and below its smallest value; subnormal values and subnormal scales (a row of tiny values).
@pytest.mark.parametrize("x,s,exponent", [(NORMAL, NORMAL, e) for e in (0, 6, 7, *range(-25, -13))]
                         + [(SUBNORMAL, NORMAL, 0), (SUBNORMAL, NORMAL * 2.0 ** -14, 0), (SUBNORMAL, SUBNORMAL, 0),
                            (NORMAL, SUBNORMAL, -14), (NORMAL, SUBNORMAL, -17 + 7)])
def test_quotient_rounds_like_the_division(x, s, exponent):
    with np.errstate(over="ignore"):
        got, want = _quotients(x * 2.0 ** exponent, s)
    assert np.array_equal(got, want)


def test_planted_uncorrected_quotient_is_caught():
    """q0 alone misses exact ties, which only quotients in the subnormal range reach (19 of a million here)."""
    got, want = _quotients(NORMAL * 2.0 ** -20, NORMAL, corrected=False)
    assert not np.array_equal(got, want)
