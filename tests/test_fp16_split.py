"""The precision that the dense kernels' split of a row states (gemm_rows.hip's
head), in numpy's fp16: a value as hi + lo, each the nearest fp16, after a power-of-two
scale that puts the row's largest magnitude in [2^11, 2^12) (the scale that follows
the row) or in [2^14, 2^15) (the row's own)."""
from __future__ import annotations

import numpy as np
import pytest


def halves(x):
    hi = x.astype(np.float16).astype(np.float64)
    return hi + (x - hi).astype(np.float16).astype(np.float64)


@pytest.mark.parametrize("top,exact_to,error", [(11, -14, -36), (14, -17, -39)], ids=["online", "own"])
def test_hi_plus_lo(top, exact_to, error):
    """22 significand bits (a relative error of at most 2^-22) down to 2^exact_to
    of the row's largest power of two, and an error of at most 2^error of it
    below: half of fp16's smallest step, 2^-25, under the scale."""
    rng = np.random.default_rng(top)
    for e in range(top, -40, -1):  # fp32 values of every binade, 24-bit significands
        x = (rng.integers(2 ** 23, 2 ** 24, 20000) * 2.0 ** (e - 23)).astype(np.float64)
        err = np.abs(halves(x) - x)
        assert err.max() <= max(2.0 ** (error + top), 2.0 ** (e - 23))
        if e >= top + exact_to:
            assert (err / x).max() <= 2.0 ** -22
    x = rng.integers(2 ** 23, 2 ** 24, 200000) * 2.0 ** (top + exact_to - 2 - 23)  # a quarter below the limit: fewer bits
    assert (np.abs(halves(x) - x) / x).max() > 2.0 ** -22
