"""The spans' integer division by a binary32 estimate (span_div in
csrc/wgc_core.h), restated in numpy: for every reciprocal within one ulp
of 1/den the corrected quotient is the truncated integer quotient, for
|num| < 2^15 and 0 <= i <= den < 2^15."""
import numpy as np
import pytest


def span_div(num, i, den, ulps):
    n = np.abs(num).astype(np.uint32)
    rcp = (np.float32(1.0) / den.astype(np.float32)).view(np.uint32) + np.uint32(ulps & 0xFFFFFFFF)
    est = n.astype(np.float32) * (i.astype(np.float32) * rcp.view(np.float32))
    q = est.astype(np.int64)
    r = n.astype(np.int64) * i - q * den
    q = np.where(r < 0, q - 1, np.where(r >= den, q + 1, q))
    return np.where(num < 0, -q, q)


@pytest.mark.parametrize("ulps", [-1, 0, 1])
def test_estimate_is_corrected_to_the_quotient(ulps):
    rng = np.random.default_rng(5 + ulps)
    small = [g.reshape(-1) for g in np.meshgrid(np.arange(-70, 71), np.arange(0, 61), np.arange(1, 61))]
    keep = small[1] <= small[2]
    den = np.concatenate([small[2][keep], rng.integers(1, 32768, 400000), np.full(4000, 32767)])
    i = np.concatenate([small[1][keep], rng.integers(0, den[keep.sum():] + 1)])
    num = np.concatenate([small[0][keep], rng.integers(-32767, 32768, 404000)])
    # exact quotients and their neighbours, where an estimate can slip
    edge = rng.integers(0, len(den), 200000)
    i[edge] = np.maximum(den[edge] - rng.integers(0, 3, len(edge)), 0)
    want = np.sign(num) * (np.abs(num) * i // den)
    assert np.array_equal(span_div(num, i, den, ulps), want)
