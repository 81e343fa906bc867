"""The sampler's quotient of a bf16 logit and a temperature (sample_logit_candidates_kernel): a correctly rounded reciprocal, a product and ONE remainder
step give the bits of the division.  Restated with float64 in the place of the fused operations: it holds the products exactly, and what it cuts off a sum
is put back as a nudge, so that the sum is rounded once."""
import numpy as np
import pytest


@pytest.mark.parametrize("seed", range(4))
def test_one_remainder_step_is_the_division(seed):
    rng = np.random.default_rng(seed)
    bits = np.concatenate([rng.integers(0, 1 << 23, 1 << 13), np.arange(256), (1 << 23) - 1 - np.arange(256)]).astype(np.uint32)
    t = (bits | np.uint32(0x3F800000)).view(np.float32)[:, None]          # every exponent rounds alike
    v = (np.arange(128, 256, dtype=np.float32) / 128)[None, :]            # the significands of bf16
    r = (np.float32(1) / t).astype(np.float32)
    d = v * r
    left = (v.astype(np.float64) - t.astype(np.float64) * d).astype(np.float32)
    a, b = d.astype(np.float64), left.astype(np.float64) * r
    s = a + b
    rest = (a - (s - (s - a))) + (b - (s - a))
    got = np.where(rest == 0, s, np.nextafter(s, np.where(rest > 0, np.inf, -np.inf))).astype(np.float32)
    np.testing.assert_array_equal(got, v / t)
