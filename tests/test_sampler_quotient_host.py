"""The sampler's quotient of a bf16 logit and a temperature (sample_logit_candidates_kernel): a correctly rounded reciprocal, a product and ONE remainder
step give the bits of the division.  Restated with float64 in the place of the fused operations: it holds the products exactly, and what it cuts off a sum
is put back as a nudge, so that the sum is rounded once."""
import ctypes
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor

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


QUOTIENTS = r"""
#include <math.h>
#include <string.h>
/* temperatures first .. last - 1 (significands of 1.0 to 2.0) under all significands of a bf16 logit: how many quotients are not the division's */
__attribute__((target_clones("avx512f", "fma", "default"), optimize("no-trapping-math"))) long wrong(unsigned first, unsigned last) {
  long n = 0;
  for (unsigned s = 128; s < 256; ++s) {
    const float v = (float)s / 128.0f;
    long bad = 0;
    for (unsigned i = first; i < last; ++i) {
      const unsigned bits = 0x3F800000u | i;
      float t;
      memcpy(&t, &bits, 4);
      const float r = 1.0f / t, d = v * r, q = __builtin_fmaf(__builtin_fmaf(-t, d, v), r, d);
      bad += q != v / t;
    }
    n += bad;
  }
  return n;
}
"""


@pytest.mark.skipif(shutil.which("gcc") is None or "fma" not in open("/proc/cpuinfo").read(), reason="no compiler, or a CPU whose fmaf is a library's")
def test_all_quotients(tmp_path):
    """Every significand of a bf16 logit over every one of a temperature; exponents only scale them."""
    (tmp_path / "q.c").write_text(QUOTIENTS)
    subprocess.run(["gcc", "-O3", "-ffp-contract=off", "-shared", "-fPIC", str(tmp_path / "q.c"), "-o", str(tmp_path / "q.so"), "-lm"], check=True)
    lib = ctypes.CDLL(str(tmp_path / "q.so"))
    lib.wrong.restype, lib.wrong.argtypes = ctypes.c_long, [ctypes.c_uint, ctypes.c_uint]
    with ThreadPoolExecutor(4) as pool:
        assert sum(pool.map(lambda i: lib.wrong(i << 19, (i + 1) << 19), range(16))) == 0
