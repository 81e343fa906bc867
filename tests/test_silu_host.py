"""silu of a bf16 gate (glu.hpp), compiled for the host: the short form against the one with a full exponential and a division."""
import ctypes
import shutil
import subprocess
from pathlib import Path

import numpy as np
import pytest

CSRC = Path(__file__).resolve().parent.parent / "sglang_amd" / "csrc"
STUB = """#include <cmath>
#include <cstdint>
#include <cstring>
#define __host__
#define __device__
#define __forceinline__ inline
#define __builtin_amdgcn_rcpf(x) (1.0f / (x))
inline float fast_exp2(float x) { return exp2f(x); }
inline float rbf(float f) {                  // (numbers only)
  uint32_t u;
  memcpy(&u, &f, 4);
  u = (u + 0x7fffu + (u >> 16 & 1u)) & 0xffff0000u;
  memcpy(&f, &u, 4);
  return f;
}
"""
SOURCE = """#include "glu.hpp"
extern "C" void both(const float* g, int n, float* near_, float* any_) {
  for (int i = 0; i < n; ++i) {
    near_[i] = rbf(sgl_amd::silu_near(g[i]));
    any_[i] = rbf(sgl_amd::silu_any(g[i]));
  }
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not installed")
def test_short_silu_of_every_bf16_gate(tmp_path):
    """The same bf16 value with the same sign, a gate of -0 included, for every gate that the short form takes.  The two evaluations differ by a few 2^-24 of
    the value before they are rounded, so a value within 2^-21 of itself of the middle between two bf16 may go to either."""
    (tmp_path / "common.hpp").write_text(STUB)
    (tmp_path / "glu.hpp").write_text((CSRC / "glu.hpp").read_text())
    (tmp_path / "silu.cpp").write_text(SOURCE)
    subprocess.run(["g++", "-O1", "-std=c++17", "-ffp-contract=off", "-shared", "-fPIC", str(tmp_path / "silu.cpp"), "-o", str(tmp_path / "silu.so")], check=True)
    g = (np.arange(65536, dtype=np.uint32) << 16).view(np.float32)
    g = np.ascontiguousarray(g[np.abs(g) <= 80])
    near, full = np.empty_like(g), np.empty_like(g)
    at = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    ctypes.CDLL(str(tmp_path / "silu.so")).both(at(g), g.size, at(near), at(full))
    assert np.array_equal(np.signbit(near), np.signbit(full)) and np.array_equal(np.signbit(near), np.signbit(g))
    off = near != full
    want = g.astype(np.float64) / (1 + np.exp(-g.astype(np.float64)))
    middle = (near.astype(np.float64) + full) / 2
    assert np.all(np.abs(want - middle)[off] <= np.abs(want)[off] * 2.0 ** -21), g[off]
