// The chunked recurrences of recurrent_chunk.hip for 16-bit activations on v_mfma_f32_16x16x32_bf16.
//
// Every product there has at least one operand that is a 16-bit input, so it is exact on the bf16 matrix cores once the other, fp32,
// operand is written as the sum of three bf16 values (8 + 8 + 8 significant bits by truncation: the sum is the fp32 value itself).
// Three instructions of 16 cycles then do what eight of 32 cycles did; the accumulators are the same fp32.
//
// A workgroup is four preparing waves and up to four column waves.  The column waves hold the state (16 value columns each) and walk
// the chunks: that walk is the serial chain which bounds the kernel, so everything that does not depend on the state -- rows to LDS,
// scan of the gates, the tokens' products among themselves -- is done by the preparing waves one chunk ahead.
//
// What bounds it now: a round's instruction issue and LDS reads (each column wave reads all rows of the chunk), 2.8 us for 64 tokens of Mamba-2
// (1 800 clocks of them matrix instructions of a SIMD) and 2.5 us for 32 tokens of the delta rule, where the inverse's wave is the longest.
// Chunks of 64 suit Mamba-2 (the state is split once a chunk); the inverse and a third image of the rows keep the delta rule at 32.
// Measured: Mamba-2 64 heads of 64 x 128, 4 segments of 1 600 - 2 460 tokens 456 -> 109 us; delta rule 32 heads of 128 x 128, 3 segments of
// 1 290 - 1 880 tokens 749 -> 156 us.  Error of the state against 64 bits (relative 2-norm, general kernel / this one, 14 draws of 17 to 1 800
// tokens each): Mamba-2 1.0e-7 / 7.4e-8, delta rule 1.4e-7 / 1.1e-7, at most 0.85 of the general kernel's in each of them; behind 2 000 to 8 000
// tokens of one sign that are hardly forgotten 6.4e-7 .. 1.6e-6 / 1.0e-7 .. 4.1e-7 and 5.5e-7 / 2.5e-7.
//
// Operand layouts of the instruction (lane = (i = lane & 15, g = lane / 16), slots j = 0..7): A[row i][8 g + j], B[8 g + j][column i],
// result rows 4 g + r, column i.  The state's registers go into the next product as they are: tiles 2 u and 2 u + 1 fill the slots of
// k-step u with rows 32 u + 16 (j >> 2) + 4 g + (j & 3), and the A operand is read in that order (two 8-byte pieces).  Transposed
// operands (tokens along the contraction) come from row-major images through ds_read_b64_tr_b16.
#pragma once

#include "elem_io.hpp"

namespace sgl_amd {

typedef short split_v4s16_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4_t mfma_bf(const U4& a, const U4& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// the same over 16 rows of the contraction: lane group g holds rows 4 g .. 4 g + 3
__device__ __forceinline__ f32x4_t mfma_bf16k(const uint2& a, const uint2& b, f32x4_t c) {
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(split_v4s16_t, a), __builtin_bit_cast(split_v4s16_t, b), c, 0, 0, 0);
}

__device__ __forceinline__ f32x4_t fma4(const f32x4_t& a, float b, const f32x4_t& c) {
  return f32x4_t{fmaf(a[0], b, c[0]), fmaf(a[1], b, c[1]), fmaf(a[2], b, c[2]), fmaf(a[3], b, c[3])};
}

// v = h + m + l exactly (above the denormals; an infinity becomes NaN): the leading 8 significant bits, the next 8 and the rest.  (Not contracted: of a v that is a
// product, fma(a, b, -h) would leave more than 8 bits to l, whose end is cut off.)
__device__ __forceinline__ void split3(float v, uint32_t& h, uint32_t& m, uint32_t& l) {
#pragma clang fp contract(off)
  h = __float_as_uint(v) & 0xffff0000u;
  const float r = v - __uint_as_float(h);
  m = __float_as_uint(r) & 0xffff0000u;
  l = __float_as_uint(r - __uint_as_float(m));
}

// two values' upper halves in one dword (a below b)
__device__ __forceinline__ uint32_t pack_hi(uint32_t a, uint32_t b) { return __builtin_amdgcn_perm(b, a, 0x07060302u); }

// eight values -> three operands
__device__ __forceinline__ void split8(const float (&v)[8], U4 (&p)[3]) {
  uint32_t* w0 = reinterpret_cast<uint32_t*>(&p[0]);
  uint32_t* w1 = reinterpret_cast<uint32_t*>(&p[1]);
  uint32_t* w2 = reinterpret_cast<uint32_t*>(&p[2]);
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    uint32_t h0, m0, l0, h1, m1, l1;
    split3(v[2 * q], h0, m0, l0);
    split3(v[2 * q + 1], h1, m1, l1);
    w0[q] = pack_hi(h0, h1);
    w1[q] = pack_hi(m0, m1);
    w2[q] = pack_hi(l0, l1);
  }
}

// rows r0 .. r0 + 3 and r0 + GAP .. r0 + GAP + 3 (r0 already the lane group's) of the 16 columns from `col` on, transposed: slots 0 - 3 and 4 - 7
// <- those rows, lane i <- column i.  GAP 4 with r0 = 8 g: natural order; GAP 16 with r0 = 4 g: the state's slot order.
template <int GAP = 4>
__device__ __forceinline__ U4 read_tr8(const uint16_t* img, int stride, int r0, int col, int i16) {
  typedef __attribute__((address_space(3))) split_v4s16_t* lds_t;
  const uint16_t* a = img + (r0 + (i16 >> 2)) * stride + col + (i16 & 3) * 4;
  const split_v4s16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(a));
  const split_v4s16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(a + GAP * stride));
  U4 o;
  o.x = __builtin_bit_cast(uint2, lo).x; o.y = __builtin_bit_cast(uint2, lo).y;
  o.z = __builtin_bit_cast(uint2, hi).x; o.w = __builtin_bit_cast(uint2, hi).y;
  return o;
}

// rows r0 .. r0 + 3 (r0 already the lane group's) of the 16 columns from `col` on, transposed
__device__ __forceinline__ uint2 read_tr4(const uint16_t* img, int stride, int r0, int col, int i16) {
  typedef __attribute__((address_space(3))) split_v4s16_t* lds_t;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(img + (r0 + (i16 >> 2)) * stride + col + (i16 & 3) * 4)));
}

// the A operand in the state's slot order: columns n0 + 4 g .. + 3 and n0 + 16 + 4 g .. + 3 of one row
__device__ __forceinline__ U4 read_pair(const uint16_t* row, int n0, int g) {
  const uint2 a = *reinterpret_cast<const uint2*>(row + n0 + 4 * g), b = *reinterpret_cast<const uint2*>(row + n0 + 16 + 4 * g);
  return U4{a.x, a.y, b.x, b.y};
}

// rows [0, ROWS) x [0, n) of a strided matrix in 16-byte pieces, a chunk ahead in registers of the preparing threads; rows >= len and
// columns >= n are zero.  The pieces' offsets are formed once: a fetch adds them to a uniform address.
constexpr int kPrepWaves = 4;

template <int ROWS, int NP>
struct RowPieces {
  static constexpr int kThreads = 64 * kPrepWaves, kPieces = (ROWS * NP / 8 + kThreads - 1) / kThreads;
  U4 raw[kPieces];
  uint32_t off[kPieces];
  __device__ __forceinline__ static int row(int i, int tid) { return (i * kThreads + tid) / (NP / 8); }
  __device__ __forceinline__ static int col(int i, int tid) { return (i * kThreads + tid) % (NP / 8) * 8; }
  __device__ __forceinline__ void place(int64_t stride, int tid) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) off[i] = static_cast<uint32_t>(row(i, tid) * static_cast<int>(stride) + col(i, tid));
  }
  __device__ __forceinline__ void fetch(const uint16_t* src, int len, int n, int tid) {
#pragma unroll
    for (int i = 0; i < kPieces; ++i) {
      const bool in = row(i, tid) < len && col(i, tid) < n;
      raw[i] = U4{0u, 0u, 0u, 0u};
      if (in) raw[i] = ld16(src + off[i]);
    }
  }
  __device__ __forceinline__ void commit(uint16_t* dst, int ls, int tid) const {
#pragma unroll
    for (int i = 0; i < kPieces; ++i)
      if (ROWS * NP / 8 % kThreads == 0 || row(i, tid) < ROWS) st16(dst + row(i, tid) * ls + col(i, tid), raw[i]);
  }
};

// v moved by a DPP pattern, 0 where the pattern has no source lane or `rows` leaves the 16-lane row out
template <int CTRL, int ROWS = 0xf>
__device__ __forceinline__ double dpp_f64(double v) {
  const uint2 w = __builtin_bit_cast(uint2, v);
  uint2 o;
  o.x = __builtin_amdgcn_update_dpp(0, static_cast<int>(w.x), CTRL, ROWS, 0xf, true);
  o.y = __builtin_amdgcn_update_dpp(0, static_cast<int>(w.y), CTRL, ROWS, 0xf, true);
  return __builtin_bit_cast(double, o);
}
template <int CTRL>
__device__ __forceinline__ float dpp_f32(float v) {
  return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, 0xf, 0xf, true));
}

// inclusive prefix sum over the wave's lanes, or over its halves of N = 32, in double (row_shr 1, 2, 4, 8, then the rows' last lanes:
// row_bcast 15 and 31)
template <int N>
__device__ __forceinline__ double scan_lanes(double v) {
  v += dpp_f64<0x111>(v);
  v += dpp_f64<0x112>(v);
  v += dpp_f64<0x114>(v);
  v += dpp_f64<0x118>(v);
  v += dpp_f64<0x142, 0xa>(v);
  if constexpr (N == 64) v += dpp_f64<0x143, 0xc>(v);
  return v;
}

// the value of one lane, for all
__device__ __forceinline__ double lane_f64(double v, int lane) {
  const uint2 w = __builtin_bit_cast(uint2, v);
  return __builtin_bit_cast(double, uint2{static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w.x), lane)),
                                          static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(w.y), lane))});
}

// e^v of a v that a float does not hold (rounded to one, an exponent of 50 is off by 3e-6 of the result): the rest as a first-order factor
__device__ __forceinline__ float exp_f64(double v) {
  const float f = static_cast<float>(v), e = expf(f);
  return e > 0.f ? fmaf(e, static_cast<float>(v - static_cast<double>(f)), e) : e;       // (v may lie beyond the floats: 0)
}

// sum over N neighbouring lanes (4, 8 or 16; quad_perm xor 1, xor 2, then mirrors of half rows and rows), left in all of them
template <int N>
__device__ __forceinline__ float sum_lanes(float v) {
  v += dpp_f32<0xb1>(v);
  v += dpp_f32<0x4e>(v);
  if constexpr (N >= 8) v += dpp_f32<0x141>(v);
  if constexpr (N >= 16) v += dpp_f32<0x140>(v);
  return v;
}

// A rendezvous of the preparing waves alone (a barrier would stop the column waves too): each adds one to a counter in LDS and waits for
// the round's total.  Every preparing wave of the workgroup calls it equally often, so every wait ends.
__device__ __forceinline__ void prep_arrive(uint32_t* count) {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(count, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void prep_sync(uint32_t* count, uint32_t& round) {
  round += kPrepWaves;
  prep_arrive(count);
  while (__hip_atomic_load(count, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) < round) __builtin_amdgcn_s_sleep(1);
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ------------------------------------------------------------------------------------------------ Mamba-2, 64 tokens a chunk
template <int NU>
struct Mamba2Split {
  static constexpr int kTok = 64, kNp = 32 * NU, kLs = kNp + 8, kXs = 64 + 8, kGs = kTok + 8;
  uint16_t b[2][kTok * kLs], c[2][kTok * kLs];
  uint16_t x[2][kTok * kXs];
  uint16_t g[2][3][kTok * kGs];                    // (C B^T) o decays, D on the diagonal, in three pieces
  float ec[3][kTok], wj[3][kTok], fix[3][4];       // e^{c_i}, e^{c_n - c_j} dt_j, e^{c_n}
  double cum[2][kTok];
  float dts[2][kTok];
  float colf[2][2][kTok];                          // e^{c_m - c_j} dt_j, m the first token behind j's tile; m the first of j's tile
  int apart[2][4];                                 // tiles whose second factor could leave the floats
  uint32_t count;
};

template <typename Params, int NU>
__device__ __forceinline__ void mamba2_split_body(const Params& p, Mamba2Split<NU>& sm) {
  using L = Mamba2Split<NU>;
  constexpr int Q = L::kTok;
  // neighbours in the launch go to different XCDs: heads of one group, which read the same B and C, lie `groups` apart
  const int b = blockIdx.y, h = blockIdx.x % p.groups * (p.heads / p.groups) + blockIdx.x / p.groups;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i16 = lane & 15, g = lane >> 4;
  const int64_t tok0 = p.seg_start[b];
  const int total = p.seg_len[b];
  if (total <= 0) return;
  const int64_t pos0 = p.positions[tok0];
  const int grp = h / (p.heads / p.groups), inner = p.heads * p.P;
  const int col0 = blockIdx.z * p.col_waves * 16;
  const int chunks = (total + Q - 1) / Q;
  if (wave < kPrepWaves) {
    const int tid = threadIdx.x;
    const float a = -expf(p.A_log[h]), dtb = p.dt_bias[h], dskip = p.D[h];
    const uint16_t* rows0 = static_cast<const uint16_t*>(p.xbc) + tok0 * p.xbc_stride;
    const uint16_t* dtp = static_cast<const uint16_t*>(p.dt) + tok0 * p.dt_stride + h;
    RowPieces<Q, L::kNp> br, cr;
    RowPieces<Q, 64> xr;
    br.place(p.xbc_stride, tid);
    xr.place(p.xbc_stride, tid);
#pragma unroll
    for (int i = 0; i < br.kPieces; ++i) cr.off[i] = br.off[i];
    const int cols = p.P - col0 < 16 * p.col_waves ? p.P - col0 : 16 * p.col_waves;
    auto fetch = [&](int k) __attribute__((always_inline)) {
      const int c0 = k * Q, len = total - c0 < Q ? total - c0 : Q;
      const uint16_t* rows = rows0 + static_cast<int64_t>(c0) * p.xbc_stride;
      br.fetch(rows + inner + grp * p.N, len, p.N, tid);
      cr.fetch(rows + inner + (p.groups + grp) * p.N, len, p.N, tid);
      xr.fetch(rows + h * p.P + col0, len, cols, tid);
    };
    auto commit = [&](int k) __attribute__((always_inline)) {
      br.commit(sm.b[k & 1], L::kLs, tid);
      cr.commit(sm.c[k & 1], L::kLs, tid);
      xr.commit(sm.x[k & 1], L::kXs, tid);
    };
    // the last preparing wave scans the gates two chunks ahead of the column waves (lane = token)
    uint16_t dtr = 0;
    auto fetch_gates = [&](int k) __attribute__((always_inline)) {
      if (k * Q + lane < total) dtr = dtp[static_cast<int64_t>(k * Q + lane) * p.dt_stride];
    };
    auto scan = [&](int k) __attribute__((always_inline)) {
      const int at = k & 1, to = k % 3;
      const float dt = k * Q + lane < total ? softplus_f(bf2f(dtr) + dtb) : 0.f;
      const double c = scan_lanes<Q>(static_cast<double>(a * dt)), cn = lane_f64(c, Q - 1);
      const double f0 = lane_f64(c, 0), f1 = lane_f64(c, 16), f2 = lane_f64(c, 32), f3 = lane_f64(c, 48);       // the tiles' first tokens
      const double cm = g == 0 ? f1 : g == 1 ? f2 : f3, cf = g == 0 ? f0 : g == 1 ? f1 : g == 2 ? f2 : f3;
      sm.cum[at][lane] = c;
      sm.dts[at][lane] = dt;
      sm.colf[at][0][lane] = lane < 48 ? expf(static_cast<float>(cm - c)) * dt : 0.f;
      sm.colf[at][1][lane] = exp_f64(cf - c) * dt;                           // (read only where it cannot overflow:)
      const unsigned long long in_range = __ballot(cf - c < 60.0 && dt < 1e12f);
      if (i16 == 0) sm.apart[at][g] = (in_range >> (16 * g) & 0xffff) != 0xffff;
      sm.ec[to][lane] = expf(static_cast<float>(c));
      sm.wj[to][lane] = expf(static_cast<float>(cn - c)) * dt;
      if (lane == 0) sm.fix[to][0] = expf(static_cast<float>(cn));
    };
    // Tiles on and below the diagonal of (C B^T)_ij e^{c_i - c_j} dt_j, formed transposed: a lane then holds four j of one i.  The
    // decay is e^{c_i - c_m} e^{c_m - c_j}, one exponential a lane: m is the first token behind j's tile, or the tile's own first on the
    // diagonal, where the second factor exceeds 1 and a tile that decays by e^60 or more (or has a dt of 1e12 or more, which is part of
    // it) takes its exponentials one by one.  There both exponents may be many times the one of their product: they keep what a float drops (exp_f64).
    auto product = [&](int k, int ti, int tj) __attribute__((always_inline)) {
      const uint16_t* B = sm.b[k & 1] + (16 * tj + i16) * L::kLs + 8 * g;
      const uint16_t* C = sm.c[k & 1] + (16 * ti + i16) * L::kLs + 8 * g;
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NU; ++u) acc = mfma_bf(ld16(B + 32 * u), ld16(C + 32 * u), acc);
      return acc;
    };
    auto put = [&](int k, int ti, int tj, const f32x4_t& acc) __attribute__((always_inline)) {
      const int at = k & 1, i = 16 * ti + i16, j0 = 16 * tj + 4 * g;
      const bool diag = ti == tj;
      const double ci = sm.cum[at][i];
      float v[4];
      if (!diag || !sm.apart[at][ti]) {
        const float w = exp_f64(ci - sm.cum[at][diag ? 16 * ti : 16 * tj + 16]);
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(&sm.colf[at][diag][j0]);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[r] * (w * e[r]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = j0 + r <= i ? acc[r] * expf(static_cast<float>(ci - sm.cum[at][j0 + r])) * sm.dts[at][j0 + r] : 0.f;
      }
      if (diag) {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = j0 + r <= i ? v[r] + (j0 + r == i ? dskip : 0.f) : 0.f;
      }
      uint32_t h[4], m[4], l[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) split3(v[r], h[r], m[r], l[r]);
      *reinterpret_cast<uint2*>(&sm.g[at][0][i * L::kGs + j0]) = uint2{pack_hi(h[0], h[1]), pack_hi(h[2], h[3])};
      *reinterpret_cast<uint2*>(&sm.g[at][1][i * L::kGs + j0]) = uint2{pack_hi(m[0], m[1]), pack_hi(m[2], m[3])};
      *reinterpret_cast<uint2*>(&sm.g[at][2][i * L::kGs + j0]) = uint2{pack_hi(l[0], l[1]), pack_hi(l[2], l[3])};
    };
    // ten tiles: three (one on the diagonal) to each wave but the last, which scans
    auto grams = [&](int k) __attribute__((always_inline)) {
      if (wave == kPrepWaves - 1) {
        put(k, 3, 2, product(k, 3, 2));
        return;
      }
      const int d = wave == 0 ? 0 : wave + 1, e = wave == 0 ? 1 : d;      // (0,0) (1,0) (1,1) | (2,2) (2,0) (2,1) | (3,3) (3,0) (3,1)
      const f32x4_t a0 = product(k, d, d), a1 = product(k, e, 0), a2 = product(k, e, 1);
      put(k, d, d, a0);
      put(k, e, 0, a1);
      put(k, e, 1, a2);
    };
    if (tid == 0) sm.count = 0;
    uint32_t round = 0;
    fetch(0);
    commit(0);
    if (wave == kPrepWaves - 1) {
      fetch_gates(0);
      scan(0);
      if (chunks > 1) {
        fetch_gates(1);
        scan(1);
        fetch_gates(2);
      }
    }
    if (chunks > 1) fetch(1);
    __syncthreads();
    grams(0);
    __syncthreads();
    for (int k = 0; k < chunks; ++k) {
      if (k + 1 < chunks) {
        commit(k + 1);
        if (k + 2 < chunks) fetch(k + 2);
        prep_sync(&sm.count, round);
        grams(k + 1);
        if (wave == kPrepWaves - 1 && k + 2 < chunks) {
          scan(k + 2);
          fetch_gates(k + 3);
        }
      }
      __syncthreads();
    }
    return;
  }
  const int cw = wave - kPrepWaves, col = col0 + cw * 16 + i16;
  const bool live = col < p.P;
  float* S = p.state + (p.slots[b] * p.heads + h) * static_cast<int64_t>(p.N) * p.P + col;
  uint16_t* yp = static_cast<uint16_t*>(p.y) + tok0 * p.y_stride + static_cast<int64_t>(i16) * p.y_stride + h * p.P + col0 + cw * 16 + 4 * g;
  const int wide = p.P - col0 - cw * 16;                 // the wave's columns (a multiple of 8; 16 and more: all of them)
  f32x4_t s[2 * NU];
#pragma unroll
  for (int t = 0; t < 2 * NU; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * t + 4 * g + r;
      s[t][r] = pos0 > 0 && live && n < p.N ? S[static_cast<int64_t>(n) * p.P] : 0.f;
    }
  __syncthreads();
  __syncthreads();
  for (int k = 0; k < chunks; ++k) {
    const int at = k & 1, c0 = k * Q, len = total - c0 < Q ? total - c0 : Q;
    const float* ec = sm.ec[k % 3];
    const float* wj = sm.wj[k % 3];
    const float fix = sm.fix[k % 3][0];
    const uint16_t* C = sm.c[at] + i16 * L::kLs;
    const uint16_t* B = sm.b[at];
    const uint16_t* G = sm.g[at][0] + i16 * L::kGs + 8 * g;
    // ---- y^T = S^T C^T (a lane holds four columns of one token): the operands of k-step u + 1 are read and split while the products of step u run ----
    f32x4_t y[4];
    U4 cf[2][4], sp[2][3], xf[2];
    uint2 xh[2];
    auto stage = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int ti = 0; ti < 4; ++ti) cf[u & 1][ti] = read_pair(C + 16 * ti * L::kLs, 32 * u, g);
      const float v[8] = {s[2 * u][0], s[2 * u][1], s[2 * u][2], s[2 * u][3], s[2 * u + 1][0], s[2 * u + 1][1], s[2 * u + 1][2], s[2 * u + 1][3]};
      split8(v, sp[u & 1]);
    };
    stage(0);
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      xf[u] = read_tr8(sm.x[at], L::kXs, 32 * u + 8 * g, cw * 16, i16);
      xh[u] = read_tr4(sm.x[at], L::kXs, 32 * u + 4 * g, cw * 16, i16);
    }
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) y[ti] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      if (u + 1 < NU) stage(u + 1);
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int ti = 0; ti < 4; ++ti) y[ti] = mfma_bf(sp[u & 1][q], cf[u & 1][ti], y[ti]);
    }
    // ---- the state: S = e^{c_n} S + B^T x' (it does not wait for y).  A chunk's addition is summed by itself: six products added to a state that is
    // hardly forgotten lost 18 x 2^-24 of it in 2048 tokens of one sign, 2 x 2^-24 this way (fp32 products one by one: 11) ----
    U4 xp[2][3];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const uint32_t* w = reinterpret_cast<const uint32_t*>(&xf[u]);
      const f32x4_t w0 = *reinterpret_cast<const f32x4_t*>(wj + 32 * u + 8 * g), w1 = *reinterpret_cast<const f32x4_t*>(wj + 32 * u + 8 * g + 4);
      float v[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) v[j] = ((j & 1) ? bf_hi(w[j >> 1]) : bf_lo(w[j >> 1])) * (j < 4 ? w0[j & 3] : w1[j & 3]);
      split8(v, xp[u]);
    }
    constexpr int W = 2 * NU < 4 ? 2 * NU : 4;                          // tiles at a time: no product waits for the one in front
    constexpr int STEPS = 2 * (2 * NU / W);
    U4 bt[2][W];
    f32x4_t add[2][W];
    auto tiles = [&](int i) __attribute__((always_inline)) {            // step i: tokens 32 (i & 1) .., tiles W (i / 2) ..
#pragma unroll
      for (int t = 0; t < W; ++t) bt[i & 1][t] = read_tr8(B, L::kLs, 32 * (i & 1) + 8 * g, 16 * (W * (i / 2) + t), i16);
    };
    auto take = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < W; ++t) s[W * j + t] = fma4(s[W * j + t], fix, add[j & 1][t]);
    };
    // tiles 1, 2 and 3 of tokens 0 .. 31 and tile 3 of tokens 32 .. 63; tiles 0 and 2 of their own 16 tokens alone: what stands beside a tile above
    // the diagonal is not multiplied by zero, so that a value that is no number stays where it is
    U4 gf[2][4];
    uint2 gh[2][2];
    auto gram = [&](int q) __attribute__((always_inline)) {
      const uint16_t* at_q = G + q * (Q * L::kGs);
#pragma unroll
      for (int f = 0; f < 4; ++f) gf[q & 1][f] = ld16(at_q + 16 * (f < 3 ? f + 1 : 3) * L::kGs + 32 * (f == 3));
#pragma unroll
      for (int f = 0; f < 2; ++f) gh[q & 1][f] = *reinterpret_cast<const uint2*>(at_q - 4 * g + 32 * f * L::kGs + 32 * f);
    };
    tiles(0);
#pragma unroll
    for (int ti = 0; ti < 4; ++ti) y[ti] *= ec[16 * ti + i16];
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
      if (i + 1 < STEPS) tiles(i + 1);
      else gram(2);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int t = 0; t < W; ++t) {
          f32x4_t& a = add[(i >> 1) & 1][t];
          a = mfma_bf(bt[i & 1][t], xp[i & 1][q], (i & 1) == 0 && q == 2 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : a);
        }
      if (i >= 2 && (i & 1) == 0) take(i / 2 - 1);                      // (the products in front have landed by now)
    }
    // ---- y += G x: a piece's six fragments are read while the piece in front is multiplied.  (Products over 32 and over 16 rows have sums of
    // their own: handed from the one to the other without an instruction in between, a sum lost what was in it.) ----
    f32x4_t y2 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 2; q >= 0; --q) {
      if (q > 0) gram(q - 1);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int f = 0; f < 4; ++f) {
        const int ti = f < 3 ? f + 1 : 3;
        y[ti] = mfma_bf(xf[f == 3], gf[q & 1][f], y[ti]);
        if (f == 0) y[0] = mfma_bf16k(xh[0], gh[q & 1][0], y[0]);
        if (f == 1) y2 = mfma_bf16k(xh[1], gh[q & 1][1], y2);
      }
      if (q == 2) take(STEPS / 2 - 1);
    }
    y[2] += y2;
    uint16_t* to = yp + static_cast<int64_t>(c0) * p.y_stride;
#pragma unroll
    for (int ti = 0; ti < 4; ++ti)
      if (16 * ti + i16 < len && 4 * g < wide)
        *reinterpret_cast<uint2*>(to + static_cast<int64_t>(16 * ti) * p.y_stride) = uint2{pack_bf2(y[ti][0], y[ti][1]), pack_bf2(y[ti][2], y[ti][3])};
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < 2 * NU; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * t + 4 * g + r;
      if (live && n < p.N) S[static_cast<int64_t>(n) * p.P] = s[t][r];
    }
}

// ------------------------------------------------------------------------------------------------ gated delta rule, 32 tokens a chunk
// The products of two fp32 operands (the inverse times the right-hand side, the read-out's matrix times U) are the products of their pieces
// but the smallest, l l, below 2^-30 of the whole: of two more, m l and l m, truncated pieces make up to 7 x 2^-24 of the product, always
// towards zero.  Rows 0 .. 15 are products over the first 16 tokens alone.  The large term h h is summed by itself: of a sum that is smaller than
// the product added to it the matrix cores cut the low bits off, 0.17 of the result's last place on average.
template <int NU>
struct DeltaSplit {
  static constexpr int kTok = 32, kNp = 32 * NU, kLs = kNp + 8, kVs = 64 + 8, kGs = kTok + 8, kAs = kTok + 4;
  uint16_t k[3][kTok * kLs], q[3][kTok * kLs];
  uint16_t v[3][kTok * kVs];
  uint16_t p[3][3][kTok * kGs];                    // (Q K^T) o decays o lengths in three pieces
  uint16_t t[2][3][kTok * kGs];                    // (I + A)^-1 in three pieces
  float a[2][kTok * kAs];                          // A transposed: row j, column i
  double cum[8][kTok];
  float ec[8][kTok], wj[8][kTok], beta[8][kTok];   // e^{c_i}, e^{c_n - c_j}
  float colf[8][2][kTok];                          // e^{c_m - c_j}, m the first token behind j's tile; m the first of j's tile
  float rowf[8][kTok];                             // e^{c_i - c_m}, m the first token of i's tile
  float ik[8][kTok], iq[8][kTok];                  // 1 / |k|, scale / |q|
  float fix[8][4];
  uint32_t count;
};

__device__ __forceinline__ f32x4_t mfma_f32(float a, float b, f32x4_t c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

template <typename Params, int NU>
__device__ __forceinline__ void delta_split_body(const Params& p, DeltaSplit<NU>& sm) {
  using L = DeltaSplit<NU>;
  constexpr int Q = L::kTok;
  // neighbours in the launch go to different XCDs: value heads of one key head lie `kv_heads` apart
  const int b = blockIdx.y, kh = blockIdx.x % p.kv_heads, h = kh * (p.heads / p.kv_heads) + blockIdx.x / p.kv_heads;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int i16 = lane & 15, g = lane >> 4;
  const int64_t tok0 = p.seg_start[b];
  const int total = p.seg_len[b];
  if (total <= 0) return;
  const int64_t pos0 = p.positions[tok0];
  const int col0 = blockIdx.z * p.col_waves * 16;
  const int chunks = (total + Q - 1) / Q;
  if (wave < kPrepWaves) {
    const int tid = threadIdx.x;
    const float a = -expf(p.A_log[h]), dtb = p.dt_bias[h];
    const uint16_t* rows0 = static_cast<const uint16_t*>(p.qkv) + tok0 * p.qkv_stride;
    const uint16_t* bp = static_cast<const uint16_t*>(p.b) + tok0 * p.ba_stride + h;
    const uint16_t* ap = static_cast<const uint16_t*>(p.a) + tok0 * p.ba_stride + h;
    RowPieces<Q, L::kNp> kr, qr;
    RowPieces<Q, 64> vr;
    kr.place(p.qkv_stride, tid);
    vr.place(p.qkv_stride, tid);
#pragma unroll
    for (int i = 0; i < kr.kPieces; ++i) qr.off[i] = kr.off[i];
    const int cols = p.V - col0 < 16 * p.col_waves ? p.V - col0 : 16 * p.col_waves;
    auto fetch = [&](int k) __attribute__((always_inline)) {
      const int c0 = k * Q, len = total - c0 < Q ? total - c0 : Q;
      const uint16_t* rows = rows0 + static_cast<int64_t>(c0) * p.qkv_stride;
      qr.fetch(rows + kh * p.K, len, p.K, tid);
      kr.fetch(rows + (p.kv_heads + kh) * p.K, len, p.K, tid);
      vr.fetch(rows + 2 * p.kv_heads * p.K + h * p.V + col0, len, cols, tid);
    };
    // 1 / sqrt(|row|^2 + 1e-6) of the rows in flight (NP / 8 neighbouring lanes hold a row): v_rsq_f32 and a Newton step; 0 for a length
    // beyond the floats, where the step would be inf * 0
    auto lengths = [&](const RowPieces<Q, L::kNp>& r, float* to, float scale) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < r.kPieces; ++i) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(&r.raw[i]);
        float ss = 0.f, st = 0.f;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float lo = bf_lo(w[j]), hi = bf_hi(w[j]);
          ss = fmaf(lo, lo, ss);
          st = fmaf(hi, hi, st);
        }
        const float n = sum_lanes<L::kNp / 8>(ss + st) + 1e-6f;
        const float y = __builtin_amdgcn_rsqf(n), e = fmaf(-n * y, y, 1.0f);
        if (r.col(i, tid) == 0 && r.row(i, tid) < Q) to[r.row(i, tid)] = n == INFINITY ? 0.f : scale * fmaf(0.5f * y, e, y);
      }
    };
    auto commit = [&](int k) __attribute__((always_inline)) {
      const int at = k % 3;
      kr.commit(sm.k[at], L::kLs, tid);
      qr.commit(sm.q[at], L::kLs, tid);
      vr.commit(sm.v[at], L::kVs, tid);
      lengths(kr, sm.ik[k & 7], 1.0f);
      lengths(qr, sm.iq[k & 7], p.q_scale);
    };
    // gates of two chunks at a time: lanes 0 - 31 chunk k, lanes 32 - 63 chunk k + 1
    uint16_t ar = 0, br = 0;
    auto fetch_gates = [&](int k) __attribute__((always_inline)) {
      if (k * Q + lane < total) {
        ar = ap[static_cast<int64_t>(k * Q + lane) * p.ba_stride];
        br = bp[static_cast<int64_t>(k * Q + lane) * p.ba_stride];
      }
    };
    auto scan = [&](int k) __attribute__((always_inline)) {
      const bool in = k * Q + lane < total;
      const float lg = in ? a * softplus_f(bf2f(ar) + dtb) : 0.f;
      const double c = scan_lanes<Q>(static_cast<double>(lg));
      const double cn = lane < Q ? lane_f64(c, Q - 1) : lane_f64(c, 2 * Q - 1), cm = lane < Q ? lane_f64(c, 16) : lane_f64(c, Q + 16);
      const double cf = (lane & 16) ? cm : lane < Q ? lane_f64(c, 0) : lane_f64(c, Q);
      const int at = (k + lane / Q) & 7, i = lane & (Q - 1);
      sm.cum[at][i] = c;
      sm.beta[at][i] = in ? sigmoid_f(bf2f(br)) : 0.f;
      sm.ec[at][i] = expf(static_cast<float>(c));
      sm.wj[at][i] = expf(static_cast<float>(cn - c));
      sm.colf[at][0][i] = i < 16 ? expf(static_cast<float>(cm - c)) : 0.f;
      sm.colf[at][1][i] = exp_f64(cf - c);                                 // (read only where it cannot overflow)
      sm.rowf[at][i] = exp_f64(c - cf);
      if (i == 0) sm.fix[at][0] = expf(static_cast<float>(cn));
    };
    // X_i . K_j over the head dim of tile (ti, tj); `turned`: a lane holds four j of one i, else four i of one j
    auto product = [&](const uint16_t* x, const uint16_t* y, bool turned, int ti, int tj) __attribute__((always_inline)) {
      const uint16_t* X = x + (16 * ti + i16) * L::kLs + 8 * g;
      const uint16_t* Y = y + (16 * tj + i16) * L::kLs + 8 * g;
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const U4 xf = ld16(X + 32 * u), yf = ld16(Y + 32 * u);
        acc = turned ? mfma_bf(yf, xf, acc) : mfma_bf(xf, yf, acc);
      }
      return acc;
    };
    // decays as in the Mamba-2 kernel, both factors from the scan; exponentials only on a diagonal tile that falls by e^60 or more
    auto put_a = [&](int k, int ti, int tj) __attribute__((always_inline)) {
      const f32x4_t acc = product(sm.k[k % 3], sm.k[k % 3], false, ti, tj);
      const int at = k & 7, j = 16 * tj + i16, i0 = 16 * ti + 4 * g;
      const bool diag = ti == tj;
      const double cj = sm.cum[at][j];
      f32x4_t v;
      if (!diag || sm.cum[at][16 * ti] - sm.cum[at][16 * ti + 15] < 60.0) {
        const float w = sm.colf[at][diag][j] * sm.ik[at][j];
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(&sm.rowf[at][i0]), be = *reinterpret_cast<const f32x4_t*>(&sm.beta[at][i0]);
        const f32x4_t n = *reinterpret_cast<const f32x4_t*>(&sm.ik[at][i0]);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[r] * (e[r] * w) * (be[r] * n[r]);
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = j < i0 + r ? acc[r] * expf(static_cast<float>(sm.cum[at][i0 + r] - cj)) * sm.beta[at][i0 + r] * sm.ik[at][i0 + r] * sm.ik[at][j] : 0.f;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (diag && j >= i0 + r) v[r] = 0.f;
      *reinterpret_cast<f32x4_t*>(&sm.a[k & 1][j * L::kAs + i0]) = v;
    };
    auto put_p = [&](int k, int ti, int tj) __attribute__((always_inline)) {
      const f32x4_t acc = product(sm.q[k % 3], sm.k[k % 3], true, ti, tj);
      const int at = k & 7, i = 16 * ti + i16, j0 = 16 * tj + 4 * g;
      const bool diag = ti == tj;
      const double ci = sm.cum[at][i];
      float v[4];
      if (!diag || sm.cum[at][16 * ti] - sm.cum[at][16 * ti + 15] < 60.0) {
        const float w = sm.rowf[at][i] * sm.iq[at][i];
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(&sm.colf[at][diag][j0]), n = *reinterpret_cast<const f32x4_t*>(&sm.ik[at][j0]);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[r] * (w * e[r]) * n[r];
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = j0 + r <= i ? acc[r] * expf(static_cast<float>(ci - sm.cum[at][j0 + r])) * sm.iq[at][i] * sm.ik[at][j0 + r] : 0.f;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (diag && j0 + r > i) v[r] = 0.f;
      uint32_t hi[4], mi[4], lo[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) split3(v[r], hi[r], mi[r], lo[r]);
      uint16_t* to = &sm.p[k % 3][0][i * L::kGs + j0];
      *reinterpret_cast<uint2*>(to) = uint2{pack_hi(hi[0], hi[1]), pack_hi(hi[2], hi[3])};
      *reinterpret_cast<uint2*>(to + Q * L::kGs) = uint2{pack_hi(mi[0], mi[1]), pack_hi(mi[2], mi[3])};
      *reinterpret_cast<uint2*>(to + 2 * Q * L::kGs) = uint2{pack_hi(lo[0], lo[1]), pack_hi(lo[2], lo[3])};
    };
    // (I + A)^-1 of chunk k by one wave: X (I + A) = I for the two 16 x 16 diagonal blocks side by side (lane = row, columns from the last),
    // x_ij = [i == j] - sum_{m > j} x_im A_mj; then the block below them, -X22 A21 X11, two small products.
    auto invert = [&](int k) __attribute__((always_inline)) {
      float* A = sm.a[k & 1];
      uint16_t* T = sm.t[k & 1][0];
      const int blk = (lane >> 4) & 1;
      const float* at = A + blk * (16 * L::kAs + 16);
      f32x4_t w[16][4];
#pragma unroll
      for (int j = 15; j >= 0; --j)
#pragma unroll
        for (int m4 = j / 4; m4 < 4; ++m4) w[j][m4] = *reinterpret_cast<const f32x4_t*>(at + j * L::kAs + 4 * m4);
      __builtin_amdgcn_sched_barrier(0);                       // (all on their way before the first is used)
      float x[16];
#pragma unroll
      for (int j = 15; j >= 0; --j) {
        float acc[2] = {i16 == j ? 1.f : 0.f, 0.f};
#pragma unroll
        for (int m4 = 3; m4 >= j / 4; --m4) {                  // (the unknown that was found last comes last)
#pragma unroll
          for (int e = 3; e >= 0; --e)
            if (4 * m4 + e > j) acc[e & 1] = fmaf(-w[j][m4][e], x[4 * m4 + e], acc[e & 1]);
        }
        x[j] = acc[0] + acc[1];
      }
      // (one wave: its LDS accesses complete in order)
      f32x4_t m = {0.f, 0.f, 0.f, 0.f}, x21 = {0.f, 0.f, 0.f, 0.f}, a21;
#pragma unroll
      for (int r = 0; r < 4; ++r) a21[r] = A[(4 * g + r) * L::kAs + 16 + i16];
      if (lane < Q) {
        float* to = A + lane * L::kAs + blk * 16;
#pragma unroll
        for (int c = 0; c < 4; ++c) *reinterpret_cast<f32x4_t*>(to + 4 * c) = f32x4_t{x[4 * c], x[4 * c + 1], x[4 * c + 2], x[4 * c + 3]};
#pragma unroll
        for (int c = 0; c < 2; ++c) {
          const float v[8] = {x[8 * c], x[8 * c + 1], x[8 * c + 2], x[8 * c + 3], x[8 * c + 4], x[8 * c + 5], x[8 * c + 6], x[8 * c + 7]};
          U4 s3[3];
          split8(v, s3);
#pragma unroll
          for (int q = 0; q < 3; ++q) {
            st16(T + q * (Q * L::kGs) + lane * L::kGs + blk * 16 + 8 * c, s3[q]);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) m = mfma_f32(a21[r], A[(4 * g + r) * L::kAs + i16], m);
      const f32x4_t x22 = *reinterpret_cast<const f32x4_t*>(A + (16 + i16) * L::kAs + 16 + 4 * g);
#pragma unroll
      for (int r = 0; r < 4; ++r) x21 = mfma_f32(m[r], -x22[r], x21);           // turned: four columns of row 16 + i16
      uint32_t hi[4], mi[4], lo[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) split3(x21[r], hi[r], mi[r], lo[r]);
      uint16_t* to = T + (16 + i16) * L::kGs + 4 * g;
      *reinterpret_cast<uint2*>(to) = uint2{pack_hi(hi[0], hi[1]), pack_hi(hi[2], hi[3])};
      *reinterpret_cast<uint2*>(to + Q * L::kGs) = uint2{pack_hi(mi[0], mi[1]), pack_hi(mi[2], mi[3])};
      *reinterpret_cast<uint2*>(to + 2 * Q * L::kGs) = uint2{pack_hi(lo[0], lo[1]), pack_hi(lo[2], lo[3])};
    };
    // Round k: rows of chunk k + 2 by all, A and the read-out's matrix of it by three waves, one of which scans the gates of chunks
    // k + 3 and k + 4 in odd rounds; the inverse of chunk k + 1 by the last.  The column waves are at chunk k.
    if (tid == 0) sm.count = 0;
    uint32_t round = 0;
    fetch(0);
    if (wave == kPrepWaves - 2) {
      fetch_gates(0);
      scan(0);
      fetch_gates(2);
    }
    __syncthreads();
    for (int k = -2; k < chunks; ++k) {
      if (k + 2 < chunks) {
        commit(k + 2);
        if (k + 3 < chunks) fetch(k + 3);
        if (wave < kPrepWaves - 1) prep_sync(&sm.count, round);
        else prep_arrive(&sm.count);
        if (wave == 0) { put_a(k + 2, 0, 0); put_a(k + 2, 1, 1); }
        else if (wave == 1) { put_a(k + 2, 1, 0); put_p(k + 2, 0, 0); }
        else if (wave == 2) { put_p(k + 2, 1, 0); put_p(k + 2, 1, 1); }
      }
      if (wave == kPrepWaves - 1) {
        if (k + 1 >= 0 && k + 1 < chunks) invert(k + 1);
      } else if (wave == kPrepWaves - 2) {
        if ((k & 1) && k + 3 < chunks) {
          scan(k + 3);
          fetch_gates(k + 5);
        }
      }
      __syncthreads();
    }
    return;
  }
  const int cw = wave - kPrepWaves, col = col0 + cw * 16 + i16;
  const bool live = col < p.V;
  float* S = p.state + (p.slots[b] * p.heads + h) * static_cast<int64_t>(p.K) * p.V + col;
  uint16_t* op = static_cast<uint16_t*>(p.o) + tok0 * p.o_stride + static_cast<int64_t>(i16) * p.o_stride + h * p.V + col0 + cw * 16 + 4 * g;
  const int wide = p.V - col0 - cw * 16;                 // the wave's columns (a multiple of 8; 16 and more: all of them)
  f32x4_t s[2 * NU];
#pragma unroll
  for (int t = 0; t < 2 * NU; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * t + 4 * g + r;
      s[t][r] = pos0 > 0 && live && n < p.K ? S[static_cast<int64_t>(n) * p.V] : 0.f;
    }
  __syncthreads();
  __syncthreads();
  __syncthreads();
  // c plus the product of two operands in pieces (the operands' type says over how many tokens)
  auto part = [](const auto& a, const auto& b, f32x4_t c) __attribute__((always_inline)) {
    if constexpr (sizeof(a) == sizeof(U4)) return mfma_bf(a, b, c);
    else return mfma_bf16k(a, b, c);
  };
  auto mul8 = [&](const auto& x, const auto& y, f32x4_t c) __attribute__((always_inline)) {
    f32x4_t a = {0.f, 0.f, 0.f, 0.f};
    a = part(x[2], y[1], a);
    a = part(x[1], y[2], a);
    a = part(x[2], y[0], a);
    c = part(x[0], y[0], c);
    a = part(x[0], y[2], a);
    a = part(x[1], y[1], a);
    a = part(x[1], y[0], a);
    a = part(x[0], y[1], a);
    return c + a;
  };
  for (int k = 0; k < chunks; ++k) {
    const int c0 = k * Q, len = total - c0 < Q ? total - c0 : Q, at = k & 7;
    const uint16_t* K = sm.k[k % 3];
    const uint16_t* Kr = K + i16 * L::kLs;
    const uint16_t* Qr = sm.q[k % 3] + i16 * L::kLs;
    const U4 vf = read_tr8<16>(sm.v[k % 3], L::kVs, 4 * g, cw * 16, i16);       // tokens 4 g + r and 16 + 4 g + r of the lane's column
    // ---- K S and (Q S)^T: the operands of k-step u + 1 are read and split while the products of step u run ----
    f32x4_t ks[2], o[2];
    U4 kf[2][2], qf[2][2], sp[2][3];
    auto stage = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int ti = 0; ti < 2; ++ti) {
        kf[u & 1][ti] = read_pair(Kr + 16 * ti * L::kLs, 32 * u, g);
        qf[u & 1][ti] = read_pair(Qr + 16 * ti * L::kLs, 32 * u, g);
      }
      const float v[8] = {s[2 * u][0], s[2 * u][1], s[2 * u][2], s[2 * u][3], s[2 * u + 1][0], s[2 * u + 1][1], s[2 * u + 1][2], s[2 * u + 1][3]};
      split8(v, sp[u & 1]);
    };
    stage(0);
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) ks[ti] = o[ti] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      if (u + 1 < NU) stage(u + 1);
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) {
          ks[ti] = mfma_bf(kf[u & 1][ti], sp[u & 1][q], ks[ti]);
          o[ti] = mfma_bf(sp[u & 1][q], qf[u & 1][ti], o[ti]);
        }
    }
    // ---- U = (I + A)^-1 beta (v - e^{c_i} K S) ----
    U4 tf[3], pf[3];
    uint2 th[3], ph[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      th[q] = *reinterpret_cast<const uint2*>(sm.t[k & 1][q] + i16 * L::kGs + 4 * g);
      tf[q] = read_pair(sm.t[k & 1][q] + (16 + i16) * L::kGs, 0, g);
    }
    float rhs[8];
    const uint32_t* vw = reinterpret_cast<const uint32_t*>(&vf);
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      const f32x4_t be = *reinterpret_cast<const f32x4_t*>(&sm.beta[at][16 * ti + 4 * g]), e = *reinterpret_cast<const f32x4_t*>(&sm.ec[at][16 * ti + 4 * g]);
      const f32x4_t ik = *reinterpret_cast<const f32x4_t*>(&sm.ik[at][16 * ti + 4 * g]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 4 * ti + r;
        const float v = (j & 1) ? bf_hi(vw[j >> 1]) : bf_lo(vw[j >> 1]);
        rhs[j] = be[r] * (v - e[r] * ik[r] * ks[ti][r]);
      }
    }
    U4 rp[3];
    split8(rhs, rp);
    f32x4_t u2[2];
    const uint2 rh[3] = {uint2{rp[0].x, rp[0].y}, uint2{rp[1].x, rp[1].y}, uint2{rp[2].x, rp[2].y}};
    u2[0] = mul8(th, rh, f32x4_t{0.f, 0.f, 0.f, 0.f});
    u2[1] = mul8(tf, rp, f32x4_t{0.f, 0.f, 0.f, 0.f});
    // ---- S = e^{c_n} S + K^T (e^{c_n - c_j} U), O^T = e^{c_i} (Q S)^T + U^T P^T ----
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      ph[q] = *reinterpret_cast<const uint2*>(sm.p[k % 3][q] + i16 * L::kGs + 4 * g);
      pf[q] = read_pair(sm.p[k % 3][q] + (16 + i16) * L::kGs, 0, g);
    }
    U4 up[3], wp[3];
    {
      float u[8], w[8];
#pragma unroll
      for (int ti = 0; ti < 2; ++ti) {
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(&sm.wj[at][16 * ti + 4 * g]), ik = *reinterpret_cast<const f32x4_t*>(&sm.ik[at][16 * ti + 4 * g]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          u[4 * ti + r] = u2[ti][r];
          w[4 * ti + r] = u2[ti][r] * (e[r] * ik[r]);
        }
      }
      split8(w, wp);
      split8(u, up);
    }
    const uint2 uh[3] = {uint2{up[0].x, up[0].y}, uint2{up[1].x, up[1].y}, uint2{up[2].x, up[2].y}};
    const float fix = sm.fix[at][0];
    constexpr int W = 2 * NU < 4 ? 2 * NU : 4;
    U4 bt[2][W];
    auto tiles = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < W; ++t) bt[i & 1][t] = read_tr8<16>(K, L::kLs, 4 * g, 16 * (W * i + t), i16);
    };
    tiles(0);
#pragma unroll
    for (int i = 0; i < 2 * NU / W; ++i) {
      if (i + 1 < 2 * NU / W) tiles(i + 1);
      f32x4_t add[W];
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int t = 0; t < W; ++t) add[t] = mfma_bf(bt[i & 1][t], wp[q], q == 2 ? f32x4_t{0.f, 0.f, 0.f, 0.f} : add[t]);
#pragma unroll
      for (int t = 0; t < W; ++t) s[W * i + t] = fma4(s[W * i + t], fix, add[t]);
    }
    uint16_t* to = op + static_cast<int64_t>(c0) * p.o_stride;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      o[ti] *= sm.ec[at][16 * ti + i16] * sm.iq[at][16 * ti + i16];
      if (ti == 0) o[0] = mul8(uh, ph, o[0]);
      else o[1] = mul8(up, pf, o[1]);
      if (16 * ti + i16 < len && 4 * g < wide)
        *reinterpret_cast<uint2*>(to + static_cast<int64_t>(16 * ti) * p.o_stride) = uint2{pack_bf2(o[ti][0], o[ti][1]), pack_bf2(o[ti][2], o[ti][3])};
    }
    __syncthreads();
  }
#pragma unroll
  for (int t = 0; t < 2 * NU; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int n = 16 * t + 4 * g + r;
      if (live && n < p.K) S[static_cast<int64_t>(n) * p.V] = s[t][r];
    }
}

}  // namespace sgl_amd
