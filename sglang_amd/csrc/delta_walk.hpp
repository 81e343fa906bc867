// The gated delta rule of recurrent_split.hpp in two launches: what does not depend on the state is formed by one wave a chunk and head, for all
// chunks of a pass at once; the walk over the chunks is left to the waves that hold the state.
//
// In one launch (delta_split_body) a chunk's preparation stands beside the walk: its inverse is a chain as long as a chunk's walk, and a SIMD's two
// waves share its issue slots (6100 clocks a chunk beside each other, the walk alone 4800).  What bounds the walk is what one wave issues, an instruction in
// five clocks at best: 720 of them there, 560 here (3800 clocks), where the preparation leaves the factors already multiplied and the operands in the order
// in which a lane reads them, the images need no address arithmetic and requests are a wave's of their own.  The two launches pay 10 KiB a chunk and head
// through the caches: the first takes 15 to 20 us for 4 500 tokens and 32 heads.
// Measured (us, one launch / two; 32 heads of 128 x 128): 3 segments of 1.3 - 1.9 k tokens 163 / 134, 1500 tokens 119 / 97, 4 of 1.6 - 2.5 k 225 / 195,
// 6 of 1.1 - 1.7 k 258 / 200, 16 of 410 - 610 223 / 171.
// (Taken back: two waves a column group, half of the state's rows each, partial products handed over in LDS: 143 us for the walk against 118, each of the
// eight waves reads what the four read.)
#pragma once

#include "recurrent_split.hpp"

namespace sgl_amd {

// One chunk of one head, as the walk's lanes read it (lane = (i = lane & 15, g = lane / 16), three pieces each): rows i of the inverse T and of the
// read-out's matrix P at 4 g .. + 3; rows 16 + i at 4 g .. + 3 and at 16 + 4 g .. + 3.  Then per token beta, e^{c_i} / |k|, e^{c_n - c_i} / |k| and
// e^{c_i} scale / |q|, the chunk's e^{c_n}, and zeros for rows that there are not.
struct DeltaUnit {
  uint2 t_top[3][64], p_top[3][64];
  U4 t_low[3][64], p_low[3][64];
  float beta[32], fall_k[32], add_k[32], out_q[32];
  float fix[4];
  U4 zero[30];
  U4 unused;
};
static_assert(sizeof(DeltaUnit) == 10240, "ten requests of 1 KiB");

// chunks of the segments in front of segment b (every lane of the wave calls it)
__device__ __forceinline__ int64_t delta_units_before(const int32_t* seg_len, int b, int lane) {
  int n = 0;
  for (int i = lane; i < b; i += 64) n += (max(seg_len[i], 0) + 31) / 32;
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) n += __shfl_xor(n, d, 64);
  return __builtin_amdgcn_readfirstlane(n);
}

struct DeltaPrep {
  static constexpr int kAs = 32 + 4;
  float a[32 * kAs];                               // A transposed: row j, column i; then the inverse of its diagonal blocks, row by row
  double cum[32];
  float beta[32], colf[2][32], rowf[32], ik[32], iq[32];
};

// What one lane left in LDS, for the other lanes of the wave: its accesses are done in order, the compiler keeps them so.
__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// One wave a chunk and head, four heads a workgroup (one a workgroup: 7 us more for 5 700 of them).
constexpr int kDeltaPrepWaves = 4;
template <typename Params, int NU>
__device__ __forceinline__ void delta_prepare_body(const Params& p, DeltaPrep& sm) {
  constexpr int Q = 32, kAs = DeltaPrep::kAs;
  const int b = blockIdx.z, h = blockIdx.x * kDeltaPrepWaves + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), kh = h / (p.heads / p.kv_heads);
  if (h >= p.heads) return;
  const int total = p.seg_len[b];
  const int chunks = (total + Q - 1) / Q;
  if (static_cast<int>(blockIdx.y) >= chunks) return;
  const int64_t tok0 = p.seg_start[b], first = delta_units_before(p.seg_len, b, threadIdx.x & 63);
  if (first + chunks > p.units) {                // more tokens than the caller said: the walk leaves the segment out, and nobody takes its outputs for results
    uint16_t* o = static_cast<uint16_t*>(p.o) + tok0 * p.o_stride + h * p.V;
    for (int k = blockIdx.y; k < chunks; k += gridDim.y)
      for (int t = k * Q; t < total && t < (k + 1) * Q; ++t)
        for (int v = threadIdx.x & 63; v < p.V; v += 64) o[t * p.o_stride + v] = 0x7fc0;
    return;
  }
  const float a = -expf(p.A_log[h]), dtb = p.dt_bias[h];
  for (int k = blockIdx.y; k < chunks; k += gridDim.y) {       // (once, but for segments beyond two million tokens)
    int lane = threadIdx.x & 63;
    asm volatile("" : "+v"(lane));                              // (nothing of it is kept across the loop)
    const int i16 = lane & 15, g = lane >> 4;
    const int c0 = k * Q, len = total - c0 < Q ? total - c0 : Q, i = lane & (Q - 1);
    const bool in = i < len;
    const uint16_t* rows = static_cast<const uint16_t*>(p.qkv) + (tok0 + c0) * p.qkv_stride;
    uint16_t ar = 0, br = 0;
    if (in) {
      ar = static_cast<const uint16_t*>(p.a)[(tok0 + c0 + i) * p.ba_stride + h];
      br = static_cast<const uint16_t*>(p.b)[(tok0 + c0 + i) * p.ba_stride + h];
    }
    U4 kf[2][NU], qf[2][NU];
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      const uint16_t* at = rows + (16 * ti + i16) * p.qkv_stride + kh * p.K + 8 * g;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const bool ok = 16 * ti + i16 < len && 32 * u + 8 * g < p.K;
        kf[ti][u] = qf[ti][u] = U4{0u, 0u, 0u, 0u};
        if (ok) {
          kf[ti][u] = ld16(at + p.kv_heads * p.K + 32 * u);
          qf[ti][u] = ld16(at + 32 * u);
        }
      }
    }
    // ---- the gates (both halves of the wave hold token i's) ----
    const double c = scan_lanes<Q>(static_cast<double>(in ? a * softplus_f(bf2f(ar) + dtb) : 0.f));
    const double c_first = lane_f64(c, 0), c_mid = lane_f64(c, 15), cm = lane_f64(c, 16), cn = lane_f64(c, Q - 1), cf = (lane & 16) ? cm : c_first;
    const bool near0 = c_first - c_mid < 60.0, near1 = cm - cn < 60.0;           // (the diagonal tiles' decays as products of two factors: recurrent_split.hpp)
    const float beta = in ? sigmoid_f(bf2f(br)) : 0.f, ec = expf(static_cast<float>(c)), wj = expf(static_cast<float>(cn - c));
    sm.cum[i] = c;
    sm.beta[i] = beta;
    sm.colf[0][i] = i < 16 ? expf(static_cast<float>(cm - c)) : 0.f;
    sm.colf[1][i] = exp_f64(cf - c);                                 // (read only where it cannot overflow)
    sm.rowf[i] = exp_f64(c - cf);
    // ---- 1 / sqrt(|row|^2 + 1e-6): v_rsq_f32 and a Newton step; 0 for a length beyond the floats, where the step would be inf * 0 ----
    auto length = [&](const U4 (&f)[NU], float scale) __attribute__((always_inline)) {
      float ss = 0.f, st = 0.f;
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(&f[u]);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float lo = bf_lo(w[j]), hi = bf_hi(w[j]);
          ss = fmaf(lo, lo, ss);
          st = fmaf(hi, hi, st);
        }
      }
      ss += st;
      ss += __shfl_xor(ss, 16, 64);
      ss += __shfl_xor(ss, 32, 64);
      const float n = ss + 1e-6f, y = __builtin_amdgcn_rsqf(n), e = fmaf(-n * y, y, 1.0f);
      return n == INFINITY ? 0.f : scale * fmaf(0.5f * y, e, y);
    };
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      sm.ik[16 * ti + i16] = length(kf[ti], 1.0f);
      sm.iq[16 * ti + i16] = length(qf[ti], p.q_scale);
    }
    wave_sync();
    DeltaUnit* unit = static_cast<DeltaUnit*>(p.ws) + (first + k) * p.heads + h;
    if (lane < Q) {
      unit->beta[i] = beta;
      unit->fall_k[i] = ec * sm.ik[i];
      unit->add_k[i] = wj * sm.ik[i];
      unit->out_q[i] = ec * sm.iq[i];
      if (lane == 0) unit->fix[0] = expf(static_cast<float>(cn));
      if (lane < 30) unit->zero[lane] = U4{0u, 0u, 0u, 0u};
    }
    // ---- A, transposed (a lane holds four i of one j) ----
    auto put_a = [&](auto ti_c, auto tj_c) __attribute__((always_inline)) {
      constexpr int ti = decltype(ti_c)::value, tj = decltype(tj_c)::value;
      constexpr bool diag = ti == tj;
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f}, v;
#pragma unroll
      for (int u = 0; u < NU; ++u) acc = mfma_bf(kf[ti][u], kf[tj][u], acc);
      const int j = 16 * tj + i16, i0 = 16 * ti + 4 * g;
      if (!diag || (ti == 0 ? near0 : near1)) {
        const float w = sm.colf[diag][j] * sm.ik[j];
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(&sm.rowf[i0]), be = *reinterpret_cast<const f32x4_t*>(&sm.beta[i0]);
        const f32x4_t n = *reinterpret_cast<const f32x4_t*>(&sm.ik[i0]);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[r] * (e[r] * w) * (be[r] * n[r]);
      } else {
        const double cj = sm.cum[j];
#pragma unroll
        for (int r = 0; r < 4; ++r)
          v[r] = j < i0 + r ? acc[r] * expf(static_cast<float>(sm.cum[i0 + r] - cj)) * sm.beta[i0 + r] * sm.ik[i0 + r] * sm.ik[j] : 0.f;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (diag && j >= i0 + r) v[r] = 0.f;
      *reinterpret_cast<f32x4_t*>(&sm.a[j * kAs + i0]) = v;
    };
    // ---- P (a lane holds four j of one i: what the walk's lane reads) ----
    auto pieces4 = [&](const float (&v)[4], uint2 (&o)[3]) __attribute__((always_inline)) {
      uint32_t hi[4], mi[4], lo[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) split3(v[r], hi[r], mi[r], lo[r]);
      o[0] = uint2{pack_hi(hi[0], hi[1]), pack_hi(hi[2], hi[3])};
      o[1] = uint2{pack_hi(mi[0], mi[1]), pack_hi(mi[2], mi[3])};
      o[2] = uint2{pack_hi(lo[0], lo[1]), pack_hi(lo[2], lo[3])};
    };
    auto make_p = [&](auto ti_c, auto tj_c, uint2 (&o)[3]) __attribute__((always_inline)) {
      constexpr int ti = decltype(ti_c)::value, tj = decltype(tj_c)::value;
      constexpr bool diag = ti == tj;
      f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int u = 0; u < NU; ++u) acc = mfma_bf(kf[tj][u], qf[ti][u], acc);
      const int i = 16 * ti + i16, j0 = 16 * tj + 4 * g;
      float v[4];
      if (!diag || (ti == 0 ? near0 : near1)) {
        const float w = sm.rowf[i] * sm.iq[i];
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(&sm.colf[diag][j0]), n = *reinterpret_cast<const f32x4_t*>(&sm.ik[j0]);
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = acc[r] * (w * e[r]) * n[r];
      } else {
        const double ci = sm.cum[i];
#pragma unroll
        for (int r = 0; r < 4; ++r) v[r] = j0 + r <= i ? acc[r] * expf(static_cast<float>(ci - sm.cum[j0 + r])) * sm.iq[i] * sm.ik[j0 + r] : 0.f;
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (diag && j0 + r > i) v[r] = 0.f;
      pieces4(v, o);
    };
    constexpr std::integral_constant<int, 0> c0_{};
    constexpr std::integral_constant<int, 1> c1_{};
    put_a(c0_, c0_);
    put_a(c1_, c0_);
    put_a(c1_, c1_);
    {
      uint2 o[3], o1[3];
      make_p(c0_, c0_, o);
#pragma unroll
      for (int q = 0; q < 3; ++q) unit->p_top[q][lane] = o[q];
      make_p(c1_, c0_, o);
      make_p(c1_, c1_, o1);
#pragma unroll
      for (int q = 0; q < 3; ++q) unit->p_low[q][lane] = U4{o[q].x, o[q].y, o1[q].x, o1[q].y};
    }
    wave_sync();
    // ---- (I + A)^-1: X (I + A) = I for the two 16 x 16 diagonal blocks side by side (lane = row, columns from the last),
    // x_ij = [i == j] - sum_{m > j} x_im A_mj; then the block below them, -X22 A21 X11, two small products ----
    const int blk = g & 1;
    const float* at = sm.a + blk * (16 * kAs + 16);
    float x[16];
#pragma unroll
    for (int j = 15; j >= 0; --j) {
      float acc[2] = {i16 == j ? 1.f : 0.f, 0.f};
#pragma unroll
      for (int m4 = 3; m4 >= j / 4; --m4) {                  // (the unknown that was found last comes last)
        const f32x4_t w = *reinterpret_cast<const f32x4_t*>(at + j * kAs + 4 * m4);
#pragma unroll
        for (int e = 3; e >= 0; --e)
          if (4 * m4 + e > j) acc[e & 1] = fmaf(-w[e], x[4 * m4 + e], acc[e & 1]);
      }
      x[j] = acc[0] + acc[1];
      if (j % 4 == 0) asm volatile("" : "+v"(x[j]) : : "memory");   // (all 40 pieces read at once would take the registers of two more waves a SIMD)
    }
    float a21[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) a21[r] = sm.a[(4 * g + r) * kAs + 16 + i16];
    wave_sync();
    if (lane < Q) {
      float* to = sm.a + lane * kAs + blk * 16;
#pragma unroll
      for (int e = 0; e < 4; ++e) *reinterpret_cast<f32x4_t*>(to + 4 * e) = f32x4_t{x[4 * e], x[4 * e + 1], x[4 * e + 2], x[4 * e + 3]};
    }
    wave_sync();
    f32x4_t m = {0.f, 0.f, 0.f, 0.f}, x21 = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) m = mfma_f32(a21[r], sm.a[(4 * g + r) * kAs + i16], m);
    const f32x4_t x11 = *reinterpret_cast<const f32x4_t*>(&sm.a[i16 * kAs + 4 * g]);
    const f32x4_t x22 = *reinterpret_cast<const f32x4_t*>(&sm.a[(16 + i16) * kAs + 16 + 4 * g]);
#pragma unroll
    for (int r = 0; r < 4; ++r) x21 = mfma_f32(m[r], -x22[r], x21);           // turned: four columns of row 16 + i16
    uint2 o[3], o1[3];
    pieces4({x11[0], x11[1], x11[2], x11[3]}, o);
#pragma unroll
    for (int q = 0; q < 3; ++q) unit->t_top[q][lane] = o[q];
    pieces4({x21[0], x21[1], x21[2], x21[3]}, o);
    pieces4({x22[0], x22[1], x22[2], x22[3]}, o1);
#pragma unroll
    for (int q = 0; q < 3; ++q) unit->t_low[q][lane] = U4{o[q].x, o[q].y, o1[q].x, o1[q].y};
    wave_sync();
  }
}

// Two stages of a chunk's rows and unit in LDS, filled by requests of a wave of their own while the others walk the other stage.
template <int NU>
struct DeltaWalk {
  static constexpr int kRow = 64 * NU;             // bytes of a K or Q row
  static constexpr int kSlots = 4 * NU;            // its 16-byte pieces
  U4 k[32 * kSlots], q[32 * kSlots];               // [token][piece ^ swz]
  U4 v[32 * 8];                                    // [token][piece ^ (token & 2)], 64 columns
  DeltaUnit unit;
  // A 16-byte read takes tokens 0 - 3 and 12 - 15 at one piece together with tokens 4 - 11 at the next (measured: 4.4 clocks where these 16 lie in different
  // slots of the 256 bytes of banks, 8.3 with t >> 2 in the place of `hi`), a transposing one four tokens 4 n .. 4 n + 3 at four neighbouring pieces
  __device__ __forceinline__ static int swz(int t) {
    const int hi = (t & 4) >> 1 ^ (t >> 3 & 1) * 3;
    return NU == 4 ? (t & 3) << 2 | hi : NU == 2 ? (t & 2) << 1 | hi : hi;
  }
};

// 16 bytes a lane from memory to 1 KiB of LDS at `to`; the issuing wave waits (vmcnt) in front of the barrier behind which they are read.
// (Nothing else here may use M0, which cannot be named as overwritten: test_no_spills.py looks for it in the listing.)
__device__ __forceinline__ void piece_to_lds(const void* from, uint32_t to) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(from), "s"(to) : "memory");
}
__device__ __forceinline__ const unsigned char* wave_pointer(const void* from) {      // (what is the same for all lanes, in scalar registers)
  const uint64_t a = reinterpret_cast<uint64_t>(from);
  const uint32_t lo = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a)), hi = __builtin_amdgcn_readfirstlane(static_cast<uint32_t>(a >> 32));
  return reinterpret_cast<const unsigned char*>(static_cast<uint64_t>(hi) << 32 | lo);
}
__device__ __forceinline__ void piece_to_lds(const unsigned char* from, uint32_t lane_offset, uint32_t to) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_offset), "s"(from), "s"(to) : "memory");
}
__device__ __forceinline__ uint32_t lds_offset(const void* at) {
  typedef __attribute__((address_space(3))) const void* lds_t;
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_t)(at)));
}

// The walk: wave 0 fetches, each of the others holds 16 value columns of the state.  SELF: the four waves with columns fetch as well, a fourth of the pieces
// each, so that two workgroups, two waves a SIMD, share a compute unit where there are more than one for each.  Tile t = 2 u + w of the state holds its rows
// 32 u + 8 (m / 4) + 4 w + m % 4, m = 0 .. 15, so that a lane's eight state values of k-step u stand against eight neighbouring elements of a K or Q row.
template <typename Params, int NU, bool SELF>
__device__ __forceinline__ void delta_walk_body(const Params& p, DeltaWalk<NU> (&sm)[2]) {
  using L = DeltaWalk<NU>;
  constexpr int Q = 32;
  const int b = blockIdx.y, kh = blockIdx.x % p.kv_heads, h = kh * (p.heads / p.kv_heads) + blockIdx.x / p.kv_heads;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int i16 = lane & 15, g = lane >> 4;
  const int64_t tok0 = p.seg_start[b];
  const int total = p.seg_len[b];
  if (total <= 0) return;
  const int chunks = (total + Q - 1) / Q;
  const int col0 = blockIdx.z * p.col_waves * 16;
  const int64_t first = delta_units_before(p.seg_len, b, lane);
  if (first + chunks > p.units) return;
  const DeltaUnit* units = static_cast<const DeltaUnit*>(p.ws) + first * p.heads + h;
  const uint16_t* rows0 = static_cast<const uint16_t*>(p.qkv) + tok0 * p.qkv_stride;
  const int cols = p.V - col0 < 16 * p.col_waves ? p.V - col0 : 16 * p.col_waves;
  // ---- requests: pieces `by`, `by` + EACH, .. of a chunk's rows and unit.  (A full chunk: the lanes' offsets stand, the addresses of rows and unit are the
  // wave's; otherwise every piece is looked at, and one that there is not is read from the unit's zeros.) ----
  constexpr int EACH = SELF ? 4 : 1, KP = 2 * NU / EACH > 0 ? 2 * NU / EACH : 1, VP = 4 / EACH;
  const int by = SELF ? wave : 0;
  uint32_t at_k[KP], at_v[VP];
  auto k_col = [&](int j) __attribute__((always_inline)) { return (((64 * j + lane) % L::kSlots) ^ L::swz((64 * j + lane) / L::kSlots)) * 8; };
  auto v_col = [&](int j) __attribute__((always_inline)) { return ((lane % 8) ^ ((8 * j + lane / 8) & 2)) * 8; };
  if (SELF || wave == 0) {
#pragma unroll
    for (int i = 0; i < KP; ++i) {
      const int j = by + EACH * i;
      at_k[i] = static_cast<uint32_t>(((64 * j + lane) / L::kSlots * static_cast<int>(p.qkv_stride) + kh * p.K + k_col(j)) * 2);
    }
#pragma unroll
    for (int i = 0; i < VP; ++i) {
      const int j = by + EACH * i;
      at_v[i] = static_cast<uint32_t>(((8 * j + lane / 8) * static_cast<int>(p.qkv_stride) + 2 * p.kv_heads * p.K + h * p.V + col0 + v_col(j)) * 2);
    }
  }
  const bool whole = p.K == 32 * NU && cols == 64;
  auto request = [&](int k, const L& to) __attribute__((always_inline)) {
    const int c0 = k * Q, len = total - c0 < Q ? total - c0 : Q;
    const unsigned char* rows = wave_pointer(rows0 + static_cast<int64_t>(c0) * p.qkv_stride);
    const unsigned char* unit = wave_pointer(units + static_cast<int64_t>(k) * p.heads);
#pragma unroll
    for (int i = 0; i < (10 + EACH - 1) / EACH; ++i)
      if (by + EACH * i < 10) piece_to_lds(unit + 1024 * (by + EACH * i), 16u * lane, lds_offset(&to.unit) + 1024 * (by + EACH * i));
    if (whole && len == Q) {
      const unsigned char* keys = rows + p.kv_heads * p.K * 2;
#pragma unroll
      for (int i = 0; i < KP; ++i) {
        const int j = by + EACH * i;
        if (j >= 2 * NU) break;
        piece_to_lds(keys, at_k[i], lds_offset(to.k) + 1024 * j);
        piece_to_lds(rows, at_k[i], lds_offset(to.q) + 1024 * j);
      }
#pragma unroll
      for (int i = 0; i < VP; ++i) piece_to_lds(rows, at_v[i], lds_offset(to.v) + 1024 * (by + EACH * i));
    } else {
      const unsigned char* zero = unit + offsetof(DeltaUnit, zero);
#pragma unroll
      for (int i = 0; i < KP; ++i) {
        const int j = by + EACH * i;
        if (j >= 2 * NU) break;
        const unsigned char* at = rows + at_k[i];
        const bool ok = (64 * j + lane) / L::kSlots < len && k_col(j) < p.K;
        piece_to_lds(ok ? at + p.kv_heads * p.K * 2 : zero, lds_offset(to.k) + 1024 * j);
        piece_to_lds(ok ? at : zero, lds_offset(to.q) + 1024 * j);
      }
#pragma unroll
      for (int i = 0; i < VP; ++i) {
        const int j = by + EACH * i;
        const unsigned char* at = rows + at_v[i];
        piece_to_lds(8 * j + lane / 8 < len && v_col(j) < cols ? at : zero, lds_offset(to.v) + 1024 * j);
      }
    }
  };
  auto landed = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); };
  if (SELF) request(0, sm[0]);
  if (!SELF && wave == 0) {
    request(0, sm[0]);
    landed();
    __syncthreads();
    for (int k = 0; k < chunks; ++k) {
      if (k + 1 < chunks) request(k + 1, sm[(k + 1) & 1]);
      landed();
      __syncthreads();
    }
    return;
  }
  const int cw = SELF ? wave : wave - 1, col = col0 + cw * 16 + i16;
  const bool live = col < p.V;
  const int64_t pos0 = p.positions[tok0];
  float* S = p.state + (p.slots[b] * p.heads + h) * static_cast<int64_t>(p.K) * p.V + col;
  uint16_t* op = static_cast<uint16_t*>(p.o) + tok0 * p.o_stride + static_cast<int64_t>(i16) * p.o_stride + h * p.V + col0 + cw * 16 + 4 * g;
  const int wide = p.V - col0 - cw * 16;                 // the wave's columns (a multiple of 8; 16 and more: all of them)
  auto row_of = [&](int t, int r) __attribute__((always_inline)) { return 32 * (t / 2) + 8 * g + 4 * (t & 1) + r; };
  f32x4_t s[2 * NU];
#pragma unroll
  for (int t = 0; t < 2 * NU; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r) s[t][r] = pos0 > 0 && live && row_of(t, r) < p.K ? S[static_cast<int64_t>(row_of(t, r)) * p.V] : 0.f;
  // lanes' places in the images: row operands (token i), transposed ones (tokens 4 g + i / 4), values
  int at_row[NU], at_tr[NU];
  {
    const int t = 4 * g + (i16 >> 2);
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      at_row[u] = i16 * L::kRow + ((4 * u + g) ^ L::swz(i16)) * 16;
      at_tr[u] = t * L::kRow + ((4 * u + (i16 & 3)) ^ L::swz(t)) * 16;
    }
  }
  const int at_val = (4 * g + (i16 >> 2)) * 128 + ((2 * cw + ((i16 & 3) >> 1)) ^ ((i16 >> 2) & 2)) * 16 + (i16 & 1) * 8;
  auto read_tr = [&](const void* image, int at, int gap) __attribute__((always_inline)) {       // rows t and t + 16 of the lane's 8 bytes
    typedef __attribute__((address_space(3))) split_v4s16_t* lds_t;
    const unsigned char* a = static_cast<const unsigned char*>(image) + at;
    const split_v4s16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(a));
    const split_v4s16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_t)(a + gap));
    const uint2 l = __builtin_bit_cast(uint2, lo), m = __builtin_bit_cast(uint2, hi);
    return U4{l.x, l.y, m.x, m.y};
  };
  // c plus the product of two operands in pieces (the operands' type says over how many tokens)
  auto part = [](const auto& a, const auto& b, f32x4_t c) __attribute__((always_inline)) {
    if constexpr (sizeof(a) == sizeof(U4)) return mfma_bf(a, b, c);
    else return mfma_bf16k(a, b, c);
  };
  auto mul8 = [&](const auto& x, const auto& y, f32x4_t c) __attribute__((always_inline)) {       // (which terms, and why: recurrent_split.hpp)
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
  auto chunk = [&](int k, const L& at, const L& next) __attribute__((always_inline)) {
    if (SELF && k + 1 < chunks) request(k + 1, next);
    const int c0 = k * Q, len = total - c0 < Q ? total - c0 : Q;
    const DeltaUnit& un = at.unit;
    const unsigned char* K = reinterpret_cast<const unsigned char*>(at.k);
    const unsigned char* Qi = reinterpret_cast<const unsigned char*>(at.q);
    const U4 vf = read_tr(at.v, at_val, 16 * 128);         // tokens 4 g + r and 16 + 4 g + r of the lane's column
    // ---- K S: the operands of k-step u + 1 are read and split while the products of step u run ((Q S)^T fills what waits behind it: 118 -> 110 us) ----
    f32x4_t ks[2], o[2];
    U4 kf[2][2], qf[NU][2], sp[NU][3];
    auto stage = [&](int u) __attribute__((always_inline)) {
#pragma unroll
      for (int ti = 0; ti < 2; ++ti) {
        kf[u & 1][ti] = *reinterpret_cast<const U4*>(K + at_row[u] + 16 * ti * L::kRow);
      }
      const float v[8] = {s[2 * u][0], s[2 * u][1], s[2 * u][2], s[2 * u][3], s[2 * u + 1][0], s[2 * u + 1][1], s[2 * u + 1][2], s[2 * u + 1][3]};
      split8(v, sp[u]);
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
          ks[ti] = mfma_bf(kf[u & 1][ti], sp[u][q], ks[ti]);
        }
    }
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int ti = 0; ti < 2; ++ti) qf[u][ti] = *reinterpret_cast<const U4*>(Qi + at_row[u] + 16 * ti * L::kRow);
    // ---- U = (I + A)^-1 beta (v - e^{c_i} K S) ----
    uint2 th[3];
    U4 tf[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      th[q] = un.t_top[q][lane];
      tf[q] = un.t_low[q][lane];
    }
    float rhs[8];
    const uint32_t* vw = reinterpret_cast<const uint32_t*>(&vf);
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      const f32x4_t be = *reinterpret_cast<const f32x4_t*>(&un.beta[16 * ti + 4 * g]), fk = *reinterpret_cast<const f32x4_t*>(&un.fall_k[16 * ti + 4 * g]);
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int j = 4 * ti + r;
        rhs[j] = be[r] * fmaf(-fk[r], ks[ti][r], (j & 1) ? bf_hi(vw[j >> 1]) : bf_lo(vw[j >> 1]));
      }
    }
    U4 rp[3];
    split8(rhs, rp);
#pragma unroll
    for (int u = 0; u < NU; ++u)
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int ti = 0; ti < 2; ++ti) o[ti] = mfma_bf(sp[u][q], qf[u][ti], o[ti]);
    f32x4_t u2[2];
    const uint2 rh[3] = {uint2{rp[0].x, rp[0].y}, uint2{rp[1].x, rp[1].y}, uint2{rp[2].x, rp[2].y}};
    u2[0] = mul8(th, rh, f32x4_t{0.f, 0.f, 0.f, 0.f});
    u2[1] = mul8(tf, rp, f32x4_t{0.f, 0.f, 0.f, 0.f});
    // ---- S = e^{c_n} S + K^T (e^{c_n - c_j} U), O^T = e^{c_i} (Q S)^T + U^T P^T ----
    uint2 ph[3];
    U4 pf[3], up[3], wp[3];
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      ph[q] = un.p_top[q][lane];
      pf[q] = un.p_low[q][lane];
    }
    {
      float u[8], w[8];
#pragma unroll
      for (int ti = 0; ti < 2; ++ti) {
        const f32x4_t e = *reinterpret_cast<const f32x4_t*>(&un.add_k[16 * ti + 4 * g]);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          u[4 * ti + r] = u2[ti][r];
          w[4 * ti + r] = u2[ti][r] * e[r];
        }
      }
      split8(w, wp);
      split8(u, up);
    }
    const uint2 uh[3] = {uint2{up[0].x, up[0].y}, uint2{up[1].x, up[1].y}, uint2{up[2].x, up[2].y}};
    const float fix = un.fix[0];
    constexpr int W = 2 * NU < 4 ? 2 * NU : 4;
    U4 bt[2][W];
    auto tiles = [&](int i) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < W; ++t) bt[i & 1][t] = read_tr(K, at_tr[(W * i + t) / 2] + 8 * (t & 1), 16 * L::kRow);
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
    if (SELF) landed();                                  // (in front of this chunk's stores, which count too)
    uint16_t* to = op + static_cast<int64_t>(c0) * p.o_stride;
#pragma unroll
    for (int ti = 0; ti < 2; ++ti) {
      o[ti] *= un.out_q[16 * ti + i16];
      if (ti == 0) o[0] = mul8(uh, ph, o[0]);
      else o[1] = mul8(up, pf, o[1]);
      if (16 * ti + i16 < len && 4 * g < wide)
        *reinterpret_cast<uint2*>(to + static_cast<int64_t>(16 * ti) * p.o_stride) = uint2{pack_bf2(o[ti][0], o[ti][1]), pack_bf2(o[ti][2], o[ti][3])};
    }
    __syncthreads();
  };
  if (SELF) landed();
  __syncthreads();
  for (int k = 0; k < chunks; k += 2) {
    chunk(k, sm[0], sm[1]);
    if (k + 1 < chunks) chunk(k + 1, sm[1], sm[0]);
  }
#pragma unroll
  for (int t = 0; t < 2 * NU; ++t)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      if (live && row_of(t, r) < p.K) S[static_cast<int64_t>(row_of(t, r)) * p.V] = s[t][r];
}

}  // namespace sgl_amd
