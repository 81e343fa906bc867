// Ragged extend (prefill) attention over the paged token->KV pool, gfx950 MFMA.
//
// Replaces (reference, /root/reference/python/sglang):
//   kernels/ops/attention/extend_attention.py:304 _fwd_kernel, :753 extend_attention_fwd
// Oracle: srt/layers/attention/torch_native_backend.py:61-174, 279-336 -- the
// new K/V rows are written to the pool first, then every query token attends
// causally over req_to_token[req, 0:prefix+i+1].
//
// Structure (one workgroup = 4 waves = 128 "rows"):
//   * a row is a (query token, q head inside the GQA group) pair, so all
//     H_q/H_kv heads that share a kv head share ONE staged K/V tile (GQA reuse
//     in LDS instead of L2); each wave owns 32 rows = 2 MFMA M-tiles;
//   * a KV tile is 64 cached tokens.  Rows of the pool are gathered through
//     req_to_token with 16-byte loads, D/8 adjacent lanes per row, so every
//     gathered row is one fully coalesced D*2-byte read;
//   * K goes to LDS row-major with an XOR swizzle of the 16-byte chunks;
//     V is transposed on the way in (8x8 bf16 blocks transposed in registers,
//     written as 16-byte chunks of V^T) with the token order inside a chunk
//     chosen so the PV operand is a single ds_read_b128;
//   * both contractions run transposed on v_mfma_f32_16x16x32_bf16:
//         S^T = K . Q^T      O^T = V^T . P^T
//     which leaves every lane owning exactly one row per M-tile: running max,
//     running sum and the rescale factor never cross lanes, and the exp'd
//     S^T registers ARE the P^T operand of the second MFMA (no LDS round trip);
//   * fp32 accumulation, exp2 with the softmax scale folded in, bf16 output.
#include <type_traits>

#include "common.hpp"
#include "kv_format.hpp"
#include "sglang_amd.h"

using namespace sgl_amd;

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kStagers = 256;     // threads that gather K/V tiles (waves 0-1: V, waves 2-3: K)
constexpr int kRows = 128;      // rows per workgroup with two 16-row M-tiles per wave (64 with one)
constexpr int kKvTile = 64;     // cached tokens per tile
constexpr float kNegBig = -1.0e30f;

__device__ __forceinline__ bf16x8_t as_frag(const U4& v) { return __builtin_bit_cast(bf16x8_t, v); }

struct ExtendParams {
  const uint16_t* q;            // [T, Hq, D]
  uint16_t* out;                // [T, Hq, D]
  const uint16_t* k_cache;      // [slots, Hkv, D]
  const uint16_t* v_cache;
  const int32_t* req_to_token;  // [reqs, max_ctx]
  const int64_t* req_pool_indices;  // [B]
  const int32_t* seq_lens;      // [B] prefix + extend
  const int32_t* prefix_lens;   // [B]
  const int32_t* qo_indptr;     // [B+1] start of each request's query tokens
  int64_t q_stride, out_stride, kc_stride, vc_stride, r2t_stride;
  int num_kv_heads;
  int group;                    // q heads per kv head
  int tokens_per_tile;          // kRows / group
  int causal;
  float scale_log2;
  KvFormat fmt;                 // layout + element format of the pool rows
  float v_scale;                // fp8 rows: multiplied into the output (k_scale is folded into scale_log2)
  int window;                   // sliding window: kv position >= q position - window (extend_attention.py:480-485); < 0: off
  float cap_log2, inv_cap_log2; // logit soft cap (extend_attention.py:546-547), 0: off
  // custom mask (speculative-decoding verify, triton_backend.py:860-919; extend_attention.py USE_CUSTOM_MASK):
  // request b's [extend_len, kv_len] row-major uint8 mask starts at custom_mask + mask_indptr[b]; it REPLACES the
  // causal rule on the extend part and is AND-ed with "inside the prefix" on the prefix part
  const uint8_t* custom_mask;
  const int64_t* mask_indptr;
  int mask_skip_prefix;         // the prefix part of the mask is not consulted (extend_attention.py:774 skip_prefix_custom_mask)
  int num_tiles, batch;         // the double-buffered kernel's 1-D grid: query tiles per request, requests
  // keys split over workgroups (extend_attention_parts_kernel): part i's unnormalised fp32 rows [num_tokens, Hq, D] and (maximum, sum)
  int parts;
  int64_t part_rows;            // num_tokens * Hq
  float* part_acc;
  float* part_ml;
  unsigned* grabbed;            // extend_attention_walk_kernel: tiles taken so far, per XCD
};

template <int D>
struct Smem {
  U4 k[kKvTile * D / 8];        // [token][chunk ^ swz]
  U4 vt[D * kKvTile / 8];       // [d][token-chunk ^ swz]
};

// MTW = 16-row M-tiles per wave: 2 shares every staged K/V tile between 128 rows (fewest gathers per flop) at
// ~256 VGPRs = one workgroup per CU; 1 halves the rows per workgroup at ~130 VGPRs = three workgroups per CU
// (head dim 64; at 128 the 170-register budget of three workgroups spilled 16 registers inside the tile loop: two),
// whose waves cover each other's barrier, softmax and gather stalls.
// NWV = waves per workgroup: 8 (x 2 M-tiles = 256 rows) halves the K/V gathers per flop once more and puts two
// waves on every SIMD (the whole register file: 512 threads x 256 VGPRs) -- the form for long prefixes, where the
// kernel is bound by the gather traffic rather than by the matrix cores.
// (The bf16 8-wave case has its own kernel below, extend_attention_dbuf_kernel; this one serves fp8 pools and the
// 4-wave shapes.)
template <int D, int MTW, int NWV, bool FP8>
__global__ __launch_bounds__(64 * NWV, (MTW == 1 && NWV == 4) ? (D > 64 ? 2 : 3) : (NWV == 8 ? 2 : 1)) void extend_attention_kernel(ExtendParams p) {
  constexpr bool DEEP = false;
  __shared__ Smem<D> sm;
  const int block_x = blockIdx.x, block_z = blockIdx.z;
  constexpr int CPR = D / 8;            // 16-byte chunks per KV row
  constexpr int KC = D / 32;            // MFMA k-steps over the head dim
  constexpr int ND = D / 16;            // 16-wide output tiles over the head dim
  constexpr int NK_LOADS = kKvTile * CPR / 128;   // K 16-byte loads per K-thread
  constexpr int V_THREADS = 8 * CPR;    // threads that each transpose one 8x8 block

  int tile = block_x;
  const int kvh = blockIdx.y;
  int b = block_z;
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int l15 = lane & 15;
  const int g = lane >> 4;

  const int q_begin = p.qo_indptr[b];
  const int ext_len = p.qo_indptr[b + 1] - q_begin;
  const int kv_len = p.seq_lens[b];
  const int prefix = p.prefix_lens[b];
  const int kv_begin = 0;
  const int32_t* idx_base = p.req_to_token + p.req_pool_indices[b] * p.r2t_stride;
  const int q0 = tile * p.tokens_per_tile;
  if (q0 >= ext_len) return;
  int q1 = q0 + p.tokens_per_tile;
  if (q1 > ext_len) q1 = ext_len;
  const uint8_t* cmask = p.custom_mask ? p.custom_mask + p.mask_indptr[b] : nullptr;
  const bool causal = p.causal && cmask == nullptr;
  const bool plain = cmask == nullptr && p.window < 0 && p.cap_log2 == 0.f;   // workgroup-uniform: the unmasked fast path is legal
  const int kv_end = causal ? (prefix + q1 < kv_len ? prefix + q1 : kv_len) : kv_len;
  // sliding window: the first query row of this tile bounds the earliest kv tile any row can see
  const int kv_first = (p.window >= 0 && prefix + q0 - p.window > 0) ? prefix + q0 - p.window : 0;
  const int t_first = (kv_begin > kv_first ? kv_begin : kv_first) / kKvTile;
  const int n_tiles = (kv_end + kKvTile - 1) / kKvTile;

  // ---- this lane's two rows (one per M-tile) ------------------------------
  int row_tok[MTW], row_limit[MTW], row_start[MTW];
  bool row_ok[MTW];
  int64_t row_off[MTW];   // element offset of (token, head) inside q / out
  U4 qfrag[MTW][KC];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    const int r = wid * (16 * MTW) + mt * 16 + l15;
    const int t = r / p.group;
    const int hg = r - t * p.group;
    row_tok[mt] = q0 + t;
    row_ok[mt] = (t < p.tokens_per_tile) && (q0 + t < q1);
    row_limit[mt] = row_ok[mt] ? (causal ? prefix + q0 + t + 1 : kv_len) : 0;
    if (row_limit[mt] > kv_len) row_limit[mt] = kv_len;
    row_start[mt] = (p.window >= 0 && prefix + q0 + t - p.window > 0) ? prefix + q0 + t - p.window : 0;
    row_off[mt] = static_cast<int64_t>(kvh * p.group + hg) * D;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      if (row_ok[mt]) {
        const int64_t qrow = q_begin + row_tok[mt];
        qfrag[mt][kc] = ld16(p.q + qrow * p.q_stride + row_off[mt] + kc * 32 + g * 8);
      } else {
        qfrag[mt][kc] = U4{0u, 0u, 0u, 0u};
      }
    }
  }

  f32x4_t ot[MTW][ND];
  float m_run[MTW], l_run[MTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    m_run[mt] = kNegBig;
    l_run[mt] = 0.f;
#pragma unroll
    for (int n = 0; n < ND; ++n) ot[mt][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // ---- staging roles -------------------------------------------------------
  // waves 0-1: V (8x8 transposing blocks), waves 2-3: K (row-major).
  const int stid = DEEP ? (tid & 255) : tid;  // role inside the stager half
  const int half = DEEP ? (tid >> 8) : 0;     // wave-uniform: which tiles of the walk this half stages
  const bool is_v = stid < 128;
  const bool is_k = stid >= 128 && stid < kStagers;
  const int st = is_v ? stid : (stid - 128) & 127;
  const int st_c = st % CPR;                 // 16-byte column of the KV row
  const int st_r = st / CPR;
  const bool v_active = is_v && st < V_THREADS;
  const int v_blk32 = st_r >> 2, v_g = st_r & 3;
  constexpr int kStage = (NK_LOADS > 8) ? NK_LOADS : 8;
  U4 stage[kStage];

  // Slot ids run one tile ahead of the rows: a row load that had to wait for its own slot-id load would
  // park the wave for a full memory round trip in front of every tile's MFMAs.
  int32_t sidx[kStage];
  auto prefetch_idx = [&](int t) {
    const int kv0 = t * kKvTile;
    const int last = kv_end - 1;
    if (is_v) {
      if (v_active) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          // token order inside the chunk: i = 4a + r  <->  token 32*blk + 16a + 4g + r
          int tok = kv0 + 32 * v_blk32 + 16 * (i >> 2) + 4 * v_g + (i & 3);
          if (tok > last) tok = last;
          sidx[i] = idx_base[tok];
        }
      }
    } else if (is_k) {
#pragma unroll
      for (int i = 0; i < NK_LOADS; ++i) {
        int tok = kv0 + st_r + (128 / CPR) * i;
        if (tok > last) tok = last;
        sidx[i] = idx_base[tok];
      }
    }
  };
  auto prefetch_rows = [&]() {
    if (is_v) {
      if (v_active) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          stage[i] = ld_kv8<FP8>(kv_row(p.v_cache, p.fmt, sidx[i], kvh), st_c);
      }
    } else if (is_k) {
#pragma unroll
      for (int i = 0; i < NK_LOADS; ++i)
        stage[i] = ld_kv8<FP8>(kv_row(p.k_cache, p.fmt, sidx[i], kvh), st_c);
    }
  };

  auto commit = [&]() {
    if (is_v) {
      if (v_active) {
        const uint32_t* w = reinterpret_cast<const uint32_t*>(stage);  // stage[i] dword q -> w[4i+q]
#pragma unroll
        for (int j = 0; j < 8; ++j) {
          const int d = st_c * 8 + j;
          U4 o;
          uint32_t* ow = reinterpret_cast<uint32_t*>(&o);
#pragma unroll
          for (int qd = 0; qd < 4; ++qd) {
            const uint32_t a = w[4 * (2 * qd) + (j >> 1)];
            const uint32_t c = w[4 * (2 * qd + 1) + (j >> 1)];
            ow[qd] = (j & 1) ? ((a >> 16) | (c & 0xffff0000u)) : ((a & 0xffffu) | (c << 16));
          }
          const int chunk = (4 * v_blk32 + v_g) ^ ((d ^ (d >> 3)) & 7);
          sm.vt[d * 8 + chunk] = o;
        }
      }
    } else if (is_k) {
#pragma unroll
      for (int i = 0; i < NK_LOADS; ++i) {
        const int row = st_r + (128 / CPR) * i;
        sm.k[row * CPR + (st_c ^ (row & (CPR - 1)))] = stage[i];
      }
    }
  };

  constexpr int STEP = DEEP ? 2 : 1;          // tiles between two stagings of the same half
  if (t_first + half < n_tiles) {
    prefetch_idx(t_first + half);
    prefetch_rows();
    if (t_first + half + STEP < n_tiles) prefetch_idx(t_first + half + STEP);
  }

  for (int t = t_first; t < n_tiles; ++t) {
    const bool mine = !DEEP || ((t - t_first) & 1) == half;      // wave-uniform
    __syncthreads();   // every wave is done reading the previous tile
    if (mine) commit();
    __syncthreads();
    if (mine && t + STEP < n_tiles) {
      prefetch_rows();                                   // this half's next tile, slot ids loaded one staging ago
      if (t + 2 * STEP < n_tiles) prefetch_idx(t + 2 * STEP);
    }

    const int kv0 = t * kKvTile;

    // ---- S^T = K . Q^T ---------------------------------------------------
    f32x4_t st_acc[MTW][4];
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) st_acc[mt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int row = nt * 16 + l15;
#pragma unroll
      for (int kc = 0; kc < KC; ++kc) {
        const U4 kf = sm.k[row * CPR + ((kc * 4 + g) ^ (row & (CPR - 1)))];
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt)
          st_acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(
              as_frag(kf), as_frag(qfrag[mt][kc]), st_acc[mt][nt], 0, 0, 0);
      }
    }

    // ---- online softmax; lane owns row (l15 + 16 mt), tokens 16nt + 4g + r --
    // The VALU work here, not the MFMAs, sets the pace of this kernel, so: hardware bf16 packing and
    // v_exp_f32, the scale folded into one fma per score, no masking on tiles that lie inside every row's
    // causal limit, and no rescale of O when no row of the wave raised its maximum.
    U4 pfrag[MTW][2];
#pragma unroll
    for (int mt = 0; mt < MTW; ++mt) {
      const bool full = plain && __ballot(kv0 + kKvTile > row_limit[mt]) == 0ull;     // wave-uniform
      float pv[4][4];
      float m_new, psum = 0.f;
      if (full) {
        float mx = st_acc[mt][0][0];
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r) mx = fmaxf(mx, st_acc[mt][nt][r]);
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        m_new = fmaxf(m_run[mt], mx * p.scale_log2);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float e = fast_exp2(fmaf(st_acc[mt][nt][r], p.scale_log2, -m_new));
            pv[nt][r] = e;
            psum += e;
          }
      } else {
        float sv[4][4];
        float mx = kNegBig;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const int kvpos = kv0 + nt * 16 + g * 4 + r;
            bool on = kvpos < row_limit[mt] && kvpos >= row_start[mt];
            if (cmask != nullptr && on && !(p.mask_skip_prefix && kvpos < prefix))   // the mask row of this query token over all kv_len positions
              on = cmask[static_cast<int64_t>(row_tok[mt]) * kv_len + kvpos] != 0;
            float s = st_acc[mt][nt][r] * p.scale_log2;
            if (p.cap_log2 != 0.f) s = soft_cap_log2(s, p.cap_log2, p.inv_cap_log2);
            s = on ? s : kNegBig;
            sv[nt][r] = s;
            mx = fmaxf(mx, s);
          }
        mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        m_new = fmaxf(m_run[mt], mx);
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float e = (sv[nt][r] > 0.5f * kNegBig) ? fast_exp2(sv[nt][r] - m_new) : 0.f;   // masked scores add nothing, even while the row's maximum is still the sentinel
            pv[nt][r] = e;
            psum += e;
          }
      }
      const float alpha = fast_exp2(m_run[mt] - m_new);
      m_run[mt] = m_new;
      l_run[mt] = l_run[mt] * alpha + psum;
      if (__ballot(alpha != 1.0f) != 0ull) {
#pragma unroll
        for (int n = 0; n < ND; ++n) ot[mt][n] *= alpha;
      }
      // P^T operand for k-step kk: [P(nt=2kk, r=0..3), P(nt=2kk+1, r=0..3)]
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        pfrag[mt][kk].x = pack_bf2(pv[2 * kk][0], pv[2 * kk][1]);
        pfrag[mt][kk].y = pack_bf2(pv[2 * kk][2], pv[2 * kk][3]);
        pfrag[mt][kk].z = pack_bf2(pv[2 * kk + 1][0], pv[2 * kk + 1][1]);
        pfrag[mt][kk].w = pack_bf2(pv[2 * kk + 1][2], pv[2 * kk + 1][3]);
      }
    }

    // ---- O^T += V^T . P^T ------------------------------------------------
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      const int d = n * 16 + l15;
#pragma unroll
      for (int kk = 0; kk < 2; ++kk) {
        const U4 vf = sm.vt[d * 8 + ((kk * 4 + g) ^ ((d ^ (d >> 3)) & 7))];
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt)
          ot[mt][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(vf), as_frag(pfrag[mt][kk]),
                                                               ot[mt][n], 0, 0, 0);
      }
    }
  }

  // ---- epilogue: lane holds O^T[d = 16n + 4g + r][row] ----------------------
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    float l = l_run[mt];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (!row_ok[mt]) continue;
    const float inv = (l > 0.f) ? p.v_scale / l : 0.f;
    uint16_t* op = p.out + static_cast<int64_t>(q_begin + row_tok[mt]) * p.out_stride + row_off[mt];
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      uint2 w;
      w.x = pack_bf2(ot[mt][n][0] * inv, ot[mt][n][1] * inv);
      w.y = pack_bf2(ot[mt][n][2] * inv, ot[mt][n][3] * inv);
      *reinterpret_cast<uint2*>(op + n * 16 + g * 4) = w;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The bf16 8-wave form (256 rows per workgroup, two M-tiles per wave): the shape every prefill of the bench runs.
// Same products, lane maps and softmax as above; what differs is how the K/V tiles travel:
//   * two LDS images per operand and ONE barrier per tile: all 512 threads ask for the rows of tile t + 1 (four 16-byte
//     loads each) before they multiply tile t, and write them to the other image once tile t is done -- the gather has
//     the whole tile's matrix work to land, and no wave waits for a commit between two barriers;
//   * V stays row-major: per 16 head dims a [64 tokens][16] sub-image (rows of 32 B, sub-images 2080 B apart so that the
//     16 pieces of a row land on 16 distinct bank slots); the V^T operand of O^T = V^T . P^T comes out of
//     ds_read_b64_tr_b16 (lane i of a 16-lane group, element j <- row j, column i of the 4 x 16 block the group points
//     at), two reads per operand: tokens 32 kk + 4 g + j and 32 kk + 16 + 4 g + j -- the token order of the P^T
//     fragments built from the S^T accumulators.  No transposition through the VALU;
//   * the running maximum follows every tile (EXT_DEFER_MAX = 0).  Round 3 raised it only when a row outgrew it by 2^8
//     (the rescale of the 64 output accumulators is the largest VALU item of a tile: 2.6-5.5 % of the kernel), but then
//     the row's largest P is exp2(s - m_stale) instead of exp2(0) = 1: the dominant term of a peaked row picks up a bf16
//     rounding error it does not have in the reference's kernels.  Against the fp64 result the deferred form measured
//     rms 0.378 / 0.389 / 0.205 bf16 ulp (flat / unit / peaked scores) where torch's bf16 SDPA has 0.370 / 0.368 / 0.145;
//     with the exact maximum this kernel's figures are the SDPA's to the last digit (benchmarks/r04_exp2_extend_error.py,
//     profiles/r04_exp2_extend_error.json).
#ifndef EXT_DEFER_MAX
#define EXT_DEFER_MAX 0.0f
#endif
constexpr float kDeferMax = EXT_DEFER_MAX;   // log2 units

#ifdef EXT_TRACE
// phase probe (benchmarks/r02_exp9_ext_trace.py): per wave, shader clocks spent in [row loads issued, S^T, softmax,
// PV, commit, barrier] summed over the tiles of the walk, and the tile count
__device__ uint64_t* g_ext_trace = nullptr;
#define EXT_T(i)                                   \
  do {                                             \
    const uint64_t now_ = __builtin_readcyclecounter(); \
    tacc[i] += now_ - tprev;                       \
    tprev = now_;                                  \
  } while (0)
#else
#define EXT_T(i)
#endif

// Maximum over the four 16-lane rows of a wave (the lanes l, l + 16, l + 32, l + 48 hold one query row's scores of
// different tokens): v_permlane16_swap exchanges the odd rows of its first operand with the even rows of its second,
// v_permlane32_swap the upper half of the first with the lower half of the second; on two copies of x each leaves
// (own, partner) in the two registers.  Inline asm on purpose: with the builtin on two copies of ONE value hipcc kept
// only the first result (max(r0, r0)), which turned the reduction into "everybody takes row 0's maximum" -- harmless
// until a row's largest score sits in another lane row and exceeds the others by 2^128 (tests/test_kernels_gpu.py,
// every_workgroup_shape).  The s_nops cover the VALU-write -> permlane-read hazard the assembler does not pad.
__device__ __forceinline__ float row_groups_max(float x) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  a = fmaxf(a, b);
  b = a;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

template <int D>
struct SmemDbuf {
  static constexpr int kVSub = 64 * 32 + 32;                   // bytes of one 16-dim V sub-image + bank skew
  U4 k[2][kKvTile * D / 8];                                    // [token][chunk ^ swz]
  U4 v[2][(D / 16) * kVSub / 16];
};

typedef short v4s16_t __attribute__((ext_vector_type(4)));

// The Q^T fragments stay in 32 registers per lane (round 2 kept them in a lane-private 64 KB LDS image: 5-8 % slower on
// the bench's prefill shapes, profiles/r03_exp0_qreg.txt).  Token-major bf16 pools only (the layout the bench and the
// reference's default pool use): paged head-major pools take the general kernel, so that no gathered row costs a branch.
template <int D>
__global__ __launch_bounds__(512, 2) void extend_attention_dbuf_kernel(ExtendParams p) {
  __shared__ SmemDbuf<D> sm;
  constexpr int MTW = 2;
  constexpr int CPR = D / 8;            // 16-byte chunks per KV row
  constexpr int KC = D / 32;            // MFMA k-steps over the head dim
  constexpr int ND = D / 16;            // 16-wide output tiles over the head dim
  constexpr int ROWS_PER_PASS = 512 / CPR;
  constexpr int LOADS = kKvTile / ROWS_PER_PASS;     // 16-byte loads per thread per operand per tile (2 at D = 128)
  constexpr int VSUB16 = SmemDbuf<D>::kVSub / 16;    // sub-image stride in 16-byte units

  // 1-D grid -> (query tile, kv head, request).  Two things ride on the order: (1) under a causal mask the last query
  // tile of a request walks the most KV tiles, so ALL pairs' heaviest tiles are handed out first and the light ones
  // fill the tail of the launch (4 x 1024 tokens: 115 -> 76 us; pair after pair measured 100); (2) workgroup L runs
  // on XCD L % 8 and every query tile of a (request, kv head) pair reads the same K/V rows, so a pair always lands on
  // the same XCD: what one of its tiles pulled from HBM the others find in that XCD's L2.
  int tile, kvh, b;
  {
    const int L = blockIdx.x;
    const int pairs = p.batch * p.num_kv_heads;
    int pair, rank;
    if (pairs % 8 == 0) {
      const int per_xcd = pairs / 8;
      const int j = L >> 3;
      pair = (j % per_xcd) * 8 + (L & 7);
      rank = j / per_xcd;
    } else {
      pair = L % pairs;
      rank = L / pairs;
    }
    tile = p.num_tiles - 1 - rank;
    kvh = pair % p.num_kv_heads;
    b = pair / p.num_kv_heads;
  }
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wid = tid >> 6;
  const int l15 = lane & 15;
  const int g = lane >> 4;

  const int q_begin = p.qo_indptr[b];
  const int ext_len = p.qo_indptr[b + 1] - q_begin;
  const int kv_len = p.seq_lens[b];
  const int prefix = p.prefix_lens[b];
  const int32_t* idx_base = p.req_to_token + p.req_pool_indices[b] * p.r2t_stride;
  const int q0 = tile * p.tokens_per_tile;
  if (q0 >= ext_len) return;
  int q1 = q0 + p.tokens_per_tile;
  if (q1 > ext_len) q1 = ext_len;
  const bool causal = p.causal != 0;                // (sliding window / soft cap / custom mask: the general kernel)
  const int kv_end = causal ? (prefix + q1 < kv_len ? prefix + q1 : kv_len) : kv_len;
  const int t_first = 0;
  const int n_tiles = (kv_end + kKvTile - 1) / kKvTile;

  // ---- this lane's two rows (one per M-tile) ------------------------------
  int row_tok[MTW], row_limit[MTW];
  bool row_ok[MTW];
  int row_off[MTW];       // element offset of the row's head inside a q / out token
  U4 qreg[MTW][KC];                                 // this lane's Q^T fragments
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    const int r = wid * (16 * MTW) + mt * 16 + l15;
    const int t = r / p.group;
    const int hg = r - t * p.group;
    row_tok[mt] = q0 + t;
    row_ok[mt] = (t < p.tokens_per_tile) && (q0 + t < q1);
    row_limit[mt] = row_ok[mt] ? (causal ? prefix + q0 + t + 1 : kv_len) : 0;
    if (row_limit[mt] > kv_len) row_limit[mt] = kv_len;
    row_off[mt] = (kvh * p.group + hg) * D;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      U4 qf = U4{0u, 0u, 0u, 0u};
      if (row_ok[mt]) {
        const int64_t qrow = q_begin + row_tok[mt];
        qf = ld16(p.q + qrow * p.q_stride + row_off[mt] + kc * 32 + g * 8);
      }
      qreg[mt][kc] = qf;
    }
  }

  f32x4_t ot[MTW][ND];
  float m_run[MTW], l_run[MTW];
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    m_run[mt] = kNegBig;
    l_run[mt] = 0.f;
#pragma unroll
    for (int n = 0; n < ND; ++n) ot[mt][n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  }

  // ---- staging: thread = (row st_r + ROWS_PER_PASS i, 16-byte chunk st_c) of a K tile and of a V tile ----
  const int st_c = tid % CPR, st_r = tid / CPR;
  int32_t idx_k[LOADS], idx_v[LOADS];       // slot ids of the K tile / V tile this thread fetches next
  U4 kst[LOADS], vst[LOADS];
  auto load_idx = [&](int t, int32_t (&dst)[LOADS]) {
    const int last = kv_end - 1;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int tok = t * kKvTile + st_r + ROWS_PER_PASS * i;
      if (tok > last) tok = last;
      dst[i] = idx_base[tok];
    }
  };
  // token-major pool: row = base + slot * row bytes, one v_mad_u64_u32 per gathered row
  const unsigned char* k_rows = reinterpret_cast<const unsigned char*>(p.k_cache) + static_cast<uint64_t>(kvh) * p.fmt.head_stride + st_c * 16;
  const unsigned char* v_rows = reinterpret_cast<const unsigned char*>(p.v_cache) + static_cast<uint64_t>(kvh) * p.fmt.head_stride + st_c * 16;
  auto load_k = [&]() {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      kst[i] = ld16(k_rows + static_cast<uint64_t>(static_cast<uint32_t>(idx_k[i])) * p.fmt.page_stride);
    }
  };
  auto load_v = [&]() {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      vst[i] = ld16(v_rows + static_cast<uint64_t>(static_cast<uint32_t>(idx_v[i])) * p.fmt.page_stride);
    }
  };
  auto commit_k = [&](int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int row = st_r + ROWS_PER_PASS * i;
      sm.k[buf][row * CPR + (st_c ^ ((row * CPR / 16) & (CPR - 1)))] = kst[i];
    }
  };
  auto commit_v = [&](int buf) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int row = st_r + ROWS_PER_PASS * i;
      sm.v[buf][(st_c >> 1) * VSUB16 + row * 2 + (st_c & 1)] = vst[i];
    }
  };
  // V^T fragment reads: byte offset of this lane inside a sub-image, token rows 4 g + (l15 >> 2), 8-byte piece l15 & 3
  const int v_lane = (4 * g + (l15 >> 2)) * 32 + (l15 & 3) * 8;

  // ---- the two halves of the workgroup run half a tile apart ---------------------------------------------------
  // Waves w and w + 4 share a SIMD.  Time is cut into slots, one barrier each; in slot s a wave is either in its
  // matrix block  [ O^T += V^T P^T of tile u - 1,  S^T = K Q^T of tile u ]  or in its vector block  [ softmax of
  // tile u, staging ]: waves 0-3 multiply in the even slots (u = s / 2), waves 4-7 in the odd ones, so on every SIMD
  // one wave feeds the matrix core while the other one runs the exp / max / pack work on the VALU (in lock-step both
  // queue for the same unit: 7100 clocks per tile, 2780 of them softmax, benchmarks/r02_exp9_ext_trace.py).
  // Staging rides at the end of the matrix blocks: the waves multiplying in slots 2 v and 2 v + 1 write their
  // share of K tile v + 1 (its image was last read in slot 2 v - 1, is first read in slot 2 v + 2) and of V tile v
  // (last read 2 v - 1, first read 2 v + 2), then ask for K tile v + 2 and V tile v + 1: a tile-time in flight.
  const int grp = __builtin_amdgcn_readfirstlane(wid >> 2);
  const int t0 = t_first;
  if (t0 < n_tiles) {
    load_idx(t0, idx_k);
    load_idx(t0, idx_v);
    load_k();
    if (t0 + 1 < n_tiles) load_idx(t0 + 1, idx_k);
    commit_k(0);
    load_v();                                        // V tile t0, written in slot 2 t0 / 2 t0 + 1
    if (t0 + 1 < n_tiles) {
      load_idx(t0 + 1, idx_v);
      load_k();                                      // K tile t0 + 1, same
    }
    if (t0 + 2 < n_tiles) load_idx(t0 + 2, idx_k);
  }
  __syncthreads();

  f32x4_t st_acc[MTW][4];
  U4 pfrag[MTW][2];
#ifdef EXT_TRACE
  uint64_t tacc[6] = {0, 0, 0, 0, 0, 0};
  uint64_t tprev = __builtin_readcyclecounter();
  const uint64_t tstart = tprev;
#endif
  // matrix block of tile u: O^T += V^T P^T of tile u - 1, then S^T of tile u.  The LDS fragment reads run ONE MFMA
  // GROUP AHEAD of the products that use them (two register sets per operand): in program order hipcc waited for every
  // group's own ds_reads with the matrix core drained (64 MFMAs took 1720 clocks instead of 1024).
  auto read_v = [&](const unsigned char* vbase, int n, U4 (&dst)[2]) {
    typedef __attribute__((address_space(3))) v4s16_t* lds_v4_t;
#pragma unroll
    for (int kk = 0; kk < 2; ++kk) {
      const v4s16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(vbase + n * SmemDbuf<D>::kVSub + kk * 1024));
      const v4s16_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(vbase + n * SmemDbuf<D>::kVSub + kk * 1024 + 512));
      dst[kk].x = __builtin_bit_cast(uint2, lo).x; dst[kk].y = __builtin_bit_cast(uint2, lo).y;
      dst[kk].z = __builtin_bit_cast(uint2, hi).x; dst[kk].w = __builtin_bit_cast(uint2, hi).y;
    }
  };
  auto read_k = [&](const U4* kimg, int nt, U4 (&dst)[KC]) {
    const int row = nt * 16 + l15;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) dst[kc] = kimg[row * CPR + ((kc * 4 + g) ^ ((row * CPR / 16) & (CPR - 1)))];
  };
  auto matrix_block = [&](int u) {
    EXT_T(5);
    const bool have_pv = u - 1 >= t0 && u - 1 < n_tiles, have_s = u < n_tiles;
    const U4* kimg = sm.k[(u - t0) & 1];
    U4 kf[2][KC];
    if (have_s) {                                       // the first K fragments travel under the PV products
      read_k(kimg, 0, kf[0]);
      __builtin_amdgcn_sched_group_barrier(0x100, KC, 0);
    }
    if (have_pv) {
      // ---- O^T += V^T . P^T (tile u - 1) ----------------------------------
      const unsigned char* vbase = reinterpret_cast<const unsigned char*>(sm.v[(u - 1 - t0) & 1]) + v_lane;
      U4 vf[2][2];
      read_v(vbase, 0, vf[0]);
      __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
      for (int n = 0; n < ND; ++n) {
        if (n + 1 < ND) read_v(vbase, n + 1, vf[(n + 1) & 1]);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
          for (int mt = 0; mt < MTW; ++mt)
            ot[mt][n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(vf[n & 1][kk]), as_frag(pfrag[mt][kk]), ot[mt][n], 0, 0, 0);
        // pin the order the source states: the NEXT group's four reads, then this group's four products
        if (n + 1 < ND) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 4, 0);
      }
    }
    EXT_T(3);
    if (have_s) {
      // ---- S^T = K . Q^T (tile u) -----------------------------------------
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt)
#pragma unroll
        for (int nt = 0; nt < 4; ++nt) st_acc[mt][nt] = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) {
        if (nt + 1 < 4) read_k(kimg, nt + 1, kf[(nt + 1) & 1]);
#pragma unroll
        for (int kc = 0; kc < KC; ++kc)
#pragma unroll
          for (int mt = 0; mt < MTW; ++mt)
            st_acc[mt][nt] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(kf[nt & 1][kc]), as_frag(qreg[mt][kc]), st_acc[mt][nt], 0, 0, 0);
        if (nt + 1 < 4) __builtin_amdgcn_sched_group_barrier(0x100, KC, 0);
        __builtin_amdgcn_sched_group_barrier(0x008, 2 * KC, 0);
      }
    }
    EXT_T(1);
    // ---- staging of this slot pair (v = u): K tile v + 1 and V tile v go to LDS, K tile v + 2 and V tile v + 1 are
    // asked for.  Behind the MFMAs: the writes wait for rows requested a tile ago while the matrix core drains.
    const int v = u;
    if (v < n_tiles) commit_v((v - t0) & 1);
    if (v + 1 < n_tiles) commit_k((v + 1 - t0) & 1);
    EXT_T(4);
    EXT_T(0);
  };
  // vector block: softmax of tile u (the scores the wave holds)
  auto vector_block = [&](int u) {
    EXT_T(5);
    if (u >= t0 && u < n_tiles) {
      const int kv0 = u * kKvTile;
      // ---- online softmax; lane owns row (l15 + 16 mt), tokens 16 nt + 4 g + r.  Both M-tiles go through each step
      // together (two independent chains in flight), the row maximum crosses the four 16-lane rows of the wave with
      // v_permlane16_swap / v_permlane32_swap (no LDS round trip), the scale rides in the exp's fma.
      const bool full = __ballot(kv0 + kKvTile > row_limit[0] || kv0 + kKvTile > row_limit[1]) == 0ull;   // wave-uniform
      float mx[MTW];
      if (full) {
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt) {
          float m = st_acc[mt][0][0];
#pragma unroll
          for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) m = fmaxf(m, st_acc[mt][nt][r]);
          mx[mt] = m * p.scale_log2;
        }
      } else {
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt) {
          float m = kNegBig;
#pragma unroll
          for (int nt = 0; nt < 4; ++nt)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const int kvpos = kv0 + nt * 16 + g * 4 + r;
              // a masked score becomes the sentinel BEFORE the scale: exp2(fma(sentinel, scale, -m)) = 0
              const float sc = kvpos < row_limit[mt] ? st_acc[mt][nt][r] : kNegBig;
              st_acc[mt][nt][r] = sc;
              m = fmaxf(m, sc);
            }
          mx[mt] = m > 0.5f * kNegBig ? m * p.scale_log2 : kNegBig;
        }
      }
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt) mx[mt] = row_groups_max(mx[mt]);
      if (__ballot(mx[0] > m_run[0] + kDeferMax || mx[1] > m_run[1] + kDeferMax) != 0ull) {
        // some row outgrew its maximum: raise them all
#pragma unroll
        for (int mt = 0; mt < MTW; ++mt) {
          const float m_new = fmaxf(m_run[mt], mx[mt]);
          const float alpha = fast_exp2(m_run[mt] - m_new);
          m_run[mt] = m_new;
          l_run[mt] *= alpha;
#pragma unroll
          for (int n = 0; n < ND; ++n) ot[mt][n] *= alpha;
        }
      }
#pragma unroll
      for (int mt = 0; mt < MTW; ++mt) {
        float psum = 0.f;
        float pv[4][4];
        // rows that have seen no key yet keep the sentinel as maximum: their (all masked) scores must give 0, not 1
        const float neg_m = m_run[mt] > 0.5f * kNegBig ? -m_run[mt] : 0.f;
#pragma unroll
        for (int nt = 0; nt < 4; ++nt)
#pragma unroll
          for (int r = 0; r < 4; ++r) {
            const float e = fast_exp2(fmaf(st_acc[mt][nt][r], p.scale_log2, neg_m));
            pv[nt][r] = e;
            psum += e;
          }
        l_run[mt] += psum;
        // P^T operand for k-step kk: [P(nt=2kk, r=0..3), P(nt=2kk+1, r=0..3)]
#pragma unroll
        for (int kk = 0; kk < 2; ++kk) {
          pfrag[mt][kk].x = pack_bf2(pv[2 * kk][0], pv[2 * kk][1]);
          pfrag[mt][kk].y = pack_bf2(pv[2 * kk][2], pv[2 * kk][3]);
          pfrag[mt][kk].z = pack_bf2(pv[2 * kk + 1][0], pv[2 * kk + 1][1]);
          pfrag[mt][kk].w = pack_bf2(pv[2 * kk + 1][2], pv[2 * kk + 1][3]);
        }
      }
    }
    EXT_T(2);
    // ---- requests for the next commit (matrix block u + 1 writes K tile u + 2 and V tile u + 1): the registers are
    // free since this wave's matrix block u wrote their previous contents to LDS
    const int v = u;
    // (each id array is loaded straight into its own registers: handing idx_k over to idx_v by a copy made hipcc wait
    // for EVERY load in flight at the end of this block -- 900-1400 clocks per tile)
    if (v + 1 < n_tiles) {
      load_v();                                     // V tile v + 1 (idx_v holds its slot ids)
      if (v + 2 < n_tiles) load_idx(v + 2, idx_v);
    }
    if (v + 2 < n_tiles) {
      load_k();                                     // K tile v + 2
      if (v + 3 < n_tiles) load_idx(v + 3, idx_k);
    }
    EXT_T(0);
  };
  // two straight-line loops instead of one loop with a role switch per slot (which hipcc spilled around)
  if (grp == 0) {
    for (int u = t0; u <= n_tiles; ++u) {
      matrix_block(u);
      __syncthreads();
      EXT_T(5);
      vector_block(u);
      __syncthreads();
      EXT_T(5);
    }
  } else {
    __syncthreads();                                  // the half-tile offset: an empty first slot
    for (int u = t0; u < n_tiles; ++u) {
      matrix_block(u);
      __syncthreads();
      EXT_T(5);
      vector_block(u);
      __syncthreads();
      EXT_T(5);
    }
    matrix_block(n_tiles);
    __syncthreads();
  }
#ifdef EXT_TRACE
  if (g_ext_trace && lane == 0) {
    uint64_t* o = g_ext_trace + static_cast<int64_t>(blockIdx.x) * 64 + wid * 8;
    for (int i = 0; i < 6; ++i) o[i] = tacc[i];
    o[6] = n_tiles - t_first;
    o[7] = tstart;
  }
#endif

  // ---- epilogue: lane holds O^T[d = 16n + 4g + r][row] ----------------------
#pragma unroll
  for (int mt = 0; mt < MTW; ++mt) {
    float l = l_run[mt];
    l += __shfl_xor(l, 16, 64);
    l += __shfl_xor(l, 32, 64);
    if (!row_ok[mt]) continue;
    const float inv = (l > 0.f) ? 1.0f / l : 0.f;
    uint16_t* op = p.out + static_cast<int64_t>(q_begin + row_tok[mt]) * p.out_stride + row_off[mt];
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      uint2 w;
      w.x = pack_bf2(ot[mt][n][0] * inv, ot[mt][n][1] * inv);
      w.y = pack_bf2(ot[mt][n][2] * inv, ot[mt][n][3] * inv);
      *reinterpret_cast<uint2*>(op + n * 16 + g * 4) = w;
    }
  }
}

// ---------------------------------------------------------------------------------------------
// The 32x32 form of the bf16 8-wave kernel: what every prefill of the bench runs (token-major bf16 pool, causal or not,
// no window / cap / mask; the ping-pong kernel above stays selectable for A/B runs).  What changes against it:
//   * v_mfma_f32_32x32x16_bf16: one wave = 32 rows (query token x head of the group), a 64-key tile = two 32-key blocks.
//     S^T = K . Q^T leaves lane (q = lane & 31, h = lane >> 5) with 32 scores of ONE row (keys 32 blk + (r & 3) +
//     8 (r >> 2) + 4 h): the row maximum is an in-lane chain + ONE v_permlane32_swap, the row sum stays a per-lane partial
//     until the epilogue, and bf16(P) of registers 8 ks .. 8 ks + 7 IS the B operand of O^T += V^T . P^T for the 16 keys
//     {32 blk + 16 ks + (j & 3) + 8 (j >> 2) + 4 h}; the V^T operand is read in that key order (two ds_read_b64_tr_b16:
//     keys kb + 4 h + 0..3 and kb + 8 + 4 h + 0..3).  Half the LDS fragment reads per flop of the 16x16x32 shape;
//   * no role split and ONE barrier per tile; the vector work of a tile rides between the matrix instructions of its
//     NEIGHBOURS (two score sets, see the kernel's own header);
//   * V image per 32 head dims: [64 tokens][64 B] (+ a bank skew between the sub-images), so that the four 16-lane groups
//     of a transposing read cover 512 contiguous bytes;
//   * a raised maximum is applied to O and l when everything exponentiated against the old one is
//     inside them (the order the softmax-rescale hazard asks for);
//   * the epilogue swaps 4-dim pieces between the lane halves and stores 16 bytes per lane.
// Measured on MI355X (benchmarks/r03_exp4_extend_32x32.py, profiles/r03_exp4_extend_32x32.json): 4 x 1024 cold 62 -> 52 us, 60 x 128
// over 896 warm 197 -> 167 us, 2 x 4096 304 -> 279 us, 8 x 2952 676 -> 629 us.  A one-score-set version of the same
// form (S^T(t) -> max(t) -> [products of t - 1 || exponentials of t]; commit 21c58e7..: 2-6 % slower) and its 4-wave /
// two-workgroups-per-CU variant (slower again: twice the row requests per flop) were measured and dropped.
typedef float f32x16_t __attribute__((ext_vector_type(16)));

// (FP8: rows that are widened on their way in, written by the threads: V in one sub-image per 32 head dims with a bank skew between them)
template <int D, bool FP8>
struct SmemLadder {
  static constexpr int kVSub = 64 * 64 + (D == 128 ? 64 : 128);   // bytes of one 32-dim V sub-image + bank skew
  U4 k[2][kKvTile * D / 8];                                       // [token][chunk ^ k_swz]
  U4 v[2][FP8 ? (D / 32) * kVSub / 16 : kKvTile * D / 8];         // [dims / 32][token][chunk] or [token][chunk ^ v_swz]
  // The scores' operand: 16 consecutive tokens at one chunk cover all chunk slots of the 256 bytes of banks.
  __device__ __forceinline__ static int k_swz(int row) { return (row * (D / 8) / 16) & (D / 8 - 1); }
  // The values' operand: four consecutive tokens at 64 bytes each (a transposing read of half a wave) cover the banks once.
  __device__ __forceinline__ static int v_swz(int row) { return D == 128 ? (row & 3) << 2 : (row & 2) << 1; }
};

// 16 bytes a lane from memory to 1 KiB of LDS at `to`, behind the compiler's back: it would wait for all of these in front of the next read
// of LDS.  Whoever issues them waits (rows_landed) and meets the others at a barrier before any of it is read.  No registers are written, and
// nothing else here uses M0 (which cannot be named as overwritten; test_no_spills.py looks for other users of it in the listing).  Rows that went through registers cost a step 300 of its 3900 clocks: all waves write LDS behind the barrier while
// no product runs.  us, through registers / straight to LDS: 60 x 128 behind 896, 32 / 8 heads, 166 / 162, six cold prompts of 1.1 to 3.1 k, 64 / 8
// heads, 619 / 603 (both at a lower clock in turn: power), 6 x 2000 cold, 14 / 2 heads of 64, 79 / 68, 1000 cold 26.0 / 23.5, 203 behind 3800 35.2 / 33.2.
__device__ __forceinline__ void rows_to_lds(const unsigned char* from, uint32_t to) {
  asm volatile("s_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, off" : : "v"(from), "s"(to) : "memory");
}
__device__ __forceinline__ void rows_landed() { asm volatile("s_waitcnt vmcnt(0)" : : : "memory"); }

__device__ __forceinline__ float lane_pair_max(float x) {         // max over lanes l and l ^ 32
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

__device__ __forceinline__ float lane_pair_sum(float x) {         // the sum of the same two
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return a + b;
}

// The query tiles of a launch as workgroups that stay take them (extend_attention_walk_kernel): one list per XCD (tile L goes to list L mod 8, as
// launched workgroups would), longest contexts first.  A request's tiles stand at consecutive levels, tile t behind a prefix of whole tiles at
// level prefix / tokens + t; a level lists its requests' kv heads, so that neighbours in the list read the same heads' rows on the same XCD.
struct WalkQueue {
  static constexpr int kRequests = 512, kThreads = 512, kLevels = 4096;
  int next;                                         // the tile taken next, for all waves
  int sums[kThreads / 64];
  int32_t ids[4 * kKvTile];                         // slots of its first four key tiles
  int first[kRequests], tiles[kRequests];           // levels [first, first + tiles)
  int q_begin[kRequests], len[kRequests], kv_len[kRequests], prefix[kRequests], row[kRequests];
  int below[kLevels];                               // tiles in front of the i-th level from the top
  int all;                                          // tiles of the launch

  // every thread of the workgroup; returns the top level
  __device__ __forceinline__ int fill(const ExtendParams& p, int tid) {
    const int lane = tid & 63, wid = tid >> 6;
    int f = 0, n = 0;
    if (tid < p.batch) {
      const int at = p.qo_indptr[tid], l = p.qo_indptr[tid + 1] - at, pre = p.prefix_lens[tid];
      n = l > 0 ? min((l + p.tokens_per_tile - 1) / p.tokens_per_tile, kLevels) : 0;
      f = min(pre / p.tokens_per_tile, kLevels - n);  // (longer contexts stand at the top together)
      q_begin[tid] = at;
      len[tid] = l;
      kv_len[tid] = p.seq_lens[tid];
      prefix[tid] = pre;
      row[tid] = static_cast<int>(p.req_pool_indices[tid]);
    }
    first[tid] = f;
    tiles[tid] = n;
    int top = n > 0 ? f + n - 1 : -1;
#pragma unroll
    for (int d = 32; d > 0; d >>= 1) top = max(top, __shfl_xor(top, d, 64));
    if (lane == 0) sums[wid] = top;
    __syncthreads();
    top = -1;
#pragma unroll
    for (int w = 0; w < kThreads / 64; ++w) top = max(top, sums[w]);
    top = __builtin_amdgcn_readfirstlane(top);
    __syncthreads();
    const int per = (top + kThreads) / kThreads;    // levels of a thread: per tid .. from the top, 1 up to 32 k tokens in tiles of 64
    int mine = 0;
    for (int i = 0; i < per; ++i) {
      const int level = top - (per * tid + i);
      int c = 0;
      if (level >= 0)
        for (int r = 0; r < p.batch; ++r) c += level >= first[r] && level - first[r] < tiles[r] ? p.num_kv_heads : 0;
      if (per * tid + i < kLevels) below[per * tid + i] = mine;
      mine += c;
    }
    int upto = mine;                                // of the wave's threads so far
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(upto, d, 64);
      if (lane >= d) upto += o;
    }
    if (lane == 63) sums[wid] = upto;
    __syncthreads();
    int front = upto - mine;
    for (int w = 0; w < wid; ++w) front += sums[w];
    for (int i = 0; i < per; ++i)
      if (per * tid + i < kLevels) below[per * tid + i] += front;
    if (tid == kThreads - 1) all = front + mine;
    __syncthreads();
    return top;
  }

  // request, kv head and query tile of tile L of the list (one that exists)
  __device__ __forceinline__ void find(int L, int top, int batch, int heads, int lane, int& b, int& kvh, int& tile) const {
    int at = 0;                                     // the last level with below[] <= L: 64 of them at a time, then one of 64
    for (int c = 64; c <= top; c += 64 * 64) {
      const int i = c + 64 * lane;
      at += 64 * __popcll(__ballot(i <= top && below[i <= top ? i : 0] <= L));
    }
    const int i = at + lane;
    at += __popcll(__ballot(i <= top && below[i <= top ? i : 0] <= L)) - 1;
    const int level = top - at, rest = L - __builtin_amdgcn_readfirstlane(below[at]);
    int nth = rest / heads;
    kvh = rest - nth * heads;
    b = 0;
    for (int c = 0; c < batch; c += 64) {
      const bool in = level >= first[c + lane] && level - first[c + lane] < tiles[c + lane];
      const unsigned long long m = __ballot(in);
      const int n = __popcll(m);
      if (nth < n) {
        const int rank = __builtin_amdgcn_mbcnt_hi(static_cast<unsigned>(m >> 32), __builtin_amdgcn_mbcnt_lo(static_cast<unsigned>(m), 0u));
        b = c + __ffsll(__ballot(in && rank == nth)) - 1;
        break;
      }
      nth -= n;
    }
    tile = level - __builtin_amdgcn_readfirstlane(first[b]);
  }
};

// A step of the walk is two phases of products with the vector work of the NEIGHBOURING tiles spread between them:
//     phase 1:  S^T(t + 1) = K(t + 1) . Q^T   ||  P(t) = exp2(S(t) scale - m)  and the row requests of the tiles ahead
//     phase 2:  O^T += V^T(t) . P^T(t)        ||  mask + row maxima of S(t + 1)
//     then the rescale decision for tile t + 1 (everything exponentiated against the old maximum -- P(t) -- is inside
//     O and l by then), and ONE barrier.
// Every product carries <= 7 vector instructions, none of them waiting for the product next to it; what is left outside
// the products' shadow is the decision (a permlane, two ballots), with e4m3 rows four LDS writes, and the barrier.
// FP8: the pool holds e4m3 rows (8 bytes per lane and chunk, held raw in the staging registers, widened to bf16 -- exact --
// on their way into the LDS images; k_scale rides in the softmax scale, v_scale in the epilogue).
// PARTS: the walk covers part `part` of p.parts equal pieces of the request's key tiles (extend_attention_parts_kernel below).
// STAYS: the workgroup takes query tiles from the queue until there are none (extend_attention_walk_kernel below).
template <int D, int NWV, bool FP8, bool PARTS, bool STAYS = false>
__device__ __forceinline__ void extend_pipe_body(const ExtendParams& p, SmemLadder<D, FP8>& sm, WalkQueue* queue = nullptr) {
  constexpr int CPR = D / 8;            // 16-byte chunks per KV row
  constexpr int KS = D / 16;            // MFMA k-steps over the head dim
  constexpr int ND = D / 32;            // 32-wide output blocks over the head dim
  constexpr int ROWS_PER_PASS = 64 * NWV / CPR;
  constexpr int LOADS = kKvTile / ROWS_PER_PASS;     // 16-byte loads per thread per operand per tile (2 at D = 128, 8 waves)
  typedef SmemLadder<D, FP8> Lds;
  constexpr bool DMA = !FP8;                         // rows go from memory to LDS as they are (rows_to_lds)
  static_assert(ROWS_PER_PASS % 16 == 0 && (64 * NWV) % CPR == 0, "a thread's rows share their swizzles");
  constexpr int NPV = ND * 4;           // PV products per tile

  // (STAYS: formed anew for each query tile, as is what only the passage from tile to tile needs: kept across the outer loop, all the addresses
  // made of them would take registers from the walk)
  auto thread = [&]() __attribute__((always_inline)) {
    int x = threadIdx.x;
    if constexpr (STAYS) asm volatile("" : "+v"(x));
    return x;
  };
  int tid, lane, wid, l31, hi;
  auto lanes = [&]() __attribute__((always_inline)) {
    tid = thread();
    lane = tid & 63;
    wid = tid >> 6;
    l31 = lane & 31;
    hi = lane >> 5;
  };
  lanes();
  // grid -> (query tile, kv head, request): as in the ping-pong kernel (heaviest tiles first, a pair stays on one XCD)
  // (with PARTS a pair is a (request, kv head, part): the query tiles that read the same keys)
  int tile, kvh, b, part = 0;
  int q_begin, ext_len, kv_len, prefix;
  const int32_t* idx_base;
  int top = 0, all = 0;                                // of the queue: its top level, its tiles
  auto of_queue = [&](int r, int t) __attribute__((always_inline)) {       // request r's figures
    q_begin = __builtin_amdgcn_readfirstlane(queue->q_begin[r]);
    ext_len = __builtin_amdgcn_readfirstlane(queue->len[r]);
    kv_len = __builtin_amdgcn_readfirstlane(queue->kv_len[r]);
    prefix = __builtin_amdgcn_readfirstlane(queue->prefix[r]);
    idx_base = p.req_to_token + __builtin_amdgcn_readfirstlane(queue->row[r]) * p.r2t_stride;
    tile = t;
  };
  if constexpr (STAYS) {
    static_assert(64 * NWV == WalkQueue::kThreads && WalkQueue::kRequests == WalkQueue::kThreads, "one request a thread");
    top = queue->fill(p, tid);
    all = __builtin_amdgcn_readfirstlane(queue->all);   // (not in `next`: a first tile without keys has no barrier in front of hand())
    if (static_cast<int>(blockIdx.x) >= all) return;
    queue->find(blockIdx.x, top, p.batch, p.num_kv_heads, lane, b, kvh, tile);
    of_queue(b, tile);
  } else {
    int heads = p.num_kv_heads;
    int64_t table_stride = p.r2t_stride;
    asm("" : "+s"(heads), "+s"(table_stride));             // (asked for with the first arguments, not in a round trip of its own behind the lengths)
    {
      const int L = blockIdx.x;
      const int pairs = p.batch * heads * (PARTS ? p.parts : 1);
      int pair, rank;
      if (pairs % 8 == 0) {
        const int per_xcd = pairs / 8;
        const int j = L >> 3;
        pair = (j % per_xcd) * 8 + (L & 7);
        rank = j / per_xcd;
      } else {
        pair = L % pairs;
        rank = L / pairs;
      }
      tile = p.num_tiles - 1 - rank;
      if constexpr (PARTS) {
        part = pair % p.parts;
        pair /= p.parts;
      }
      kvh = pair % heads;
      b = pair / heads;
    }
    q_begin = p.qo_indptr[b];
    ext_len = p.qo_indptr[b + 1] - q_begin;
    kv_len = p.seq_lens[b];
    prefix = p.prefix_lens[b];
    int64_t row = p.req_pool_indices[b];
    // (one round trip for all five: left to itself the compiler sinks the last three below the branch.  Not volatile: behind that they would be vector loads)
    asm("" : "+s"(ext_len), "+s"(kv_len), "+s"(prefix), "+s"(row));
    idx_base = p.req_to_token + row * table_stride;
    if (tile * p.tokens_per_tile >= ext_len) return;
  }

  // ---- the query tile: its tokens, its keys, this lane's row (both lane halves of a row hold the same query, other head dims / keys) ----
  const bool causal = p.causal != 0;
  int r_tok, r_hg;
  auto row_of = [&](int x) __attribute__((always_inline)) {
    // (PARTS: of two workgroups on a compute unit, the launch's w and w + 256, one takes its rows from the last wave on, so that waves without rows stand on
    // different SIMDs)
    const int r_row = ((x >> 6) ^ (PARTS && DMA ? (blockIdx.x >> 8 & 1) * (NWV - 1) : 0)) * 32 + (x & 31);
    int group = p.group;
    if constexpr (STAYS || PARTS) asm volatile("" : "+s"(group));
    r_tok = r_row / group;
    r_hg = r_row - r_tok * group;
  };
  int q0, q1, kv_end, n_tiles, row_limit, row_off;
  bool row_ok;
  auto place = [&]() __attribute__((always_inline)) {
    row_of(thread());
    q0 = tile * p.tokens_per_tile;
    q1 = q0 + p.tokens_per_tile;
    if (q1 > ext_len) q1 = ext_len;
    kv_end = causal ? (prefix + q1 < kv_len ? prefix + q1 : kv_len) : kv_len;
    n_tiles = (kv_end + kKvTile - 1) / kKvTile;
    row_ok = (r_tok < p.tokens_per_tile) && (q0 + r_tok < q1);
    row_limit = row_ok ? (causal ? prefix + q0 + r_tok + 1 : kv_len) : 0;
    if (row_limit > kv_len) row_limit = kv_len;
    row_off = (kvh * p.group + r_hg) * D;
  };
  place();
  // this part's tiles become tiles 0 .. n_tiles - 1 of the walk: the row of the request table, the end and the rows' limits move
  int part_begin = 0;
  bool empty = n_tiles <= 0;                               // workgroup-uniform: no key to read (below)
  if constexpr (PARTS) {
    const int per = (n_tiles + p.parts - 1) / p.parts;
    const int t0 = part * per;
    empty = t0 >= n_tiles;
    if (!empty) {
      n_tiles = n_tiles - t0 < per ? n_tiles - t0 : per;
      part_begin = t0 * kKvTile;
      kv_end -= part_begin;
      idx_base += part_begin;
    }
    row_limit -= part_begin;
  }
  auto put_zeros = [&]() __attribute__((always_inline)) {
    uint16_t* op = p.out + static_cast<int64_t>(q_begin + q0 + r_tok) * p.out_stride + row_off;
#pragma unroll
    for (int c = 0; c < CPR / 2; ++c) *reinterpret_cast<U4*>(op + (2 * c + hi) * 8) = U4{0u, 0u, 0u, 0u};
  };
  if (!STAYS && empty) {                                   // a part without keys has no weight, a request without keys gives zeros
    if (PARTS && p.parts > 1) {
      if (row_ok && hi == 0) {
        float* ml = p.part_ml + 2 * (part * p.part_rows + static_cast<int64_t>(q_begin + q0 + r_tok) * (p.num_kv_heads * p.group) + kvh * p.group + r_hg);
        ml[0] = kNegBig;
        ml[1] = 0.f;
      }
    } else if (row_ok) put_zeros();
    return;
  }
  U4 qreg[KS];                                      // Q^T operand of k-step s: dims 16 s + 8 h .. + 7 of the row
  if constexpr (!STAYS) {
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      U4 qf = U4{0u, 0u, 0u, 0u};
      if (row_ok) qf = ld16(p.q + static_cast<int64_t>(q_begin + q0 + r_tok) * p.q_stride + row_off + s * 16 + hi * 8);
      qreg[s] = qf;
    }
  }

  f32x16_t ot[ND];
  float m_run, l_run;                               // l: this lane's share of the row sum
  auto fresh = [&]() __attribute__((always_inline)) {
    m_run = kNegBig;
    l_run = 0.f;
#pragma unroll
    for (int n = 0; n < ND; ++n)
#pragma unroll
      for (int r = 0; r < 16; ++r) ot[n][r] = 0.f;
  };
  if constexpr (!STAYS) fresh();

  // ---- staging: thread = (row st_r + ROWS_PER_PASS i, 16-byte chunk st_c) of a K tile and of a V tile ----
  int st_c, st_r;
  int32_t idx_k[LOADS], idx_v[LOADS], idx_n[LOADS];
  typedef typename std::conditional<FP8, uint2, U4>::type Stage;   // a gathered 8-dim piece as it travels: raw bytes
  Stage kst[LOADS], vst[LOADS];
  auto ld_stage = [&](const unsigned char* ptr) __attribute__((always_inline)) -> Stage {
    if constexpr (FP8) return *reinterpret_cast<const uint2*>(ptr);
    else return ld16(ptr);
  };
  auto widen = [&](const Stage& v) __attribute__((always_inline)) -> U4 {
    if constexpr (FP8) return fp8x8_to_bf16x8(v);
    else return v;
  };
  auto load_idx = [&](int t, int32_t (&dst)[LOADS]) {
    const int last = kv_end - 1;
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      int tok = t * kKvTile + st_r + ROWS_PER_PASS * i;
      if (tok > last) tok = last;
      dst[i] = idx_base[tok];
    }
  };
  // V^T operand reads: lane i of 16-lane group g points at token row 4 (g >> 1) + (i >> 2), dims 16 (g & 1) + 4 (i & 3) of a 32-dim block
  int v_lane[DMA ? ND : 1];
  uint32_t to_lds = 0;                              // the wave's 1 KiB of a pass, from the images' start
  auto v_lanes = [&]() __attribute__((always_inline)) {
    const int r = 4 * hi + ((lane & 15) >> 2), in = ((lane >> 4) & 1) * 32 + (lane & 3) * 8;
    if constexpr (DMA) {
#pragma unroll
      for (int n = 0; n < ND; ++n) v_lane[n] = r * (2 * D) + (((4 * n) ^ Lds::v_swz(r)) << 4) + in;
    } else {
      v_lane[0] = r * 64 + in;
    }
  };
  auto pieces = [&]() __attribute__((always_inline)) {
    st_c = tid % CPR;
    st_r = tid / CPR;
  };
  auto staging = [&]() __attribute__((always_inline)) {
    if constexpr (STAYS) {
      lanes();
      pieces();
    }
    v_lanes();
    to_lds = static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(wid)) * 1024u;
  };
  if constexpr (STAYS) staging();
  else pieces();
  auto head_rows = [&](const uint16_t* cache, int head, int c) __attribute__((always_inline)) {
    return reinterpret_cast<const unsigned char*>(cache) + static_cast<uint64_t>(head) * p.fmt.head_stride + c * (FP8 ? 8 : 16);
  };
  // (DMA: a thread writes chunk slot st_c of its rows, so that it fetches the chunk that belongs there)
  const unsigned char *k_rows, *v_rows;
  auto rows_of = [&](int head) __attribute__((always_inline)) {
    k_rows = head_rows(p.k_cache, head, DMA ? st_c ^ Lds::k_swz(st_r) : st_c);
    v_rows = head_rows(p.v_cache, head, DMA ? st_c ^ Lds::v_swz(st_r) : st_c);
  };
  rows_of(kvh);
  if constexpr (!STAYS) staging();

  // (STAYS: a stride widened in front of the outer loop would be multiplied in 64 x 32 bits, two quarter-rate instructions a row for one)
  auto row_stride = [&]() __attribute__((always_inline)) {
    uint32_t x = p.fmt.page_stride;
    if constexpr (STAYS) asm volatile("" : "+s"(x));
    return x;
  };
  auto load_rows = [&](const unsigned char* base, const int32_t (&ids)[LOADS], Stage (&dst)[LOADS]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) dst[i] = ld_stage(base + static_cast<uint64_t>(static_cast<uint32_t>(ids[i])) * row_stride());
  };
  auto put_k = [&](int buf, const Stage (&src)[LOADS]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int row = st_r + ROWS_PER_PASS * i;
      sm.k[buf][row * CPR + (st_c ^ Lds::k_swz(row))] = widen(src[i]);
    }
  };
  auto put_v = [&](int buf, const Stage (&src)[LOADS]) __attribute__((always_inline)) {
    unsigned char* base = reinterpret_cast<unsigned char*>(sm.v[buf]) + (DMA ? (st_c ^ Lds::v_swz(st_r)) * 16 : (st_c >> 2) * Lds::kVSub + (st_c & 3) * 16);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) *reinterpret_cast<U4*>(base + (st_r + ROWS_PER_PASS * i) * (DMA ? 2 * D : 64)) = widen(src[i]);
  };
  // (behind rows_landed(): the compiler takes ids to be on their way still, and would wait in the next step for what that has asked for since)
  auto held_ids = [&](int32_t (&ids)[LOADS]) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < LOADS; ++i) asm volatile("" : "+v"(ids[i]));
  };
  // piece i of the rows `ids` of one image, asked for
  auto send = [&](const unsigned char* base, int32_t id, const U4* image, int i) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) const U4* lds_t;
    uint32_t wave = to_lds;
    if constexpr (STAYS) asm volatile("" : "+s"(wave));
    rows_to_lds(base + static_cast<uint64_t>(static_cast<uint32_t>(id)) * row_stride(),
                static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_t)(image))) + wave + i * (64 * NWV * 16));
  };
  // ---- prologue: K(0), K(1), V(0) go to LDS in one round trip; K(2) and V(1) are asked for; ids of tiles 2 / 3 held.
  // (DMA: a step asks for V(t + 1) and K(t + 2) itself, the ids of tiles 1 / 2 are held.)
  // (Tiles behind the end of the walk: load_idx clamps to the walk's last row, nobody reads those images.) ----------
  // STAYS: the next query tile's rows (kst, k1st, vst) and queries are asked for while this one is walked.
  int32_t id1[LOADS];
  Stage k1st[LOADS];
  auto first_rows = [&](int head, int64_t q_at, int q_len) __attribute__((always_inline)) {      // (queue->ids holds the slots)
    const int c = thread() % CPR;
    const unsigned char* kr = head_rows(p.k_cache, head, c);
    const unsigned char* vr = head_rows(p.v_cache, head, c);
    int32_t id0[LOADS];
#pragma unroll
    for (int i = 0; i < LOADS; ++i) {
      const int32_t* ids = queue->ids + thread() / CPR + ROWS_PER_PASS * i;
      id0[i] = ids[0];
      id1[i] = ids[kKvTile];
      (DMA ? idx_k : idx_v)[i] = ids[2 * kKvTile];
      if constexpr (!DMA) idx_k[i] = ids[3 * kKvTile];
    }
    load_rows(kr, id0, kst);
    load_rows(kr, id1, k1st);
    load_rows(vr, id0, vst);
    // (a row beyond the tile's tokens takes its last token's queries: all its keys are masked)
    row_of(thread());
    const uint16_t* qp = p.q + (q_at + (r_tok < q_len ? r_tok : q_len - 1)) * p.q_stride + (head * p.group + r_hg) * D + (thread() >> 5 & 1) * 8;
#pragma unroll
    for (int s = 0; s < KS; ++s) qreg[s] = ld16(qp + s * 16);
  };
  if constexpr (!STAYS && DMA) {
    int32_t id0[LOADS];
    load_idx(0, id0);
    load_idx(1, idx_v);
    load_idx(2, idx_k);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) send(k_rows, id0[i], sm.k[0], i);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) send(k_rows, idx_v[i], sm.k[1], i);
#pragma unroll
    for (int i = 0; i < LOADS; ++i) send(v_rows, id0[i], sm.v[0], i);
    rows_landed();
    held_ids(idx_v);
    held_ids(idx_k);
    __syncthreads();
  } else if constexpr (!STAYS) {
    Stage k0[LOADS], v0[LOADS];
    int32_t id0[LOADS];
    load_idx(0, id0);
    load_idx(1, id1);
    load_rows(k_rows, id0, k0);
    load_rows(k_rows, id1, k1st);
    load_rows(v_rows, id0, v0);
    load_idx(2, idx_v);
    load_idx(3, idx_k);
    put_k(0, k0);
    put_k(1, k1st);
    put_v(0, v0);
    load_rows(k_rows, idx_v, kst);                   // K(2): written at the top of step 0
    load_rows(v_rows, id1, vst);                     // V(1): same
    __syncthreads();
  }

  // ---- STAYS: the tile taken next.  Taken eight to nine steps before the end of this one, handed to all waves two steps later, looked up another
  // two later, its slots left in LDS another two later; its rows travel under the last step and the epilogue. ----
  bool more = false;                                 // there is one
  int n_b = 0, n_kvh = 0, n_tile = 0;
  int32_t held = 0;                                  // what is on its way: the count of tiles taken (thread 0), a slot id
  auto take = [&]() __attribute__((always_inline)) {
    if (thread() == 0) held = static_cast<int32_t>(__hip_atomic_fetch_add(p.grabbed + (blockIdx.x & 7), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  };
  auto hand = [&]() __attribute__((always_inline)) {
    if (thread() == 0) queue->next = 8 * (static_cast<int>(gridDim.x / 8) + held) + static_cast<int>(blockIdx.x & 7);
  };
  int n_q0 = 0, n_len = 0;                           // its tokens
  int64_t n_at = 0;
  auto slot_of = [&](const int32_t* base, int end) __attribute__((always_inline)) {
    const int x = thread(), tok = x < 4 * kKvTile ? x : 0;
    held = base[tok < end ? tok : end - 1];
  };
  auto look = [&]() __attribute__((always_inline)) {
    const int L = __builtin_amdgcn_readfirstlane(queue->next);
    more = L < all;
    if (more) queue->find(L, top, p.batch, p.num_kv_heads, thread() & 63, n_b, n_kvh, n_tile);
    const int32_t* base = idx_base;
    int end = 0;
    if (more) {
      const int len = __builtin_amdgcn_readfirstlane(queue->len[n_b]), keys = __builtin_amdgcn_readfirstlane(queue->kv_len[n_b]);
      const int pre = __builtin_amdgcn_readfirstlane(queue->prefix[n_b]);
      base = p.req_to_token + __builtin_amdgcn_readfirstlane(queue->row[n_b]) * p.r2t_stride;
      n_q0 = n_tile * p.tokens_per_tile;
      n_len = len - n_q0 < p.tokens_per_tile ? len - n_q0 : p.tokens_per_tile;
      n_at = __builtin_amdgcn_readfirstlane(queue->q_begin[n_b]) + n_q0;
      end = causal && pre + n_q0 + n_len < keys ? pre + n_q0 + n_len : keys;
    }
    if (end <= 0) {                                  // nothing to read ahead: this tile's own rows once more
      base = idx_base;
      end = kv_end;
      n_len = q1 - q0;
      n_at = q_begin + q0;
      if (!more) n_kvh = kvh;
    }
    if (end > 0) slot_of(base, end);
  };
  auto leave = [&]() __attribute__((always_inline)) {
    const int x = thread();
    if (x < 4 * kKvTile) queue->ids[x] = held;
  };
  auto from_scratch = [&]() __attribute__((always_inline)) {                // this tile's first rows, nothing read ahead
    if (n_tiles > 0) {
      staging();
      slot_of(idx_base, kv_end);
      leave();
      __syncthreads();
      first_rows(kvh, q_begin + q0, q1 - q0);
    }
  };
  if constexpr (STAYS) from_scratch();

  for (;;) {                                         // (STAYS: the tiles of the workgroup)
  if constexpr (STAYS) {
    if (empty) {                                     // no key: zeros, and the next tile from scratch
      if (row_ok) put_zeros();
      take();
      hand();
      __syncthreads();
      look();
      __syncthreads();
      if (!more) return;
      kvh = n_kvh;
      of_queue(n_b, n_tile);
      place();
      empty = n_tiles <= 0;
      from_scratch();
      continue;
    }
    staging();
    if (n_tiles < 9) take();                         // too few steps to hide it all
    rows_of(kvh);
    put_k(0, kst);
    put_k(1, k1st);
    put_v(0, vst);
    if constexpr (DMA) {
#pragma unroll
      for (int i = 0; i < LOADS; ++i) idx_v[i] = id1[i];
      held_ids(idx_k);
    } else {
      load_rows(k_rows, idx_v, kst);
      load_rows(v_rows, id1, vst);
    }
    __syncthreads();
  }
  if constexpr (STAYS) fresh();
  f32x16_t s_a[2], s_b[2];                           // the two score sets: tile t and tile t + 1 trade places every step
  U4 pp[4];                                          // bf16(P(t)): [2 blk + ks] -> the 16 keys of one PV k-step
#pragma unroll
  for (int i = 0; i < 4; ++i) pp[i] = U4{0u, 0u, 0u, 0u};
#ifdef EXT_TRACE
  uint64_t tacc[6] = {0, 0, 0, 0, 0, 0};            // [commit, phase 1, mask, phase 2, decision, barrier] clocks over the walk
  uint64_t tprev = __builtin_readcyclecounter();
  const uint64_t tstart = tprev;
#endif

  auto read_k = [&](const U4* kimg, int i) __attribute__((always_inline)) {   // product i = (block i & 1, k-step i >> 1)
    const int row = (i & 1) * 32 + l31;
    return kimg[row * CPR + ((2 * (i >> 1) + hi) ^ Lds::k_swz(row))];
  };
  // mask (when the tile needs it), the row maximum of the lane pair, and the rescale decision for tile t: m_run, l_run
  // and O move to the new maximum together.  `links_done`: the in-lane maxima of registers 4..15 are in m4 already.
  auto mask_tile = [&](f32x16_t (&sc)[2], int t) __attribute__((always_inline)) {
    const int kv0 = t * kKvTile;
    if (__ballot(kv0 + kKvTile > row_limit) != 0ull) {                      // wave-uniform
      // the sentinel goes in BEFORE the scale: exp2(sentinel * scale - m) = 0 whatever m is
#pragma unroll
      for (int bk = 0; bk < 2; ++bk)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int kvpos = kv0 + 32 * bk + (r & 3) + 8 * (r >> 2) + 4 * hi;
          sc[bk][r] = kvpos < row_limit ? sc[bk][r] : kNegBig;
        }
    }
  };
  auto decide = [&](const float (&m4)[4], float psum) __attribute__((always_inline)) {
    const float mraw = fmaxf(fmaxf(m4[0], m4[1]), fmaxf(m4[2], m4[3]));
    float mx = mraw > 0.5f * kNegBig ? mraw * p.scale_log2 : kNegBig;      // a row with every key masked keeps the sentinel
    mx = lane_pair_max(mx);
    l_run += psum;
    if (__ballot(mx > m_run + kDeferMax) != 0ull) {                         // wave-uniform
      const float m_new = fmaxf(m_run, mx);
      const float alpha = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int n = 0; n < ND; ++n) ot[n] *= alpha;
    }
  };
  constexpr int LINKS = 24;                          // in-lane maxima behind the first four: registers 4..15 of both blocks
  auto link = [&](const f32x16_t (&sc)[2], float (&m4)[4], int j) __attribute__((always_inline)) {
    const int bk = j / 12, r = 4 + j % 12;
    m4[r & 3] = fmaxf(m4[r & 3], sc[bk][r]);
  };

  // ---- S(0) and its decision stand alone; the barrier keeps step 0's write of K(2) off the image they read --------
  {
    U4 kf[3];
    kf[0] = read_k(sm.k[0], 0);
    kf[1] = read_k(sm.k[0], 1);
#pragma unroll
    for (int i = 0; i < 2 * KS; ++i) {
      if (i + 2 < 2 * KS) kf[(i + 2) % 3] = read_k(sm.k[0], i + 2);
      f32x16_t acc = s_a[i & 1];
      if (i < 2) {
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[r] = 0.f;
      }
      s_a[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(kf[i % 3]), as_frag(qreg[i >> 1]), acc, 0, 0, 0);
    }
    mask_tile(s_a, 0);
    float m4[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) m4[c] = fmaxf(s_a[0][c], s_a[1][c]);
#pragma unroll
    for (int j = 0; j < LINKS; ++j) link(s_a, m4, j);
    decide(m4, 0.f);
  }
  __syncthreads();

  // request j of step t (of 3 LOADS)
  auto request_of = [&](int t, int j) __attribute__((always_inline)) {
    if constexpr (DMA) {                            // ids of tile t + 3, V(t + 1), K(t + 2): landed in front of the barrier
      if (j < LOADS) {
        const int last = kv_end - 1, tok = (t + 3) * kKvTile + st_r + ROWS_PER_PASS * j;
        idx_n[j] = idx_base[tok > last ? last : tok];
      } else if (j < 2 * LOADS) {
        send(v_rows, idx_v[j - LOADS], sm.v[(t + 1) & 1], j - LOADS);
      } else {
        send(k_rows, idx_k[j - 2 * LOADS], sm.k[t & 1], j - 2 * LOADS);
      }
    } else if (j < LOADS) {
      vst[j] = ld_stage(v_rows + static_cast<uint64_t>(static_cast<uint32_t>(idx_v[j])) * row_stride());
    } else if (j < 2 * LOADS) {
      if (j == LOADS) {
#pragma unroll
        for (int i = 0; i < LOADS; ++i) idx_v[i] = idx_k[i];          // the ids of K(t + 3) are those of V(t + 3) a step on
      }
      kst[j - LOADS] = ld_stage(k_rows + static_cast<uint64_t>(static_cast<uint32_t>(idx_k[j - LOADS])) * row_stride());
    } else {
      const int last = kv_end - 1;
      const int tok = (t + 4) * kKvTile + st_r + ROWS_PER_PASS * (j - 2 * LOADS);
      idx_k[j - 2 * LOADS] = idx_base[tok > last ? last : tok];
    }
  };

  // A wave without rows (behind the last token of a request's last tile; 44 tokens of one query head leave two of four) asks for its rows of the tiles and
  // leaves its SIMD to the other workgroup's.  us, all waves walking / this: 30 x 44 behind one prefix of 833, 32 / 32 heads, 66.9 / 64.3; where the rows of the keys
  // bound (16 x 40 behind 1500 each) equal.  (Not for e4m3 rows: 109 registers spilled, 74 behind 5452 39 / 42.)
  if constexpr (PARTS && DMA) {
    if (__ballot(row_ok) == 0ull) {                  // (wave-uniform)
      for (int t = 0; t + 1 < n_tiles; ++t) {
#pragma unroll
        for (int j = 0; j < 3 * LOADS; ++j) request_of(t, j);
        rows_landed();
        held_ids(idx_n);
#pragma unroll
        for (int i = 0; i < LOADS; ++i) {
          idx_v[i] = idx_k[i];
          idx_k[i] = idx_n[i];
        }
        __syncthreads();
      }
      __syncthreads();
      return;
    }
  }

  auto step = [&](int t, f32x16_t (&sc)[2], f32x16_t (&sn)[2], auto have_next_tag) __attribute__((always_inline)) {
    constexpr bool HAVE_NEXT = decltype(have_next_tag)::value;
    // ---- what was asked for a step ago goes to LDS: K(t + 2), V(t + 1) -- images nobody reads before the barrier below.
    // (Between the phases instead, with the requests beside the phase-2 products: same time per tile, the wait moves
    // with the writes; and the registers no longer fit.)
    // (STAYS: in the last step kst and vst hold the next query tile's rows)
    if constexpr (!DMA && (!STAYS || HAVE_NEXT)) {
      put_k(t & 1, kst);
      put_v((t + 1) & 1, vst);
    }
    EXT_T(0);
    // (8 waves: in phase 1, where most vector instructions are, a wave goes first; the SIMD's other wave has matrix instructions to issue
    // beside them when it is in phase 2, and the older of two waves in phase 1 no longer holds the younger back: 696 -> 665 us for 12.6 k
    // cold tokens of six requests, 64 / 8 heads, 406 -> 394 for 4096 behind 4000, 171 -> 166 for 60 x 128 behind 896.  Two workgroups of 4 waves a CU lose by it, 183 -> 203.)
    if constexpr (NWV == 8) __builtin_amdgcn_s_setprio(1);
    // ---- phase 1 ------------------------------------------------------------------------------------------
    constexpr int KF = 3;                            // K fragment sets: reads run two products ahead (1 or 3 ahead: same time)
    constexpr int G1 = 2 * KS;                       // products (16 at D = 128)
    constexpr int SPP = 32 / G1;                     // scores exponentiated beside each (2 at D = 128, 4 at D = 64)
    const float neg_m = m_run > 0.5f * kNegBig ? -m_run : 0.f;   // rows without a key so far: exp2(sentinel * scale) = 0
    float psum = 0.f;
    {
      // the staging registers are free again: V(t + 2) rows, K(t + 3) rows, the ids of tile t + 4 -- one request per
      // RSTRIDE products (in one burst the eight waves' requests queue for the CU's one address unit)
      constexpr int NREQ = 3 * LOADS;
      constexpr int RSTRIDE = G1 / NREQ > 0 ? G1 / NREQ : 1;
      static_assert(NREQ * RSTRIDE <= G1, "requests fit the products of phase 1");
      auto request = [&](int j) __attribute__((always_inline)) { request_of(t, j); };
      // the exponentials as a three-stage software pipeline:  A(i) scale + subtract,  B(i) exp2,  C(i) sum + pack
      float ta[SPP], eb[SPP];
      auto stage_a = [&](int i) __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < SPP; ++j) {
          const int x = SPP * i + j;                 // flat score index: block x >> 4, register x & 15
          ta[j] = fmaf(sc[x >> 4][x & 15], p.scale_log2, neg_m);
        }
      };
      auto stage_b = [&]() __attribute__((always_inline)) {
#pragma unroll
        for (int j = 0; j < SPP; ++j) eb[j] = fast_exp2(ta[j]);
      };
      auto stage_c = [&](int i) __attribute__((always_inline)) {
        uint32_t* pw = reinterpret_cast<uint32_t*>(pp);
#pragma unroll
        for (int j = 0; j < SPP; j += 2) {
          psum += eb[j] + eb[j + 1];
          pw[(SPP * i + j) >> 1] = pack_bf2(eb[j], eb[j + 1]);   // word (x & 7) >> 1 of pp[x >> 3]
        }
      };
      const U4* kimg = sm.k[(t + 1) & 1];
      U4 kf[KF];
      if constexpr (HAVE_NEXT) {
#pragma unroll
        for (int i = 0; i < KF - 1; ++i) kf[i] = read_k(kimg, i);
      }
      stage_a(0);
#pragma unroll
      for (int i = 0; i < G1; ++i) {
        if constexpr (HAVE_NEXT) {
          if (i + KF - 1 < G1) kf[(i + KF - 1) % KF] = read_k(kimg, i + KF - 1);
          f32x16_t acc = sn[i & 1];
          if (i < 2) {
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[r] = 0.f;
          }
          sn[i & 1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(kf[i % KF]), as_frag(qreg[i >> 1]), acc, 0, 0, 0);
          if (i % RSTRIDE == 0 && i / RSTRIDE < NREQ) request(i / RSTRIDE);
        }
        if (i >= 1) stage_c(i - 1);
        stage_b();
        if (i + 1 < G1) stage_a(i + 1);
        if constexpr (HAVE_NEXT || STAYS) __builtin_amdgcn_sched_barrier(0);   // groups stay as written
      }
      stage_c(G1 - 1);
      // P(t) and its sum are "used" here: hipcc otherwise sinks the exponential stream below later branches
      asm volatile("" : "+v"(psum));
#pragma unroll
      for (int i = 0; i < 4; ++i) asm volatile("" : "+v"(pp[i].x), "+v"(pp[i].y), "+v"(pp[i].z), "+v"(pp[i].w));
    }
    if constexpr (NWV == 8) __builtin_amdgcn_s_setprio(0);
    EXT_T(1);
    if constexpr (HAVE_NEXT) mask_tile(sn, t + 1);
    EXT_T(2);
    // ---- phase 2 ------------------------------------------------------------------------------------------
    float m4[4];
    {
      const unsigned char* vbase = reinterpret_cast<const unsigned char*>(sm.v[t & 1]);
      typedef __attribute__((address_space(3))) v4s16_t* lds_v4_t;
      auto read_v = [&](int i) __attribute__((always_inline)) {   // product i = (output block i % ND, k-step i / ND of the tile)
        constexpr int kRow = DMA ? 2 * D : 64;       // bytes from token to token
        const unsigned char* a = vbase + (DMA ? v_lane[DMA ? i % ND : 0] : v_lane[0] + (i % ND) * Lds::kVSub) + (i / ND) * (16 * kRow);
        const v4s16_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(a));
        const v4s16_t hi4 = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(a + 8 * kRow));
        U4 o;
        o.x = __builtin_bit_cast(uint2, lo).x; o.y = __builtin_bit_cast(uint2, lo).y;
        o.z = __builtin_bit_cast(uint2, hi4).x; o.w = __builtin_bit_cast(uint2, hi4).y;
        return o;
      };
      constexpr int LSTART = NPV / 4;                // the first products run while the last S^T products still finish
      constexpr int PER = LINKS / (NPV - LSTART);    // maxima per product behind them (2 at D = 128, 4 at D = 64)
      static_assert(PER * (NPV - LSTART) == LINKS, "maxima spread evenly");
      U4 vf[3];
      vf[0] = read_v(0);
      vf[1] = read_v(1);
#pragma unroll
      for (int i = 0; i < NPV; ++i) {
        if (i + 2 < NPV) vf[(i + 2) % 3] = read_v(i + 2);
        ot[i % ND] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(as_frag(vf[i % 3]), as_frag(pp[i / ND]), ot[i % ND], 0, 0, 0);
        if constexpr (HAVE_NEXT) {
          if (i == LSTART) {
#pragma unroll
            for (int c = 0; c < 4; ++c) m4[c] = fmaxf(sn[0][c], sn[1][c]);
          }
          if (i >= LSTART) {
#pragma unroll
            for (int j = PER * (i - LSTART); j < PER * (i - LSTART + 1); ++j) link(sn, m4, j);
          }
        }
        if constexpr (HAVE_NEXT || STAYS) __builtin_amdgcn_sched_barrier(0);
      }
    }
    EXT_T(3);
    // ---- the decision for tile t + 1: P(t) is inside O and l, nothing at the new maximum exists yet ----------
    if constexpr (HAVE_NEXT) decide(m4, psum);
    else l_run += psum;
    EXT_T(4);
    if constexpr (DMA && HAVE_NEXT) {
      rows_landed();
      held_ids(idx_n);
#pragma unroll
      for (int i = 0; i < LOADS; ++i) {
        idx_v[i] = idx_k[i];
        idx_k[i] = idx_n[i];
      }
    }
    __syncthreads();
    EXT_T(5);
  };
  {
    int t = 0;
    const int t_take = n_tiles >= 9 ? (n_tiles - 9) & ~1 : -8;
    if constexpr (STAYS) {
      if (n_tiles < 9) {                               // (taken in front of the first scores)
        hand();
        __syncthreads();
        look();
        leave();
        __syncthreads();
      }
      staging();
    }
    for (; t + 2 < n_tiles; t += 2) {
      if constexpr (STAYS) {
        if (__builtin_expect(t >= t_take, 0)) {
          if (t == t_take) take();
          else if (t == t_take + 2) hand();
          else if (t == t_take + 4) look();
          else if (t == t_take + 6) leave();
        }
      }
      step(t, s_a, s_b, std::true_type{});
      step(t + 1, s_b, s_a, std::true_type{});
    }
    if constexpr (STAYS) {                             // (one last step for both: a copy of the scores costs less than its code twice)
      staging();
      if (n_tiles - t == 2) {
        step(t, s_a, s_b, std::true_type{});
        s_a[0] = s_b[0];
        s_a[1] = s_b[1];
        ++t;
        staging();
      }
      first_rows(n_kvh, n_at, n_len);
      __builtin_amdgcn_sched_barrier(0);
      step(t, s_a, s_b, std::false_type{});
    } else if (n_tiles - t == 2) {
      step(t, s_a, s_b, std::true_type{});
      step(t + 1, s_b, s_a, std::false_type{});
    } else {
      step(t, s_a, s_b, std::false_type{});
    }
  }
#ifdef EXT_TRACE
  if (g_ext_trace && lane == 0) {
    uint64_t* o = g_ext_trace + static_cast<int64_t>(blockIdx.x) * 64 + wid * 8;
    for (int i = 0; i < 6; ++i) o[i] = tacc[i];
    o[6] = n_tiles;
    o[7] = tstart;
  }
#endif

  // ---- epilogue: lane (q, h) holds O^T[d = 32 n + 8 c + 4 h + e][q], c = 0..3, e = 0..3.  The lane halves trade
  // 4-dim pieces (v_permlane32_swap on the packed words) so that h = 0 owns the 8 dims of c = 0, 2 and h = 1 those of
  // c = 1, 3: eight 16-byte stores per lane instead of sixteen 8-byte ones ------------------------------------
  const float l = lane_pair_sum(l_run);
  if constexpr (STAYS || PARTS) {                    // (again: not kept across the walk)
    int x = threadIdx.x;
    asm volatile("" : "+v"(x));
    row_of(x);
    row_ok = r_tok < q1 - q0;
    row_off = (kvh * p.group + r_hg) * D;
  }
  if constexpr (PARTS) {
    if (p.parts > 1) {                                 // unnormalised rows for extend_merge_kernel
      if (row_ok) {
        const int64_t row = part * p.part_rows + static_cast<int64_t>(q_begin + q0 + r_tok) * (p.num_kv_heads * p.group) + kvh * p.group + r_hg;
        float* acc = p.part_acc + row * D + 4 * hi;
#pragma unroll
        for (int n = 0; n < ND; ++n)
#pragma unroll
          for (int c = 0; c < 4; ++c)
            *reinterpret_cast<f32x4_t*>(acc + 32 * n + 8 * c) = f32x4_t{ot[n][4 * c], ot[n][4 * c + 1], ot[n][4 * c + 2], ot[n][4 * c + 3]};
        if (hi == 0) {
          p.part_ml[2 * row] = m_run;
          p.part_ml[2 * row + 1] = l;
        }
      }
      return;
    }
  }
  const float inv = (l > 0.f) ? p.v_scale / l : 0.f;
  uint16_t* op = p.out + static_cast<int64_t>(q_begin + q0 + r_tok) * p.out_stride + row_off;
#pragma unroll
  for (int n = 0; n < ND; ++n) {
#pragma unroll
    for (int cp = 0; cp < 2; ++cp) {                  // the piece pair (c = 2 cp, c = 2 cp + 1)
      uint32_t a0 = pack_bf2(ot[n][8 * cp + 0] * inv, ot[n][8 * cp + 1] * inv);
      uint32_t a1 = pack_bf2(ot[n][8 * cp + 2] * inv, ot[n][8 * cp + 3] * inv);
      uint32_t b0 = pack_bf2(ot[n][8 * cp + 4] * inv, ot[n][8 * cp + 5] * inv);
      uint32_t b1 = pack_bf2(ot[n][8 * cp + 6] * inv, ot[n][8 * cp + 7] * inv);
      // swap: upper half of a <-> lower half of b.  Afterwards a = dims 0-3, b = dims 4-7 of the lane's own piece
      asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a0), "+v"(b0));
      asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a1), "+v"(b1));
      if (row_ok) {
        U4 w;
        w.x = a0; w.y = a1; w.z = b0; w.w = b1;
        *reinterpret_cast<U4*>(op + n * 32 + (2 * cp + hi) * 8) = w;
      }
    }
  }
  if (!STAYS || !more) return;
  kvh = n_kvh;
  of_queue(n_b, n_tile);
  place();
  empty = n_tiles <= 0;
  }
}

template <int D, int NWV, bool FP8>
__global__ __launch_bounds__(64 * NWV, 2) void extend_attention_pipe_kernel(ExtendParams p) {
  __shared__ SmemLadder<D, FP8> sm;
  extend_pipe_body<D, NWV, FP8, false>(p, sm);
}

// 256 workgroups that stay and take the query tiles of a large launch of mixed contexts from the queue, longest contexts first.  A launch deals its
// workgroups by query tile alone, whatever stands in front of them, and hands out empty ones for the shorter requests; a workgroup of this shape has its CU
// alone, so that nothing covers its prologue (lengths, slot ids, rows, one behind the other: 10 000 clocks beside a walk of 60 000 to 76 000).  Here the next
// tile's slots, rows and queries travel under the walk of this one and the longest contexts end first.  The same instructions a tile, the same bits.
// p.grabbed: eight counters, zero at the launch.  Figures at extend_ragged().  Formed anew for each tile (thread(), staging()): lane constants and what the
// compiler makes of them; kept across the outer loop they spilled 20 to 400 registers around the walk.
template <bool FP8>
__global__ __launch_bounds__(512, 2) void extend_attention_walk_kernel(ExtendParams p) {
  __shared__ struct {
    SmemLadder<128, FP8> sm;
    WalkQueue queue;
  } lds;
  extend_pipe_body<128, 8, FP8, false, true>(p, lds.sm, &lds.queue);
}

// The same walk by four waves (128 rows, two workgroups a CU), with a request's key tiles dealt over p.parts workgroups.  Few new tokens
// behind a long context leave most of the chip idle otherwise, and what runs is a serial chain of tiles.  Each part leaves unnormalised
// fp32 rows that extend_merge_kernel joins; a single part writes the output itself.
// Measured (us; general 4-wave kernel -> this one): 203 tokens behind 3800, 32 / 8 heads: 168 -> 33 in four parts; 22 x 3 behind 4549,
// 32 / 32 heads: 210 -> 53 in five; 1000 cold: 53 -> 23.5 in one part; 16 x 20 behind 500: 31 -> 18.5 in one.
// (Two groups of four waves a workgroup, half of a part's tiles each, joined in LDS: 63 tiles in one part 80 -> 65, but two waves a SIMD need 4300 clocks for
// two tiles where one needs 2700 for one, and with parts to choose from 90 drawn launches gained 0.8 %.)
constexpr int kPartWaves = 4;

// How many parts, from what a launch of them costs (us).  A workgroup walks its tiles in about 1.35 us each (1.05 at head dim 64; bf16 rows a tenth
// less) and pays four more for its first fetches; up to 256 workgroups have a CU alone, two on a CU take 0.65 of the time of one behind the
// other.  The merge is a launch (5 us), half a microsecond a part, and the parts' fp32 rows through the caches at about 6 TB/s.
// Against the best of 1, 2, 3, 4, 5, 6, 8 .. 16 parts this picks 1.8 % above it on the mean of 90 drawn launches, 14 % at worst.
int extend_parts(int64_t wgs, int64_t rows, int max_kv_len, int head_dim) {
  const int tiles = (max_kv_len + kKvTile - 1) / kKvTile;
  const double tile_us = head_dim == 128 ? 1.35 : 1.05;
  int best = 1;
  double best_us = 0;
  for (int n = 1; n <= 16 && n <= tiles; ++n) {
    const double per_cu = static_cast<double>((wgs * n + 255) / 256);
    const double crowd = per_cu > 1 ? 0.65 * per_cu : 1.0;
    double us = tile_us * ((tiles + n - 1) / n + 4) * crowd;
    if (n > 1) us += 5.0 + 0.5 * n + static_cast<double>(rows) * n * head_dim * 8.0 / 6e6;
    if (n == 1 || us < best_us) {
      best = n;
      best_us = us;
    }
  }
  return best;
}

// The 8-wave kernel (256 rows) or the 4-wave one for a launch of one part.  Eight waves ask for half the key rows per flop; four
// waste fewer rows of a last tile and, two workgroups a CU, leave less of the chip idle in the last round (about 0.3 of a round
// where eight leave up to a whole one), at 7 % more per round.  Past two rounds the key rows decide (44 ragged extends of 122 behind 1874
// 289 / 302 us, 60 x 128 behind 896 182 / 197), unless the second half of a 256-row tile would be empty anyway (64 x 20 behind 3000 231 / 161).
// Below (us, eight / four): 5 x 600 behind 1000 92 / 87, 8 x 300 behind 1000, 32 kv heads 102 / 85, 4 x 1024 cold 52 / 54.  At D = 64 four
// waves were never slower (6 x 2000 cold 82 / 76, 4 x 1024 cold 29 / 23).
// The counts are of the longest request's tiles.  Up to two rounds of those, where the launch knows its tokens, a request's last tile is
// taken to be half full instead (6 ragged extends of 77 .. 271 behind 2862, 32 kv heads: 110 / 115, and the padded counts say four); past
// them ragged batches stay with eight (8 of 60 .. 314 behind 1500, 64 / 8 heads: 112 / 121, and the held counts say four).
bool extend_eight_waves(int64_t tokens, int64_t batch, int64_t rows, int group, int kv_heads, int head_dim) {
  auto padded = [&](int tile) { return (rows + tile - 1) / tile * batch * kv_heads; };
  auto held = [&](int tile) {
    const int64_t n = (2 * tokens * group + batch * tile) / (2 * tile) * kv_heads;
    return tokens > 0 && n < padded(tile) ? n : padded(tile);
  };
  constexpr int kFour = 32 * kPartWaves;
  if (padded(256) < 256 || head_dim != 128 || padded(kFour) * 4 <= padded(256) * 5) return false;
  return padded(256) > 512 || static_cast<double>((held(256) + 255) / 256) <= 1.07 * (static_cast<double>(held(kFour)) / 512.0 + 0.3);
}

// Whether a launch of eight waves can be one of workgroups that stay: more query tiles than CUs (ragged batches counted as held() does above).
int64_t extend_held(int64_t tokens, int64_t batch, int group, int kv_heads) { return (2 * tokens * group + batch * 256) / 512 * kv_heads; }
bool extend_walks(int64_t tokens, int64_t batch, int64_t rows, int group, int kv_heads, int head_dim) {
  if (head_dim != 128 || tokens <= 0 || batch > WalkQueue::kRequests || group > 256 || !extend_eight_waves(tokens, batch, rows, group, kv_heads, head_dim)) return false;
  if (rows / group > static_cast<int64_t>(256 / group) * WalkQueue::kLevels) return false;       // a request's tiles stand at levels of their own
  return extend_held(tokens, batch, group, kv_heads) > 256;
}
// Whether it pays, from the sums that the caller has.  It saves the wait for a long context that a launch deals last, empty workgroups and hidden prologues;
// it costs 3 % a step, and where walks are over before the next tile has arrived (eight key tiles and fewer) two barriers and a look at the list a tile.
// So: never while all contexts are about as long (mean over longest above 0.92); where the longest prefix stands 512 keys and more above the mean one;
// else where a CU walks key tiles enough to pay for the ends: 12, or 24 with less to balance (mean over longest above 0.7).  A
// query head to a kv head, whose heads share no rows: only where the longest prefix stands apart by 1024 (without that -3 to +2 %).
// us, launched / staying: 6 cold prompts of 1.1 - 3.1 k, 64 / 8 heads, 662 / 606, 12 of 60 - 3000 behind 10 - 6000 1322 / 745, 30 of 200 behind 10 - 1000 87 / 80,
// 40 of 237 and 200 behind 1500 126 / 89, 24 of 140 - 560 93 / 83.  Launched: 30 of 200 behind 300 and a cold one of 700 111 / 115, 8 of 490 - 910, 32 / 32
// heads, 113 / 119.  The lines cannot tell every batch: of 2400 drawn ones (3 to 90 requests of 60 to 1600 new tokens, cold, behind one prefix, behind
// log-uniform ones, one long request among short ones; three in ten in e4m3) 3.4 % are slower than launched by more than 2 %, worst 0.89 (8.9 % and 0.79 with
// lines on the longest context, at 640 and 400 tokens); over all of them launching takes 1.057 times as long.
bool extend_ragged(int64_t held, int64_t batch, int64_t num_tokens, int64_t sum_kv_len, int max_extend_len, int max_kv_len, int group) {
  const int64_t longest = batch * max_kv_len;
  if (sum_kv_len <= 0 || sum_kv_len * 100 > longest * 92) return false;
  const int64_t apart = longest - batch * max_extend_len - (sum_kv_len - num_tokens);            // times batch
  const int64_t walked = held * (2 * sum_kv_len - num_tokens) / (batch * 2 * kKvTile * 256);      // key tiles a CU: the mean prefix and half of the mean extend
  if (group == 1) return apart >= 1024 * batch;
  return (apart >= 512 * batch && walked >= 8) || walked >= (sum_kv_len * 100 <= longest * 70 ? 12 : 24);
}

template <int D, bool FP8>
__global__ __launch_bounds__(64 * kPartWaves, D > 64 ? 2 : 3) void extend_attention_parts_kernel(ExtendParams p) {
  __shared__ SmemLadder<D, FP8> sm;
  extend_pipe_body<D, kPartWaves, FP8, true>(p, sm);
}

// out = sum_i e^{m_i - m} acc_i / sum_i e^{m_i - m} l_i: a (token, head) row is D / 8 lanes, 8 dims each.  Rows outside the requests'
// tokens stay untouched; a part without keys for the row (sum 0) is not read, one whose sum is NaN makes the row NaN as in one part.
template <int D>
__global__ __launch_bounds__(256) void extend_merge_kernel(ExtendParams p) {
  constexpr int LPR = D / 8;
  const int heads = p.num_kv_heads * p.group;
  const int64_t row = (static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x) / LPR;
  const int c = threadIdx.x % LPR;
  const int64_t tok = row / heads;
  if (row >= p.part_rows || tok < p.qo_indptr[0] || tok >= p.qo_indptr[p.batch]) return;
  float m = kNegBig;
  for (int i = 0; i < p.parts; ++i) m = fmaxf(m, p.part_ml[2 * (i * p.part_rows + row)]);
  float o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f}, l = 0.f;
  for (int i = 0; i < p.parts; ++i) {
    const float* ml = p.part_ml + 2 * (i * p.part_rows + row);
    if (ml[1] == 0.f) continue;
    const float w = fast_exp2(ml[0] - m);
    const f32x4_t* a = reinterpret_cast<const f32x4_t*>(p.part_acc + (i * p.part_rows + row) * D + c * 8);
    const f32x4_t a0 = a[0], a1 = a[1];
    l += ml[1] * w;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      o[j] += a0[j] * w;
      o[4 + j] += a1[j] * w;
    }
  }
  const float inv = l > 0.f ? p.v_scale / l : 0.f;
  U4 w;
  w.x = pack_bf2(o[0] * inv, o[1] * inv);
  w.y = pack_bf2(o[2] * inv, o[3] * inv);
  w.z = pack_bf2(o[4] * inv, o[5] * inv);
  w.w = pack_bf2(o[6] * inv, o[7] * inv);
  *reinterpret_cast<U4*>(p.out + tok * p.out_stride + (row - tok * heads) * D + c * 8) = w;
}

// Test-only probe: C[16x16] = A[16x32] . B[32x16] with the operand/result lane
// maps this file assumes (A row = lane&15, k = 8*(lane>>4)+j; C row = 4*(lane>>4)+r,
// col = lane&15).  tests/ checks it against a plain matmul.
__global__ void mfma_probe_kernel(const uint16_t* __restrict__ a, const uint16_t* __restrict__ bm,
                                  float* __restrict__ c) {
  const int lane = threadIdx.x;
  const int l15 = lane & 15, g = lane >> 4;
  U4 af, bf;
  uint16_t* ap = reinterpret_cast<uint16_t*>(&af);
  uint16_t* bp = reinterpret_cast<uint16_t*>(&bf);
  for (int j = 0; j < 8; ++j) {
    ap[j] = a[l15 * 32 + g * 8 + j];          // A[i = l15][k = 8g + j]
    bp[j] = bm[(g * 8 + j) * 16 + l15];        // B[k = 8g + j][n = l15]
  }
  f32x4_t acc = {0.f, 0.f, 0.f, 0.f};
  acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(af), as_frag(bf), acc, 0, 0, 0);
  for (int r = 0; r < 4; ++r) c[(g * 4 + r) * 16 + l15] = acc[r];
}

}  // namespace

// test / tuning overrides (process-wide, set through sgl_amd_debug_extend_attention_shape; never read from the environment)
static int g_extend_debug_shape = 0;      // 0: automatic; 41 / 42 / 82: waves x M-tiles per wave
static int g_extend_debug_flags = 0;      // bit 0: bf16 8-wave launches stay on the general single-image kernel; bit 1: they take the ping-pong kernel

extern "C" {

int sgl_amd_debug_extend_attention_shape(int shape, int flags) {
  if (shape != 0 && shape != 41 && shape != 42 && shape != 82) {
    set_last_error("debug_extend_attention_shape: shape must be 0 (automatic), 41, 42 or 82");
    return -1;
  }
  g_extend_debug_shape = shape;
  g_extend_debug_flags = flags;
  return 0;
}

int sgl_amd_extend_attention(const void* q, void* out, const void* k_cache, const void* v_cache,
                             const int32_t* req_to_token, int64_t req_to_token_stride,
                             const int64_t* req_pool_indices, const int32_t* seq_lens,
                             const int32_t* prefix_lens, const int32_t* qo_indptr, int64_t batch,
                             int max_extend_len, int num_q_heads, int num_kv_heads, int head_dim,
                             int64_t q_token_stride, int64_t out_token_stride,
                             int64_t k_cache_row_stride, int64_t v_cache_row_stride, float sm_scale,
                             int causal, void* stream) {
  return sgl_amd_extend_attention_ex(q, out, k_cache, v_cache, req_to_token, req_to_token_stride, req_pool_indices, seq_lens,
                                     prefix_lens, qo_indptr, batch, max_extend_len, num_q_heads, num_kv_heads, head_dim,
                                     q_token_stride, out_token_stride, k_cache_row_stride, v_cache_row_stride, sm_scale, causal,
                                     0, 1.0f, 1.0f, 1, 0, -1, 0.0f, nullptr, nullptr, 0, stream);
}

static int extend_attention_any(const void* q, void* out, const void* k_cache, const void* v_cache,
                                const int32_t* req_to_token, int64_t req_to_token_stride,
                                const int64_t* req_pool_indices, const int32_t* seq_lens,
                                const int32_t* prefix_lens, const int32_t* qo_indptr, int64_t batch,
                                int max_extend_len, int num_q_heads, int num_kv_heads, int head_dim,
                                int64_t q_token_stride, int64_t out_token_stride,
                                int64_t k_cache_row_stride, int64_t v_cache_row_stride, float sm_scale,
                                int causal, int kv_fp8, float k_scale, float v_scale, int page_size, int kv_layout_hnd,
                                int sliding_window, float logit_cap, const void* custom_mask, const int64_t* mask_indptr,
                                int skip_prefix_custom_mask, int64_t num_tokens, int max_kv_len, int parts, void* ws_acc, void* ws_ml, void* stream,
                                unsigned* grabbed = nullptr) {

  SGL_CLEAR_STALE_ERROR();
  SGL_CHECK_ARG(k_cache_row_stride == v_cache_row_stride, "extend_attention: K and V pools must share a row stride");
  SGL_CHECK_ARG(!kv_fp8 || (k_scale > 0.f && v_scale > 0.f), "extend_attention: fp8 KV needs positive k_scale / v_scale");
  SGL_CHECK_ARG(logit_cap >= 0.f, "extend_attention: logit_cap must be >= 0 (0 = off)");
  SGL_CHECK_ARG((custom_mask == nullptr) == (mask_indptr == nullptr), "extend_attention: custom_mask and mask_indptr come together");
  SGL_CHECK_ARG(head_dim == 64 || head_dim == 128, "extend_attention: head_dim=%d not supported (64/128)", head_dim);
  SGL_CHECK_ARG(num_kv_heads > 0 && num_q_heads % num_kv_heads == 0,
                "extend_attention: num_q_heads=%d not a multiple of num_kv_heads=%d", num_q_heads, num_kv_heads);
  const int group = num_q_heads / num_kv_heads;
  SGL_CHECK_ARG(group <= kRows, "extend_attention: GQA group %d too large", group);
  SGL_CHECK_ARG(q_token_stride % 8 == 0 && out_token_stride % 4 == 0 && k_cache_row_stride % 8 == 0 && v_cache_row_stride % 8 == 0,
                "extend_attention: strides must keep 16-byte row alignment");
  SGL_CHECK_ARG(batch <= 65535 && num_kv_heads <= 65535, "extend_attention: grid too large");
  if (batch == 0 || max_extend_len <= 0) return 0;
  ExtendParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.out = static_cast<uint16_t*>(out);
  p.k_cache = static_cast<const uint16_t*>(k_cache);
  p.v_cache = static_cast<const uint16_t*>(v_cache);
  p.req_to_token = req_to_token;
  p.req_pool_indices = req_pool_indices;
  p.seq_lens = seq_lens;
  p.prefix_lens = prefix_lens;
  p.qo_indptr = qo_indptr;
  p.q_stride = q_token_stride;
  p.out_stride = out_token_stride;
  p.kc_stride = k_cache_row_stride;
  p.vc_stride = v_cache_row_stride;
  p.r2t_stride = req_to_token_stride;
  p.num_kv_heads = num_kv_heads;
  p.group = group;
  // Workgroup shape (waves x M-tiles per wave -> rows that share one staged K/V tile):
  //   32x32 kernels:   token-major pools without window, cap and mask: eight waves or four (extend_eight_waves), four with
  //                    the keys dealt over workgroups (extend_parts).  Only contexts of one tile are left to the general kernel,
  //                    whose 64-row workgroups spread them wider (37 cold tokens, 32 heads: 6.1 against 6.7 us);
  //   8 x 2 = 256 rows, two waves per SIMD and the whole register file: fewest K/V gathers per flop; measured
  //                    fastest on MI355X for every shape that gives each CU a workgroup (benchmarks/micro.py);
  //   4 x 1 =  64 rows, 3 workgroups / CU: short extends whose wider grids would leave CUs idle;
  //   4 x 2 = 128 rows: what is left (GQA groups above 64 on a small grid).
  const int64_t rows_total = static_cast<int64_t>(max_extend_len) * group;
  auto wgs = [&](int rows) { return ((rows_total + rows - 1) / rows) * num_kv_heads * batch; };
  int mtw = 2, nwv = 4;
  // eligible for the 32x32 kernels (flag bit 0, or a forced shape but 8 x 2: the general kernel)
  // (rows_to_lds() takes whole 16-byte pieces: bf16 pools that do not begin at one stay with the general kernel)
  const bool plain = !kv_layout_hnd && sliding_window < 0 && logit_cap == 0.f && custom_mask == nullptr && (g_extend_debug_flags & 1) == 0 &&
                     (kv_fp8 || ((reinterpret_cast<uintptr_t>(k_cache) | reinterpret_cast<uintptr_t>(v_cache)) & 15) == 0);
  const bool small = plain && g_extend_debug_shape == 0 && group <= 32 * kPartWaves && out_token_stride % 8 == 0 &&
                     !extend_eight_waves(num_tokens, batch, rows_total, group, num_kv_heads, head_dim) && !(max_kv_len > 0 && max_kv_len <= kKvTile);
  if (group <= 256 && wgs(256) >= 256) { mtw = 2; nwv = 8; }
  else if (group <= 64) { mtw = 1; nwv = 4; }
  if (const int v = g_extend_debug_shape) {                   // sgl_amd_debug_extend_attention_shape(): tests / tuning
    if (v == 41 && group <= 64) { nwv = 4; mtw = 1; }
    if (v == 42) { nwv = 4; mtw = 2; }
    if (v == 82) { nwv = 8; mtw = 2; }
  }
  p.tokens_per_tile = (nwv * 16 * mtw) / group;
  p.causal = causal;
  p.scale_log2 = sm_scale * 1.4426950408889634f * (kv_fp8 ? k_scale : 1.0f);
  p.v_scale = kv_fp8 ? v_scale : 1.0f;
  p.window = sliding_window;
  p.cap_log2 = logit_cap > 0.f ? logit_cap * 1.4426950408889634f : 0.f;
  p.inv_cap_log2 = logit_cap > 0.f ? 1.0f / p.cap_log2 : 0.f;
  p.custom_mask = static_cast<const uint8_t*>(custom_mask);
  p.mask_indptr = mask_indptr;
  p.mask_skip_prefix = skip_prefix_custom_mask ? 1 : 0;
  SGL_CHECK_ARG(make_kv_format(&p.fmt, k_cache_row_stride, num_kv_heads, head_dim, page_size, kv_layout_hnd, kv_fp8),
                "extend_attention: HND pools need a power-of-two page_size (got %d); row / page strides must stay below 4 GiB", page_size);
  const int tiles = (max_extend_len + p.tokens_per_tile - 1) / p.tokens_per_tile;
  dim3 grid(tiles, num_kv_heads, batch);
  hipStream_t st = as_stream(stream);
  // token-major pools (bf16 or e4m3 rows), 8-wave shape: the 32x32 two-score-set kernel (debug flag bit 1: the bf16
  // ping-pong kernel it replaced)
  if (small && (g_extend_debug_flags & 2) == 0) {
    p.tokens_per_tile = 32 * kPartWaves / group;
    p.num_tiles = (max_extend_len + p.tokens_per_tile - 1) / p.tokens_per_tile;
    p.batch = static_cast<int>(batch);
    p.parts = parts > 1 ? parts : 1;
    p.part_rows = num_tokens * num_q_heads;
    p.part_acc = static_cast<float*>(ws_acc);
    p.part_ml = static_cast<float*>(ws_ml);
    const int64_t blocks = static_cast<int64_t>(p.num_tiles) * num_kv_heads * batch * p.parts;
    SGL_CHECK_ARG(blocks < (int64_t{1} << 31), "extend_attention: grid too large");
    const dim3 grid4(static_cast<unsigned>(blocks));
    if (kv_fp8) {
      if (head_dim == 128) hipLaunchKernelGGL((extend_attention_parts_kernel<128, true>), grid4, dim3(64 * kPartWaves), 0, st, p);
      else hipLaunchKernelGGL((extend_attention_parts_kernel<64, true>), grid4, dim3(64 * kPartWaves), 0, st, p);
    } else if (head_dim == 128) hipLaunchKernelGGL((extend_attention_parts_kernel<128, false>), grid4, dim3(64 * kPartWaves), 0, st, p);
    else hipLaunchKernelGGL((extend_attention_parts_kernel<64, false>), grid4, dim3(64 * kPartWaves), 0, st, p);
    if (p.parts > 1) {
      const dim3 gridm(static_cast<unsigned>((p.part_rows * (head_dim / 8) + 255) / 256));
      if (head_dim == 128) hipLaunchKernelGGL((extend_merge_kernel<128>), gridm, dim3(256), 0, st, p);
      else hipLaunchKernelGGL((extend_merge_kernel<64>), gridm, dim3(256), 0, st, p);
    }
    SGL_CHECK_LAUNCH("extend_attention");
    return 0;
  }
  const bool fast = plain && nwv == 8 && !(kv_fp8 && (g_extend_debug_flags & 2) != 0);
  if (fast) {
    p.num_tiles = tiles; p.batch = static_cast<int>(batch);
    if (grabbed != nullptr && g_extend_debug_flags == 0 && extend_walks(num_tokens, batch, rows_total, group, num_kv_heads, head_dim)) {
      p.grabbed = grabbed;
      if (kv_fp8) hipLaunchKernelGGL((extend_attention_walk_kernel<true>), dim3(256), dim3(512), 0, st, p);
      else hipLaunchKernelGGL((extend_attention_walk_kernel<false>), dim3(256), dim3(512), 0, st, p);
      SGL_CHECK_LAUNCH("extend_attention");
      return 0;
    }
    const dim3 grid1(static_cast<unsigned>(tiles) * num_kv_heads * static_cast<unsigned>(batch));
    if ((g_extend_debug_flags & 2) != 0) {
      if (head_dim == 128) hipLaunchKernelGGL((extend_attention_dbuf_kernel<128>), grid1, dim3(512), 0, st, p);
      else hipLaunchKernelGGL((extend_attention_dbuf_kernel<64>), grid1, dim3(512), 0, st, p);
    } else if (kv_fp8) {
      if (head_dim == 128) hipLaunchKernelGGL((extend_attention_pipe_kernel<128, 8, true>), grid1, dim3(512), 0, st, p);
      else hipLaunchKernelGGL((extend_attention_pipe_kernel<64, 8, true>), grid1, dim3(512), 0, st, p);
    } else if (head_dim == 128) hipLaunchKernelGGL((extend_attention_pipe_kernel<128, 8, false>), grid1, dim3(512), 0, st, p);
    else hipLaunchKernelGGL((extend_attention_pipe_kernel<64, 8, false>), grid1, dim3(512), 0, st, p);
    SGL_CHECK_LAUNCH("extend_attention");
    return 0;
  }
#define SGL_LAUNCH_EXT(D_, M_, W_)                                                                                        \
  do {                                                                                                                    \
    if (kv_fp8) hipLaunchKernelGGL((extend_attention_kernel<D_, M_, W_, true>), grid, dim3(64 * W_), 0, st, p);           \
    else hipLaunchKernelGGL((extend_attention_kernel<D_, M_, W_, false>), grid, dim3(64 * W_), 0, st, p);                 \
  } while (0)
  if (head_dim == 128) {
    if (nwv == 8) SGL_LAUNCH_EXT(128, 2, 8);
    else if (mtw == 1) SGL_LAUNCH_EXT(128, 1, 4);
    else SGL_LAUNCH_EXT(128, 2, 4);
  } else {
    if (nwv == 8) SGL_LAUNCH_EXT(64, 2, 8);
    else if (mtw == 1) SGL_LAUNCH_EXT(64, 1, 4);
    else SGL_LAUNCH_EXT(64, 2, 4);
  }
#undef SGL_LAUNCH_EXT
  SGL_CHECK_LAUNCH("extend_attention");
  return 0;
}

int sgl_amd_extend_attention_ex(const void* q, void* out, const void* k_cache, const void* v_cache,
                                const int32_t* req_to_token, int64_t req_to_token_stride,
                                const int64_t* req_pool_indices, const int32_t* seq_lens,
                                const int32_t* prefix_lens, const int32_t* qo_indptr, int64_t batch,
                                int max_extend_len, int num_q_heads, int num_kv_heads, int head_dim,
                                int64_t q_token_stride, int64_t out_token_stride,
                                int64_t k_cache_row_stride, int64_t v_cache_row_stride, float sm_scale,
                                int causal, int kv_fp8, float k_scale, float v_scale, int page_size, int kv_layout_hnd,
                                int sliding_window, float logit_cap, const void* custom_mask, const int64_t* mask_indptr,
                                int skip_prefix_custom_mask, void* stream) {
  return extend_attention_any(q, out, k_cache, v_cache, req_to_token, req_to_token_stride, req_pool_indices, seq_lens, prefix_lens,
                              qo_indptr, batch, max_extend_len, num_q_heads, num_kv_heads, head_dim, q_token_stride, out_token_stride,
                              k_cache_row_stride, v_cache_row_stride, sm_scale, causal, kv_fp8, k_scale, v_scale, page_size, kv_layout_hnd,
                              sliding_window, logit_cap, custom_mask, mask_indptr, skip_prefix_custom_mask, 0, 0, 1, nullptr, nullptr, stream);
}

int sgl_amd_extend_attention_parts(int64_t batch, int64_t num_tokens, int max_extend_len, int max_kv_len, int num_q_heads, int num_kv_heads, int head_dim) {
  if (batch <= 0 || max_extend_len <= 0 || max_kv_len <= kKvTile || num_kv_heads <= 0 || num_q_heads % num_kv_heads != 0 ||
      (head_dim != 64 && head_dim != 128) || num_q_heads / num_kv_heads > 32 * kPartWaves || g_extend_debug_shape != 0 || g_extend_debug_flags != 0)
    return 1;
  const int group = num_q_heads / num_kv_heads;
  if (extend_eight_waves(num_tokens, batch, static_cast<int64_t>(max_extend_len) * group, group, num_kv_heads, head_dim)) return 1;
  const int tokens = 32 * kPartWaves / group;               // whole tokens a tile, as the launch deals them
  const int64_t wgs4 = static_cast<int64_t>((max_extend_len + tokens - 1) / tokens) * num_kv_heads * batch;
  return extend_parts(wgs4, batch * static_cast<int64_t>(max_extend_len) * num_q_heads, max_kv_len, head_dim);
}

int sgl_amd_extend_attention_kv(const void* q, void* out, const void* k_cache, const void* v_cache,
                                const int32_t* req_to_token, int64_t req_to_token_stride,
                                const int64_t* req_pool_indices, const int32_t* seq_lens,
                                const int32_t* prefix_lens, const int32_t* qo_indptr, int64_t batch, int64_t num_tokens,
                                int max_extend_len, int max_kv_len, int num_q_heads, int num_kv_heads, int head_dim,
                                int64_t q_token_stride, int64_t out_token_stride, int64_t cache_row_stride, float sm_scale,
                                int causal, int kv_fp8, float k_scale, float v_scale, int parts, void* ws_acc, void* ws_ml,
                                void* stream) {
  SGL_CLEAR_STALE_ERROR();
  SGL_CHECK_ARG(parts >= 1 && parts <= 64 && (parts == 1 || (ws_acc && ws_ml)), "extend_attention_kv: 1..64 parts, workspaces for more than one");
  SGL_CHECK_ARG(parts == 1 || (num_kv_heads > 0 && num_q_heads > 0 && num_tokens >= 0 && num_tokens * num_q_heads < (int64_t{1} << 31)),
                "extend_attention_kv: num_tokens=%lld", static_cast<long long>(num_tokens));
  return extend_attention_any(q, out, k_cache, v_cache, req_to_token, req_to_token_stride, req_pool_indices, seq_lens, prefix_lens,
                              qo_indptr, num_tokens == 0 ? 0 : batch, max_extend_len, num_q_heads, num_kv_heads, head_dim, q_token_stride,
                              out_token_stride, cache_row_stride, cache_row_stride, sm_scale, causal, kv_fp8, k_scale, v_scale, 1, 0, -1, 0.0f,
                              nullptr, nullptr, 0, num_tokens, max_kv_len, parts, ws_acc, ws_ml, stream);
}

int sgl_amd_extend_attention_store(const void* q, void* out, void* k_cache, void* v_cache, const int32_t* req_to_token, int64_t req_to_token_stride,
                                   const int64_t* req_pool_indices, const int32_t* seq_lens, const int32_t* prefix_lens, const int32_t* qo_indptr,
                                   int64_t batch, int64_t num_tokens, int max_extend_len, int max_kv_len, int num_q_heads, int num_kv_heads,
                                   int head_dim, int64_t q_token_stride, int64_t out_token_stride, int64_t cache_row_stride, float sm_scale, int causal,
                                   int kv_fp8, float k_scale, float v_scale, int parts, void* ws_acc, void* ws_ml, const void* k_new,
                                   const void* v_new, const int64_t* new_loc, int64_t k_new_stride, int64_t v_new_stride, void* stream) {
  SGL_CHECK_ARG(parts >= 0 && (parts > 0 || (ws_ml && max_kv_len > 0 && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0)),
                "extend_attention_store: counters for workgroups that stay");
  unsigned* grabbed = parts == 0 ? static_cast<unsigned*>(ws_ml) : nullptr;
  const int rc = store_kv_rows(k_new, v_new, k_cache, v_cache, new_loc, num_tokens, num_kv_heads, head_dim, k_new_stride, v_new_stride, cache_row_stride, kv_fp8,
                               k_scale, v_scale, grabbed, stream);
  if (rc != 0) return rc;
  if (parts > 0)
    return sgl_amd_extend_attention_kv(q, out, k_cache, v_cache, req_to_token, req_to_token_stride, req_pool_indices, seq_lens, prefix_lens, qo_indptr,
                                       batch, num_tokens, max_extend_len, max_kv_len, num_q_heads, num_kv_heads, head_dim, q_token_stride,
                                       out_token_stride, cache_row_stride, sm_scale, causal, kv_fp8, k_scale, v_scale, parts, ws_acc, ws_ml, stream);
  return extend_attention_any(q, out, k_cache, v_cache, req_to_token, req_to_token_stride, req_pool_indices, seq_lens, prefix_lens,
                              qo_indptr, num_tokens == 0 ? 0 : batch, max_extend_len, num_q_heads, num_kv_heads, head_dim, q_token_stride,
                              out_token_stride, cache_row_stride, cache_row_stride, sm_scale, causal, kv_fp8, k_scale, v_scale, 1, 0, -1, 0.0f,
                              nullptr, nullptr, 0, num_tokens, max_kv_len, 1, nullptr, nullptr, stream, grabbed);
}

int sgl_amd_extend_attention_store_parts(int64_t batch, int64_t num_tokens, int64_t sum_kv_len, int max_extend_len, int max_kv_len, int num_q_heads,
                                         int num_kv_heads, int head_dim) {
  if (batch > 0 && max_extend_len > 0 && max_kv_len > kKvTile && num_kv_heads > 0 && num_q_heads % num_kv_heads == 0 && g_extend_debug_shape == 0 &&
      g_extend_debug_flags == 0) {
    const int group = num_q_heads / num_kv_heads;
    if (extend_ragged(extend_held(num_tokens, batch, group, num_kv_heads), batch, num_tokens, sum_kv_len, max_extend_len, max_kv_len, group) &&
        extend_walks(num_tokens, batch, static_cast<int64_t>(max_extend_len) * group, group, num_kv_heads, head_dim)) return 0;
  }
  return sgl_amd_extend_attention_parts(batch, num_tokens, max_extend_len, max_kv_len, num_q_heads, num_kv_heads, head_dim);
}

#ifdef EXT_TRACE
int sgl_amd_debug_ext_trace(void* buf) {
  uint64_t* p = static_cast<uint64_t*>(buf);
  return hipMemcpyToSymbol(HIP_SYMBOL(g_ext_trace), &p, sizeof(p)) == hipSuccess ? 0 : 1;
}
#endif

int sgl_amd_probe_mfma_16x16x32(const void* a, const void* b, void* c, void* stream) {
  SGL_CLEAR_STALE_ERROR();
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, as_stream(stream),
                     static_cast<const uint16_t*>(a), static_cast<const uint16_t*>(b),
                     static_cast<float*>(c));
  SGL_CHECK_LAUNCH("probe_mfma_16x16x32");
  return 0;
}

}  // extern "C"
