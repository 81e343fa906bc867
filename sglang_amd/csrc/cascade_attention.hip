// Shared-prefix (cascade) decode attention for gfx950, one launch for the whole step + an LSE merge.
//
// Replaces (reference, /root/reference/python/sglang):
//   srt/layers/attention/triton_backend.py:136-1012 forward_decode -> kernels/ops/attention/
//   decode_attention.py:1163 decode_attention_fwd, which re-reads a radix-shared prefix once per
//   request.  Oracle: srt/layers/attention/torch_native_backend.py:176-277 (oracle/ops.py).
//
// RadixAttention batches share KV rows: requests whose req_to_token rows start with the same slots
// attend to the SAME rows of the pool.  The device plan (sgl_amd_cascade_plan) groups them; this
// kernel then works on "chunk items", each one workgroup:
//   shared item  = (group, 128-token chunk of the shared prefix, <= 64/G members): the chunk's K/V
//                  rows are read ONCE and multiplied with the decode queries of all members
//                  (members x G query heads = up to 64 rows) on the matrix cores;
//   private item = (request, 128-token chunk of its unshared suffix): the same code with one member.
// Every item is a single shot -- no KV loop: 128 slot ids -> 128 K rows + 128 V rows gathered in one
// burst (16 x 16 B loads in flight per lane), S^T = K Q^T and O^T = V^T P^T with MFMA 16x16x32 bf16,
// softmax state lane-local (transposed products).  That keeps the dependent-load chain at three
// hops (plan -> slot ids -> rows) whatever the context length; parallelism comes from the number of
// items.  Each item writes an unnormalised (acc, max, sum) partial into its slot of every member;
// the merge kernel combines the slots of a (request, head) in slot order.
#include <type_traits>

#include "common.hpp"
#include "cascade_plan.hpp"
#include "kv_format.hpp"
#include "sglang_amd.h"

using namespace sgl_amd;

namespace {

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));

constexpr int kThreads = 256;
constexpr int kChunk = 128;       // kv tokens per item
constexpr int kRowsPerItem = 64;  // (member, q head) rows per item: 4 waves x one 16-row tile
constexpr float kNegBig = -1.0e30f;
// launch-form policy of the chunk kernel (see cascade_chunk_kernel); process-wide tuning knobs behind
// sgl_amd_debug_cascade_launch_form, like the extend kernel's shape switch
constexpr int64_t kSingleShotHardCap = 16384;    // the largest value the switch below may take: what the plan clears for is decided against THIS, not the switch
constexpr int64_t kSingleShotUnits = 10240;
// ... and for requests of at most 8 query rows a kv head behind tables of at least kSpanChunks chunks, whose private tokens the plan cuts into
// spans: the looping form.  us a layer, Llama-3-8B heads, single-shot against spans, at an 8 k-token table: 8 requests of 5 k 57 / 51, 16 of
// 4 k 77 / 70, 2 of 7 k 25.0 / 24.0; 4 of 17 k at a 32 k-token table 82.8 / 64.6.  At tables of 1.2 and 2.5 k tokens, whose requests are
// short: 64 of 0.9 k 51.9 / 53.1, 64 behind a shared prefix 22.5 / 23.5, 32 of 0.3 k 15.8 / 17.9.
// Not for bf16 rows of head dim 64: four layers of 14 / 2 heads, 16 requests of 700 54 / 57 us, 64 of 400 66 / 69, 16 of 3 k 81 / 83, and above
// the line items against spans 128 of 600 88 / 94, 128 of 400 behind a shared 1 k 88 / 95.  (Of e4m3 rows 64 of 1.5 k 101 / 92.)
constexpr int64_t kSpanSingleShotUnits = 2048;
constexpr int kSpanChunks = 64;
inline int64_t single_shot_most(int chunks, bool spans) { return spans && chunks >= kSpanChunks ? kSpanSingleShotUnits : kSingleShotUnits; }
inline bool walks_spans(int group, int head_dim, bool fp8) { return group <= 8 && (head_dim > 64 || fp8); }
int64_t g_cascade_single_shot_units = 0;       // worst-case workgroups up to which the one-workgroup-per-unit form is launched (0: the rule above)
// Grid of the looping form.  Units inside it are dealt as workgroups end, those behind it before the launch.  Items of bf16 rows of head dim 128 gain by
// the first (136 batches at 1280 / 2048 / 4096 / 8192 workgroups: 5.3, 1.7, 0.6 and 0.9 % behind the best of six grids).  Beside spans, never more than
// 1024, the workgroups without a unit cost 0.3 us a layer of 58.  That is as much beside e4m3 rows (37 requests of 0.9 to 5.1 k 270 us at 1280, 273 at
// 2048, four layers), whose items are walked only where there are few, and rows of 64 elements gain nothing (128 of 1.2 k, 14 / 2 heads, 130 / 134).
constexpr int64_t kLoopGrid = 256 * 16, kLoopGridSmallRows = 256 * 5;
int64_t g_cascade_loop_grid = 0;               // 0: these

__device__ __forceinline__ bf16x8_t as_frag(const U4& v) { return __builtin_bit_cast(bf16x8_t, v); }

#ifdef CASC_TRACE
// timeline probe (benchmarks/r02_exp8_casc_trace.py): per workgroup, the chip-wide 100 MHz clock at entry, record read,
// K image staged, scores done, V image staged, partials stored
__device__ uint64_t* g_casc_trace = nullptr;
#define CASC_STAMP(i)                                                                                     \
  do {                                                                                                    \
    if (g_casc_trace && threadIdx.x == 0) g_casc_trace[static_cast<int64_t>(blockIdx.x) * 8 + (i)] = wall_clock64(); \
  } while (0)
#else
#define CASC_STAMP(i)
#endif

struct ChunkParams {
  const uint16_t* q;            // [B, Hq, D]
  const uint16_t* k_cache;      // [slots, Hkv, D]
  const uint16_t* v_cache;
  const int32_t* req_to_token;
  const int64_t* req_pool_indices;
  const int32_t* seq_lens;
  const int32_t* plan;
  float* ws_acc;                // [B, Hq, slots_total, D]
  float* ws_ml;                 // [B, Hq, slots_total, 2]
  int64_t q_stride, kc_stride, vc_stride, r2t_stride;
  KvFormat fmt;                 // pool layout (token-major or paged head-major) + element format (bf16 / e4m3 rows)
  int batch, max_items, num_q_heads, group, members_per_item;
  int num_kv_heads;
  int slots_total;
  float scale_log2;
  int walks_spans;              // the looping kernel takes the plan's spans, where it has any, in the place of the private items
};

// A pointer that came as a bare word, known to lie in device memory.  Left generic, all 650 loads of the looping kernels were flat ones: those count as LDS
// accesses too, so that every wait for the image drained the rows on their way.  us for four layers: 100 requests of 0.6 to 1.4 k, 32 / 8 heads, 433 -> 415,
// 8 of 5 k, 64 / 8 heads, 196 -> 188, 16 of 1 k, 32 kv heads, 272 -> 263, 64 of 1.5 k in e4m3 252 -> 249.
template <typename T>
__device__ __forceinline__ T* global_ptr(T* x) {
  return (T*)(__attribute__((address_space(1))) T*)(uint64_t)x;
}

// ---- The rows of the step itself (sgl_amd_cascade_decode_attention_store).  A launch of their own in front of every layer's attention is little more than launch, so
// each row is stored by the one unit of a kv head that reads it as its request's newest token: by every wave of the unit that reads it, before it does (the
// accesses of a wave to one address complete in order, and what the other waves store is the same).  Nobody else reads the slot, unless a table holds
// another row's new slot; the plan looks for that once a step (cascade_check_rows), and then every wave stores the rows that it found first (put_rows_first), the later
// of two with one slot; all rows, where the plan was not made for these slots.  The row of a request without tokens, which no unit reads, is stored by the first
// workgroup of its kv head.
// us of attention a step, store launch / this: 64 requests behind shared prefixes, 32 / 8 heads, 8 layers, 232 / 215; 37 of 0.9 to 5.1 k in e4m3, 4 layers,
// 266 / 256; 21 of 180 in e4m3, 64 / 8 heads, 4 layers, 70 / 61.  What is left of the launch: 0.8 us a layer in units of 128 tokens (with nothing stored 209).
struct NewRows {
  const uint16_t* k;            // [B, Hkv, D]
  const uint16_t* v;
  const int64_t* loc;
  int64_t k_stride, v_stride;
  float inv_k_scale, inv_v_scale;
};
struct StoreParams {
  ChunkParams chunk;
  NewRows rows;
};
constexpr int kNewest = -2, kOlder = -1;              // word 7 of a private item's or piece's record: it ends in the request's newest token, or not
enum RowsToStore { kInPool = 0, kOwnRow = 1, kMetRows = 2, kAllRows = 3 };

// a lane's piece of request b's new rows of a kv head: asked for, stored (K by the first D / 8 lanes, V by the next)
template <int D>
__device__ __forceinline__ U4 ask_new_row(const NewRows& rows, const int b, const int kvh, const int lane) {
  return ld16((lane & (D / 8) ? rows.v + b * rows.v_stride : rows.k + b * rows.k_stride) + kvh * D + (lane & (D / 8 - 1)) * 8);
}
template <int D, bool FP8>
__device__ __forceinline__ void put_new_row(const ChunkParams& p, const NewRows& rows, const U4& x, const int slot, const int kvh, const int lane) {
  const bool of_v = (lane & (D / 8)) != 0;
  unsigned char* to = const_cast<unsigned char*>(kv_row(of_v ? p.v_cache : p.k_cache, p.fmt, slot, kvh));
  if (lane < D / 4) put_kv8<FP8>(to, lane & (D / 8 - 1), x, of_v ? rows.inv_v_scale : rows.inv_k_scale);
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
}
template <int D, bool FP8>
__device__ __forceinline__ void put_own_row(const ChunkParams& p, const NewRows& rows, const int b, const int kvh, const int lane) {
  const int slot = static_cast<int>(rows.loc[b]);
  put_new_row<D, FP8>(p, rows, ask_new_row<D>(rows, b, kvh, lane), slot, kvh, lane);
}
// whether no later row of the step has request b's slot
__device__ __forceinline__ bool latest_row(const ChunkParams& p, const NewRows& rows, const int b, const int lane) {
  const int64_t slot = rows.loc[b];
  bool again = false;
#pragma clang loop unroll(disable)
  for (int c = b + 1 + lane; c < p.batch; c += 64) again |= rows.loc[c] == slot;
  return __ballot(again) == 0ull;
}
// In front of all units where others may read some rows, or the plan was made for other slots: the rows that the plan found, or all.  us a layer, a launch for
// the rows / all of them in front of every unit / these: 64 requests of 1 k 52 / 107 / 59, 1024 of 300 304 / 16058 / 370.
template <int D, bool FP8>
__device__ __forceinline__ void put_rows_first(const ChunkParams& p, const NewRows& rows, const bool all, const int first_kvh, const int end_kvh, const int lane) {
  const CascadePlanView pv = cascade_plan_view(p.plan, p.batch, p.max_items);
  const bool found = pv.meet[lane] != 0;
#pragma clang loop unroll(disable)
  for (int b0 = 0; b0 < p.batch; b0 += 32) {
    uint32_t some = found ? pv.met_rows[32 * lane + (b0 >> 5)] : 0u;
    for (int off = 32; off > 0; off >>= 1) some |= __shfl_xor(some, off, 64);
    if (all) some = b0 + 32 <= p.batch ? ~0u : (1u << (p.batch - b0)) - 1u;
#pragma clang loop unroll(disable)
    for (uint32_t todo = __builtin_amdgcn_readfirstlane(some); todo != 0u; todo &= todo - 1u) {
      const int b = b0 + __ffs(static_cast<int>(todo)) - 1;
      if (!latest_row(p, rows, b, lane)) continue;
#pragma clang loop unroll(disable)
      for (int kvh = first_kvh; kvh < end_kvh; ++kvh) put_own_row<D, FP8>(p, rows, b, kvh, lane);
    }
  }
}

// The rows of the requests without tokens (a call for the whole batch, of one workgroup a kv head, where the plan found any).  As a meeting of slots, which every wave
// answers by storing all rows, one such request among 64 of 1 k took a layer from 50 to 105 us.
template <int D, bool FP8>
__device__ __forceinline__ void put_unread_rows(const ChunkParams& p, const NewRows& rows, const int kvh, const int lane) {
#pragma clang loop unroll(disable)
  for (int b0 = 0; b0 < p.batch; b0 += 64) {
    unsigned long long todo = __ballot(b0 + lane < p.batch && p.seq_lens[b0 + lane < p.batch ? b0 + lane : 0] < 1);
#pragma clang loop unroll(disable)
    for (; todo != 0ull; todo &= todo - 1) put_own_row<D, FP8>(p, rows, b0 + __ffsll(static_cast<long long>(todo)) - 1, kvh, lane);
  }
}

// Whether rows have to be stored first: a table holds a new slot elsewhere, or the plan does not know these slots (every wave for itself).
// The first 64 requests' slots and the words are asked for by ask(), beside what else a kernel begins with: behind it they are a round trip of their own.
struct RowsMeet {
  int word, planned, now;
  __device__ __forceinline__ void ask(const ChunkParams& p, const NewRows& rows, const int lane) {
    const CascadePlanView pv = cascade_plan_view(p.plan, p.batch, p.max_items);
    const int first = lane < p.batch ? lane : p.batch - 1;
    word = pv.meet[lane];
    planned = pv.new_slots[first];
    now = static_cast<int32_t>(rows.loc[first]);
  }
  __device__ __forceinline__ int answer(const ChunkParams& p, const NewRows& rows, const int lane) const {
    bool other = (word & kPlanUntold) | (planned != now);
    if (p.batch > 64) {
      const CascadePlanView pv = cascade_plan_view(p.plan, p.batch, p.max_items);
      for (int b = 64 + lane; b < p.batch; b += 64) other |= pv.new_slots[b] != static_cast<int32_t>(rows.loc[b]);
    }
    if (__ballot(other | (word & kPlanMeet)) == 0ull) return kOwnRow;
    return __ballot(other) != 0ull ? kAllRows : kMetRows;
  }
  __device__ __forceinline__ bool unread() const { return __ballot(word & kPlanUnread) != 0ull; }
};

// The K rows, then (after S^T) the transposed V rows, pass through ONE 16 KiB LDS image; at D = 128 it is filled twice
// per operand: K by token halves (64 tokens x 128 dims: each score tile is complete inside its half), V^T by head-dim
// halves (64 dims x 128 tokens: each output tile is complete inside its half).  With <= 96 VGPRs that makes five
// workgroups per CU resident -- 1280 on the chip: the bench batch's 1248 units run as one round
// (at four per CU the last 224 started when the first finished, 7 us of a 20 us kernel, benchmarks/r02_exp8).
// Two forms of the launch.
//   cascade_chunk_kernel: one workgroup per unit; the grid covers the worst-case item count of the batch and the workgroups behind
//     the end of the device-built list leave after one load.  96 registers: five workgroups per CU.  Chosen while the worst
//     case stays below kSingleShotUnits workgroups (a request table of a few thousand tokens: the bench's 1.2 k-token table
//     asks for 9.5 k).
//   cascade_chunk_loop_kernel: a grid of kLoopGrid resident workgroups walks the list -- workgroup w takes units w, 2 G - 1 - w, 2 G + w,
//     ... (a snake over the passes: the shared items at the head of the list are the heavy ones, the workgroups that got
//     them in one pass get the far end of the next) below the list's end, which every workgroup knows after ONE scalar load
//     (header[5]) that travels with its first item record.  Where the plan has cut the private tokens into spans, a unit behind the shared
//     items is one span, piece by piece.  Chosen for large request tables: the worst case of a 64-request
//     batch is 58 k workgroups at an 8 k-token table (Llama-3-8B's own context length under the reference's scheduler), ~1 M at
//     128 k, and a workgroup behind the list's end costs ~0.25 ns of dispatch -- 20 -> 33.7 us per layer at 8 k, measured
//     under the reference's scheduler (profiles/r05_sched_step_timeline_hooks.txt).  The loop keeps the thread index and the
//     kernel arguments opaque per pass (nothing lane-derived or argument-derived is loop-invariant to the compiler: round 2's
//     persistent loop died of hoisted LDS addresses), and it is given 128 registers -- four workgroups per CU, no spills --
//     because at the 96 budget hipcc parks ~30 registers in scratch once there is a loop around the body: that instance was
//     built and measured (profiles/r05_exp1b_cascade_forms.json): 34.1 us per layer against 26.7 at four per CU and 25.6 for
//     the one-workgroup-per-unit form on the bench's own table; grids of 1280 / 2048 equal there, 1024 (= what is resident) 28.0.
template <int D, bool FP8, bool HND>
__global__ __launch_bounds__(kThreads, 5) void cascade_chunk_kernel(ChunkParams p) {
  __shared__ U4 sm[(kChunk / (D > 64 ? D / 64 : 1)) * (D / 8)];   // K: [token of the part][piece ^ swz];  V^T: [d of the part][8-token chunk ^ swz]
  __shared__ float ml_s[64];                                      // token-split units: (max, sum) of [wave][row < 8]
  __shared__ U4 side_s[D > 64 ? 4 * 8 * (D - 64) / 4 : 1];        // ... and their O^T partials of every V^T part but the last
  const int unit = blockIdx.x;
  const int tid = threadIdx.x;
  constexpr bool STORE = false;
  const NewRows new_rows{};
  RowsMeet meet;
#define CASC_ONE_SHOT
#include "cascade_chunk_body.inc"
#undef CASC_ONE_SHOT
}

// ... with the step's rows to store (token-major pools)
template <int D, bool FP8>
__global__ __launch_bounds__(kThreads, 5) void cascade_store_kernel(StoreParams sp) {
  __shared__ U4 sm[(kChunk / (D > 64 ? D / 64 : 1)) * (D / 8)];
  __shared__ float ml_s[64];
  __shared__ U4 side_s[D > 64 ? 4 * 8 * (D - 64) / 4 : 1];
  const ChunkParams& p = sp.chunk;
  const NewRows& new_rows = sp.rows;
  const int unit = blockIdx.x;
  const int tid = threadIdx.x;
  constexpr bool HND = false, STORE = true;
  RowsMeet meet;
  meet.ask(p, new_rows, tid & 63);
#define CASC_ONE_SHOT
#include "cascade_chunk_body.inc"
#undef CASC_ONE_SHOT
}

template <int D, bool FP8, bool HND, bool STORE>
__device__ __forceinline__ void cascade_chunk_unit(const ChunkParams& p, const NewRows& new_rows, U4* sm, float* ml_s, U4* side_s, const int unit, const int tid,
                                                   const int store_rows) {
#include "cascade_chunk_body.inc"
}

// max over the four 16-lane rows of a wave (inline asm: with the builtin on two copies of one value hipcc kept only the first result)
__device__ __forceinline__ float lane_rows_max(float x) {
  float a = x, b = x;
  asm volatile("s_nop 1\n\tv_permlane16_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  a = fmaxf(a, b);
  b = a;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1\n\ts_nop 1" : "+v"(a), "+v"(b));
  return fmaxf(a, b);
}

// A unit of at most 8 query rows (a piece of a span; an e4m3 item of few members) in the looping kernel: any number of tokens, wave w
// takes the 16-token tiles w, w + 4, ...  No barrier until the waves' (max, sum, O) sets meet: K rows are the matrix operand as they
// come (lane = token, four lanes a row), V rows pass through the wave's own 4 KiB image and come out transposed by
// ds_read_b64_tr_b16.  The next tile's K rows are asked for once this tile's scores are formed, its V rows once this tile's have left
// the registers, so a wave always has rows in flight; the twelve waves a CU of the spans do the rest (16 tokens, not 32: at 32 the 128 registers spill,
// 256 against 211 us for 32 requests of 2 k tokens in e4m3).
// What bounds it: the gathered rows -- four layers of 37 requests of 0.9 to 5.1 k tokens in e4m3 481 -> 268 us (2.0 -> 3.6 TB/s), 128
// requests of 1.5 k in bf16 910 -> 729 us (4.6 TB/s; a large copy reaches 4.9).  Before, a unit was 128 tokens staged through one image
// behind six barriers.  A bf16 item of 128 tokens keeps that form: its rows come in one burst, 257 against 265 us in the shared-prefix batch.
// Image: row (token) t at t * 2 D bytes, its 16-byte piece c in slot c ^ kSw(t): the four rows of a transposing read lie on distinct banks.
template <int D, bool FP8, bool HND, bool STORE>
__device__ __forceinline__ void cascade_few_rows_unit(const ChunkParams& p, const NewRows& new_rows, U4* sm, float* ml_s, const int32_t* rec, const int kvh,
                                                      const int tid, const int store_rows) {
  const int4 ra = *reinterpret_cast<const int4*>(rec), rb = *reinterpret_cast<const int4*>(rec + 4);
  constexpr int KC = D / 32, ND = D / 16;
  constexpr int KL = FP8 ? D / 64 : D / 32;                    // 16-byte pieces of a K row a lane holds
  constexpr int VL = FP8 ? D / 64 : D / 32;                    // ... of the 16 V rows
  constexpr int VPR = FP8 ? D / 16 : D / 8;                    // lanes a V row
  typedef short v4s16_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) v4s16_t* lds_v4_t;
  auto swz = [](int t) __attribute__((always_inline)) { return D == 128 ? 2 * (t & 3) : 2 * ((t >> 1) & 3); };
  const CascadePlanView pv = cascade_plan_view(p.plan, p.batch, p.max_items);
  const int lane = tid & 63, wid = tid >> 6, i16 = lane & 15, g = lane >> 4;
  const int slot = __builtin_amdgcn_readfirstlane(ra.x), kv_begin = __builtin_amdgcn_readfirstlane(ra.y), kv_n = __builtin_amdgcn_readfirstlane(ra.z);
  const int n_rows = __builtin_amdgcn_readfirstlane(ra.w) * p.group;
  const int rec_x = __builtin_amdgcn_readfirstlane(rb.x), rec_private = __builtin_amdgcn_readfirstlane(rb.y);
  const int32_t* idx_base = p.req_to_token + static_cast<int64_t>(__builtin_amdgcn_readfirstlane(rb.z)) * p.r2t_stride + kv_begin;
  const int tiles = (kv_n + 15) / 16;
  auto slot_id = [&](int t) __attribute__((always_inline)) {   // of token lane & 15 of tile t
    const int tok = 16 * t + i16;
    return idx_base[tok < kv_n ? tok : kv_n - 1];
  };
  int ids = wid < tiles ? slot_id(wid) : 0;
  // ---- this lane's query row ----
  const int mem_i = i16 / p.group, hg = i16 - mem_i * p.group;
  const bool row_ok = i16 < n_rows;
  int req = rec_x;
  if (row_ok && !rec_private) req = pv.member_rows[rec_x + mem_i];
  U4 qf[KC];
#pragma unroll
  for (int kc = 0; kc < KC; ++kc) qf[kc] = U4{0u, 0u, 0u, 0u};
  if (row_ok) {
    const uint16_t* qp = p.q + static_cast<int64_t>(req) * p.q_stride + (kvh * p.group + hg) * D;
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) qf[kc] = ld16(qp + (FP8 ? (kc >> 1) * 64 + g * 16 + (kc & 1) * 8 : kc * 32 + g * 8));
  }
  const uint32_t row_bytes = p.fmt.page_stride;
  const unsigned char* k_rows = reinterpret_cast<const unsigned char*>(p.k_cache) + static_cast<uint32_t>(kvh) * p.fmt.head_stride;
  const unsigned char* v_rows = reinterpret_cast<const unsigned char*>(p.v_cache) + static_cast<uint32_t>(kvh) * p.fmt.head_stride;
  auto row_at = [&](const unsigned char* rows, const void* pool, int id) __attribute__((always_inline)) {
    if constexpr (HND) return kv_row(pool, p.fmt, id, kvh);
    else return rows + static_cast<uint64_t>(static_cast<uint32_t>(id)) * row_bytes;
  };
  U4 kr[KL], vr[VL];
  auto load_k = [&](int id) __attribute__((always_inline)) {
    const unsigned char* row = row_at(k_rows, p.k_cache, id) + g * 16;
#pragma unroll
    for (int c = 0; c < KL; ++c) kr[c] = ld16(row + 64 * c);
  };
  auto load_v = [&](int id) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < VL; ++i) vr[i] = ld16(row_at(v_rows, p.v_cache, __shfl(id, lane / VPR + (64 / VPR) * i, 64)) + lane % VPR * 16);
  };
  f32x4_t ot[ND];
#pragma unroll
  for (int n = 0; n < ND; ++n) ot[n] = f32x4_t{0.f, 0.f, 0.f, 0.f};
  float m_run = kNegBig, l_run = 0.f;                          // l: this lane's tokens
  unsigned char* img = reinterpret_cast<unsigned char*>(sm) + wid * 4096;
  auto put_v = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < VL; ++i) {
      const int t = lane / VPR + (64 / VPR) * i, c = lane % VPR, sw = swz(t);
      if constexpr (FP8) {
        *reinterpret_cast<U4*>(img + t * (2 * D) + ((2 * c) ^ sw) * 16) = fp8x8_to_bf16x8(uint2{vr[i].x, vr[i].y});
        *reinterpret_cast<U4*>(img + t * (2 * D) + ((2 * c + 1) ^ sw) * 16) = fp8x8_to_bf16x8(uint2{vr[i].z, vr[i].w});
      } else {
        *reinterpret_cast<U4*>(img + t * (2 * D) + (c ^ sw) * 16) = vr[i];
      }
    }
  };
  const int vrow = 4 * g + (i16 >> 2), vsw = swz(vrow);
  const unsigned char* vlane = img + vrow * (2 * D) + ((i16 >> 1) & 1) * 16 + (i16 & 1) * 8;
  // The newest token is in the last tile: its wave alone reads it, and stores it behind the requests for its first tile's rows where that is another one (in front
  // of them the wait for it was 4 us of a launch of 57).
  bool mine = STORE && __builtin_amdgcn_readfirstlane(rb.w) == kNewest && wid < tiles && ((tiles - 1 - wid) & 3) == 0;
  if (mine && store_rows != kOwnRow) mine = latest_row(p, new_rows, rec_x, lane);
  U4 own;
  if (mine) {
    if (tiles - 1 == wid) put_own_row<D, FP8>(p, new_rows, rec_x, kvh, lane);
    else own = ask_new_row<D>(new_rows, rec_x, kvh, lane);
  }
  if (wid < tiles) {
    load_k(ids);
    load_v(ids);
  }
  if (mine && tiles - 1 != wid) put_new_row<D, FP8>(p, new_rows, own, static_cast<int>(new_rows.loc[rec_x]), kvh, lane);
  for (int t = wid; t < tiles; t += 4) {
    const bool more = t + 4 < tiles;                           // (wave-uniform)
    if (more) ids = slot_id(t + 4);
    // ---- S^T: lane holds row i16, tokens 4 g + r ----
    f32x4_t st = f32x4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int kc = 0; kc < KC; ++kc) {
      U4 kf;
      if constexpr (FP8) {
        const U4 w = kr[kc >> 1];
        kf = (kc & 1) ? fp8x8_to_bf16x8(uint2{w.z, w.w}) : fp8x8_to_bf16x8(uint2{w.x, w.y});
      } else {
        kf = kr[kc];
      }
      st = __builtin_amdgcn_mfma_f32_16x16x32_bf16(as_frag(kf), as_frag(qf[kc]), st, 0, 0, 0);
    }
    if (more) load_k(ids);
    // ---- running softmax ----
    float mx = kNegBig;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      st[r] = 16 * t + 4 * g + r < kv_n ? st[r] * p.scale_log2 : kNegBig;
      mx = fmaxf(mx, st[r]);
    }
    mx = lane_rows_max(mx);
    if (__ballot(mx > m_run) != 0ull) {
      const float m_new = fmaxf(m_run, mx), alpha = fast_exp2(m_run - m_new);
      m_run = m_new;
      l_run *= alpha;
#pragma unroll
      for (int n = 0; n < ND; ++n) ot[n] *= alpha;
    }
    float e[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      e[r] = st[r] > 0.5f * kNegBig ? fast_exp2(st[r] - m_run) : 0.f;
      l_run += e[r];
    }
    const v4s16_t pf = __builtin_bit_cast(v4s16_t, uint2{pack_bf2(e[0], e[1]), pack_bf2(e[2], e[3])});
    // ---- O^T += V^T P^T (the wave's own image: its LDS accesses complete in order) ----
    put_v();
    if (more) load_v(ids);
#pragma unroll
    for (int n = 0; n < ND; ++n) {
      const v4s16_t vf = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4_t)(vlane + ((2 * n) ^ vsw) * 16));
      ot[n] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(vf, pf, ot[n], 0, 0, 0);
    }
  }
  // ---- the four waves' sets meet, each in its own image as [row < 8][dim] (another wave may still read its own) ----
  l_run += __shfl_xor(l_run, 16, 64);
  l_run += __shfl_xor(l_run, 32, 64);
  if (i16 < 8) {
#pragma unroll
    for (int n = 0; n < ND; ++n) sm[wid * 256 + i16 * (D / 4) + 4 * n + g] = __builtin_bit_cast(U4, ot[n]);
    if (g == 0) { ml_s[(wid * 8 + i16) * 2] = m_run; ml_s[(wid * 8 + i16) * 2 + 1] = l_run; }
  }
  __syncthreads();
  constexpr int PER_ROW = D / 4;
  const int row = tid / PER_ROW, dq = tid - row * PER_ROW;
  if (row < n_rows) {
    float big = kNegBig;
#pragma unroll
    for (int w = 0; w < 4; ++w)
      if (ml_s[(w * 8 + row) * 2 + 1] > 0.f) big = fmaxf(big, ml_s[(w * 8 + row) * 2]);
    f32x4_t o = f32x4_t{0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
      const float lw = ml_s[(w * 8 + row) * 2 + 1], sc = lw > 0.f ? fast_exp2(ml_s[(w * 8 + row) * 2] - big) : 0.f;
      o += __builtin_bit_cast(f32x4_t, sm[w * 256 + row * PER_ROW + dq]) * sc;
      l += lw * sc;
    }
    const int mi = row / p.group;
    const int rq = rec_private ? rec_x : pv.member_rows[rec_x + mi];
    const int64_t sl = static_cast<int64_t>(rq * p.num_q_heads + kvh * p.group + (row - mi * p.group)) * p.slots_total + slot;
    *reinterpret_cast<f32x4_t*>(p.ws_acc + sl * D + dq * 4) = o;
    if (dq == 0) {
      p.ws_ml[sl * 2 + 0] = big;
      p.ws_ml[sl * 2 + 1] = l;
    }
  }
}

// The looping form's walk; ARG: the kernel's one argument, a ChunkParams or what begins with one.
template <int D, bool FP8, bool HND, typename ARG>
__device__ __forceinline__ void cascade_chunk_loop(const ChunkParams& p, const NewRows* new_rows) {
  constexpr bool STORE = std::is_same<ARG, StoreParams>::value;
  __shared__ U4 sm[(kChunk / (D > 64 ? D / 64 : 1)) * (D / 8)];
  __shared__ float ml_s[64];
  __shared__ U4 side_s[D > 64 ? 4 * 8 * (D - 64) / 4 : 1];
  RowsMeet meet;
  if constexpr (STORE) meet.ask(p, *new_rows, threadIdx.x & 63);
  // the line of the workgroup's first item record travels with the header (a grid never reaches beyond max_items x kv heads)
  const int first_rec = cascade_plan_view(p.plan, p.batch, p.max_items).items[8 * (blockIdx.x / static_cast<unsigned>(p.num_kv_heads))];
  // one hop for all of the header that the loop needs: the list's length (shared items, then private items or spans) and what the tail is.
  // (The items stand beside the spans for a launch that does not walk these.)
  const int n_items = __builtin_amdgcn_readfirstlane(p.plan[p.walks_spans ? 5 : 0]), n_shared = __builtin_amdgcn_readfirstlane(p.plan[3]);
  const bool spans = p.walks_spans && __builtin_amdgcn_readfirstlane(p.plan[4]) > 0;
  asm volatile("" ::"v"(first_rec));
  const int n_units = n_items * p.num_kv_heads;
  const int G = static_cast<int>(gridDim.x), w0 = static_cast<int>(blockIdx.x);
  int store_rows = kInPool;
  if constexpr (STORE) {
    asm volatile("" : "+v"(meet.word), "+v"(meet.planned), "+v"(meet.now));
    store_rows = __builtin_amdgcn_readfirstlane(meet.answer(p, *new_rows, threadIdx.x & 63));
    if (store_rows != kOwnRow) put_rows_first<D, FP8>(p, *new_rows, store_rows == kAllRows, 0, p.num_kv_heads, threadIdx.x & 63);
    else if (meet.unread() && w0 < p.num_kv_heads) put_unread_rows<D, FP8>(p, *new_rows, w0, threadIdx.x & 63);
  }
  // The kernel's one argument sits at the start of the kernarg segment; every pass re-reads it through an address the
  // compiler cannot see through, exactly as a fresh launch would (scalar loads, served by the scalar cache), and takes the
  // thread index as an opaque value.
  typedef const __attribute__((address_space(4))) uint64_t KernargWord;
  const uint64_t kp = (uint64_t)__builtin_amdgcn_kernarg_segment_ptr();
  int next = 0;                                                               // > 0: the next piece of a span begun before
  for (int base = 0, pass = 0; base < n_units;) {
    const int unit = base + ((pass & 1) ? G - 1 - w0 : w0);
    if (unit >= n_units) break;                                               // (workgroup-uniform; only in the last pass)
    uint64_t ka = kp;
    asm volatile("" : "+s"(ka));
    KernargWord* kw = reinterpret_cast<KernargWord*>(ka);
    static_assert(sizeof(ARG) % 8 == 0 && std::is_trivially_copyable<ARG>::value, "kernarg image copied as 8-byte words");
    struct Raw { uint64_t w[sizeof(ARG) / 8]; } raw;
#pragma unroll
    for (unsigned i = 0; i < sizeof(ARG) / 8; ++i) raw.w[i] = kw[i];
    ARG arg = __builtin_bit_cast(ARG, raw);
    NewRows nr{};
    ChunkParams pl;
    if constexpr (STORE) {
      pl = arg.chunk;
      nr = arg.rows;
      nr.k = global_ptr(nr.k);
      nr.v = global_ptr(nr.v);
      nr.loc = global_ptr(nr.loc);
    } else {
      pl = arg;
    }
    pl.q = global_ptr(pl.q);
    pl.k_cache = global_ptr(pl.k_cache);
    pl.v_cache = global_ptr(pl.v_cache);
    pl.req_to_token = global_ptr(pl.req_to_token);
    pl.plan = global_ptr(pl.plan);
    pl.ws_acc = global_ptr(pl.ws_acc);
    pl.ws_ml = global_ptr(pl.ws_ml);
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int item = unit / pl.num_kv_heads, kvh = unit - item * pl.num_kv_heads;
    const CascadePlanView pv = cascade_plan_view(pl.plan, pl.batch, pl.max_items);
    const int span = item - n_shared;
    const bool in_span = spans && span >= 0;                                  // (workgroup-uniform)
    const int32_t* rec = pv.items + 8 * item;
    if (in_span) {
      const int i = next > 0 ? next : __builtin_amdgcn_readfirstlane(pv.span_first[span]);
      rec = pv.pieces + 8 * i;
      next = i + 1 < __builtin_amdgcn_readfirstlane(pv.span_first[span + 1]) ? i + 1 : 0;
    }
    if (in_span || (FP8 && __builtin_amdgcn_readfirstlane(rec[3]) * pl.group <= 8))
      cascade_few_rows_unit<D, FP8, HND, STORE>(pl, nr, sm, ml_s, rec, kvh, tid, store_rows);
    else
      cascade_chunk_unit<D, FP8, HND, STORE>(pl, nr, sm, ml_s, side_s, unit, tid, store_rows);
    __syncthreads();                                                          // the image is reused by the next unit
    if (next == 0) { base += G; ++pass; }
  }
}

template <int D, bool FP8, bool HND>
__global__ __launch_bounds__(kThreads, 4) void cascade_chunk_loop_kernel(ChunkParams p) {
  cascade_chunk_loop<D, FP8, HND, ChunkParams>(p, nullptr);
}
template <int D, bool FP8>
__global__ __launch_bounds__(kThreads, 4) void cascade_store_loop_kernel(StoreParams p) {
  cascade_chunk_loop<D, FP8, false, StoreParams>(p.chunk, &p.rows);
}

// ---- cascade plan: group the requests of a decode batch that share a KV prefix ----------------
// One workgroup, once per decode step.  Requests that share ANY cached prefix share their first slot
// (page_size-agnostic: identical slot ids <=> the same cached tokens), so the leader of request b is the
// lowest batch index with the same first slot; the shared length with the leader is the first mismatch
// of the two req_to_token rows.  A group's shared part is the minimum over its members, rounded down
// to kv_tile; groups with < 2 members or a short shared part are dropped.  The output is ONE compact
// list of self-contained chunk items: the shared chunks of every group (x member tiles), then the
// private chunks of every request.
constexpr int kPlanThreads = 1024;
constexpr int kPlanMaxBatch = 1024;

// One wave: request b's leader (the lowest batch index with the same first slot) and the length of the prefix it shares with that leader.
__device__ __forceinline__ void compare_request(const int32_t* req_to_token, int64_t r2t_stride, const int* first_slot, const int* pool_row, const int* len_s,
                                                int b, int lane, int& l, int& common) {
  l = b;
  const int fs = first_slot[b];
  for (int c0 = 0; c0 < b; c0 += 64) {
    const int c = c0 + lane;
    const unsigned long long m = __ballot(c < b && first_slot[c] == fs);
    if (m != 0ull) { l = c0 + __ffsll(static_cast<long long>(m)) - 1; break; }
  }
  // 2048 positions per round (32 loads in flight per lane and row)
  constexpr int kCmpLoads = 32;
  common = 0;
  if (l != b) {
    const int32_t* ra = req_to_token + static_cast<int64_t>(pool_row[b]) * r2t_stride;
    const int32_t* rb = req_to_token + static_cast<int64_t>(pool_row[l]) * r2t_stride;
    int lim = len_s[b] - 1;                    // the newest token's slot is never shared
    const int ll = len_s[l] - 1;
    if (ll < lim) lim = ll;
    common = lim;
    for (int t0 = 0; t0 < lim; t0 += 64 * kCmpLoads) {
      int va[kCmpLoads], vb[kCmpLoads];
#pragma unroll
      for (int u = 0; u < kCmpLoads; ++u) {
        const int t = t0 + 64 * u + lane;
        const int tc = t < lim ? t : lim - 1;
        va[u] = ra[tc];
        vb[u] = rb[tc];
      }
      int first = 0x7fffffff;
#pragma unroll
      for (int u = kCmpLoads - 1; u >= 0; --u) {
        const int t = t0 + 64 * u + lane;
        const unsigned long long mm = __ballot(t < lim && va[u] != vb[u]);
        if (mm != 0ull) first = t0 + 64 * u + __ffsll(static_cast<long long>(mm)) - 1;
      }
      if (first != 0x7fffffff) { common = first; break; }
    }
  }
}

// First launch of the plan: every request's leader (the lowest batch index with the same first slot) and the length of
// the prefix it shares with that leader.  One WAVE per request, sixteen requests per workgroup: inside ONE workgroup the
// sixteen waves walked their requests one after the other, a memory round trip each -- 26 / 183 us at 64 / 512 requests
// (benchmarks/r03_exp7_plan_batch.py).  Results go through the plan buffer's `compare` scratch to the second launch.
__global__ __launch_bounds__(kPlanThreads) void cascade_plan_compare_kernel(
    const int32_t* __restrict__ req_to_token, int64_t r2t_stride, const int64_t* __restrict__ req_pool_indices,
    const int32_t* __restrict__ seq_lens, int batch, int32_t* __restrict__ compare) {
  __shared__ int first_slot[kPlanMaxBatch];
  __shared__ int pool_row[kPlanMaxBatch], len_s[kPlanMaxBatch];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  for (int b = tid; b < batch; b += kPlanThreads) {
    const int len = seq_lens[b];
    const int row = static_cast<int>(req_pool_indices[b]);
    pool_row[b] = row;
    len_s[b] = len;
    first_slot[b] = len > 1 ? req_to_token[static_cast<int64_t>(row) * r2t_stride] : -1 - b;   // unique when too short
  }
  __syncthreads();
  const int b = static_cast<int>(blockIdx.x) * (kPlanThreads / 64) + wid;
  if (b >= batch) return;
  int l, common;
  compare_request(req_to_token, r2t_stride, first_slot, pool_row, len_s, b, lane, l, common);
  if (lane == 0) {
    compare[b] = l;
    compare[batch + b] = common;
  }
}

// A batch of up to kPlanOneLaunch requests, one a wave, is compared by the plan's own workgroup (ONE).  us, both launches / one: 8 requests behind
// 500 and 3500 shared tokens 9.4 / 9.0 and 13.1 / 10.8, 16 11.7 / 10.6 and 15.9 / 12.7, and the gap between two launches; a second request a wave
// takes it back (24: 12.9 / 12.3 and 16.5 / 15.8, 32: 13.8 / 12.8 and 15.9 / 19.1, 64: 15.0 / 21.7 and 15.9 / 32.3).
constexpr int kPlanOneLaunch = 16;

// Whether a request's table holds the slot of a row of this step anywhere but at its own newest token, looked up by workgroups beside the plan's own (one
// launch; they take less time than it).  The new slots are bits of two hashes in LDS; what both hold is compared with every slot.  Slot 0 is the sink of padded
// entries, which may share it.  Requests without tokens, whose row no unit would store, are found by the way.
__device__ __forceinline__ void cascade_check_rows(const int32_t* req_to_token, int64_t r2t_stride, const int64_t* req_pool_indices, const int32_t* seq_lens,
                                                   const int64_t* new_loc, int batch, int checker, int checkers, uint32_t* bits0, uint32_t* bits1, int* slots,
                                                   uint32_t* met, const CascadePlanView& pv) {
  const int tid = threadIdx.x;
  if (tid < kPlanMaxBatch / 32) met[tid] = 0u;
  for (int i = tid; i < 1024; i += kPlanThreads) bits0[i] = bits1[i] = 0u;
  __syncthreads();
  auto hash = [](uint32_t s) { return (s * 0x9e3779b1u) >> 17; };
  bool meet = false, unread = false, seen[kPlanMaxBatch / kPlanThreads];
#pragma unroll
  for (int i = 0; i < kPlanMaxBatch / kPlanThreads; ++i) {
    const int b = tid + i * kPlanThreads;
    seen[i] = false;
    if (b < batch) {
      const uint32_t s = static_cast<uint32_t>(new_loc[b]), h = hash(s);
      slots[b] = static_cast<int>(s);
      seen[i] = (atomicOr(&bits0[(s & 32767u) >> 5], 1u << (s & 31u)) >> (s & 31u)) & 1u;
      atomicOr(&bits1[h >> 5], 1u << (h & 31u));
      if (checker == 0) pv.new_slots[b] = static_cast<int>(s);
    }
  }
  __syncthreads();
  auto mark = [&](int b) { atomicOr(&met[b >> 5], 1u << (b & 31)); };
  auto mark_rows_of = [&](int s, int but) {
    bool found = false;
    for (int c = 0; c < batch; ++c)
      if (slots[c] == s && c != but) {
        mark(c);
        found = true;
      }
    return found;
  };
#pragma unroll
  for (int i = 0; i < kPlanMaxBatch / kPlanThreads; ++i) {
    const int b = tid + i * kPlanThreads;
    if (checker == 0 && seen[i] && slots[b] != 0 && mark_rows_of(slots[b], b)) {
      mark(b);
      meet = true;
    }
  }
  constexpr int kAhead = 8;
  for (int b = checker; b < batch; b += checkers) {
    const int32_t* row = req_to_token + req_pool_indices[b] * r2t_stride;
    const int len = seq_lens[b], own = slots[b];
    if (len < 1 && tid == 0) {
      mark(b);
      unread = true;
    }
    for (int t0 = tid; t0 < len; t0 += kAhead * kPlanThreads) {
      int s[kAhead];
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const int t = t0 + u * kPlanThreads;
        s[u] = row[t < len ? t : len - 1];
      }
#pragma unroll
      for (int u = 0; u < kAhead; ++u) {
        const uint32_t x = static_cast<uint32_t>(s[u]), h = hash(x);
        if ((bits0[(x & 32767u) >> 5] >> (x & 31u)) & (bits1[h >> 5] >> (h & 31u)) & 1u) {
          const bool newest = t0 + u * kPlanThreads >= len - 1;                  // (or behind it: that token again)
          if (!(newest && s[u] == own) && mark_rows_of(s[u], -1)) meet = true;
        }
      }
    }
  }
  const int found = (__syncthreads_or(meet) ? kPlanMeet : 0) | (__syncthreads_or(unread) ? kPlanUnread : 0);
  if (tid == 0) pv.meet[checker] = found;
  if (found != 0 && tid < kPlanMaxBatch / 32) pv.met_rows[kPlanMaxBatch / 32 * checker + tid] = static_cast<int>(met[tid]);
}

template <bool ONE>
__global__ __launch_bounds__(kPlanThreads) void cascade_plan_kernel(
    const int32_t* __restrict__ req_to_token, int64_t r2t_stride, const int64_t* __restrict__ req_pool_indices,
    const int32_t* __restrict__ seq_lens, const int64_t* __restrict__ new_loc, int batch, int min_shared, int chunk_tokens, int tokens_per_tile,
    int kv_tile, int max_shared, int32_t* __restrict__ plan, int max_items, int zero_items, int num_kv_heads, int span_units) {
  __shared__ int first_slot[kPlanMaxBatch];
  __shared__ int leader[kPlanMaxBatch];
  __shared__ int grp_min[kPlanMaxBatch];
  __shared__ int grp_cnt[kPlanMaxBatch];
  __shared__ int grp_id[kPlanMaxBatch];
  __shared__ __align__(16) int scan[kPlanMaxBatch];
  __shared__ int order[kPlanMaxBatch];
  __shared__ int g_leader[kPlanMaxBatch / 2], g_kv[kPlanMaxBatch / 2], g_first[kPlanMaxBatch / 2], g_tiles[kPlanMaxBatch / 2],
      g_rows0[kPlanMaxBatch / 2], g_members[kPlanMaxBatch / 2];
  __shared__ int n_shared_items, n_groups, n_rows;
  __shared__ int pool_row[kPlanMaxBatch], len_s[kPlanMaxBatch];   // read once: every later phase would pay the hop again
  __shared__ int wave_tot[kPlanThreads / 64], wave_tiles[kPlanThreads / 64];
  const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
  const CascadePlanView pv = cascade_plan_view(plan, batch, max_items);
  if (blockIdx.x > 0) {
    static_assert(kPlanMaxBatch == 1024, "the arrays hold 32768 bits");
    cascade_check_rows(req_to_token, r2t_stride, req_pool_indices, seq_lens, new_loc, batch, static_cast<int>(blockIdx.x) - 1, static_cast<int>(gridDim.x) - 1,
                       reinterpret_cast<uint32_t*>(first_slot), reinterpret_cast<uint32_t*>(leader), grp_min, reinterpret_cast<uint32_t*>(grp_cnt), pv);
    return;
  }
  // members == 0 marks the end of the list for the one-workgroup-per-unit chunk kernel, whose grid never reaches beyond
  // zero_items entries (the looping form reads the list's length from the header): 13.8 -> 98 us per step at a 128 k-token
  // request table when all max_items entries were cleared (profiles/r05_exp1_cascade_table_width.json)
  for (int i = tid; i < zero_items; i += kPlanThreads) pv.items[8 * i + 3] = 0;
  for (int b = tid; b < batch; b += kPlanThreads) {
    const int row = static_cast<int>(req_pool_indices[b]), len = seq_lens[b];
    pool_row[b] = row;
    len_s[b] = len;
    if constexpr (ONE) {
      first_slot[b] = len > 1 ? req_to_token[static_cast<int64_t>(row) * r2t_stride] : -1 - b;
    } else {
      leader[b] = pv.compare[b];                       // first launch: leader and common prefix of every request
      scan[b] = pv.compare[batch + b];
    }
    grp_min[b] = 0x7fffffff;
    grp_cnt[b] = 0;
  }
  __syncthreads();
  if constexpr (ONE) {
    for (int b = wid; b < batch; b += kPlanThreads / 64) {
      int l, common;
      compare_request(req_to_token, r2t_stride, first_slot, pool_row, len_s, b, lane, l, common);
      if (lane == 0) { leader[b] = l; scan[b] = common; }
    }
    __syncthreads();
  }
  for (int b = tid; b < batch; b += kPlanThreads) {
    const int l = leader[b];
    if (l != b) {
      atomicMin(&grp_min[l], scan[b]);
      atomicAdd(&grp_cnt[l], 1);
    }
  }
  __syncthreads();
  // ---- grouping decisions.  (One thread walking the batch through LDS took ~0.3 us per request -- every step of it a
  // dependent LDS round trip: 25 us of a 39 us kernel at 64 requests.)  Three parallel passes instead:
  // (1) every request works out whether it LEADS a candidate group and what the group would cost;
  for (int b = tid; b < batch; b += kPlanThreads) {
    grp_id[b] = -1;
    int cost = 0;
    if (leader[b] == b && grp_cnt[b] >= 1) {
      int kv = grp_min[b] / kv_tile * kv_tile;
      if (kv > max_shared) kv = max_shared;
      if (kv >= min_shared) {
        const int members = grp_cnt[b] + 1;
        const int tiles = (members + tokens_per_tile - 1) / tokens_per_tile;
        const int chunks = (kv + chunk_tokens - 1) / chunk_tokens;
        cost = tiles * chunks;
        scan[b] = kv;                                  // parked for pass (2): kv, tiles (members = grp_cnt + 1)
        order[b] = tiles;
      }
    }
    first_slot[b] = cost;                              // first_slot is dead after the leader search: reused as "cost"
  }
  __syncthreads();
  // (2) wave 0 accepts the candidates in batch order -- the running item count decides (plan full: the rest stay
  // ungrouped), so this is sequential, but over wave-uniform scalars read with readlane, not over LDS;
  if (wid == 0) {
    int ng = 0, rows = 0, n_items = 0;
    for (int base = 0; base < batch; base += 64) {
      const int bb = base + lane;
      const int cost = bb < batch ? first_slot[bb] : 0;
      const int members = bb < batch ? grp_cnt[bb] + 1 : 0;
      unsigned long long todo = __ballot(cost > 0);
      int my_gid = -1, my_first = 0, my_rows0 = 0;
      while (todo != 0ull) {
        const int j = __ffsll(static_cast<long long>(todo)) - 1;
        todo &= todo - 1;
        const int cj = __builtin_amdgcn_readlane(cost, j);
        const int mj = __builtin_amdgcn_readlane(members, j);
        // plan full (leave room for the private chunks of every request): the rest stay ungrouped
        if (n_items + cj > max_items / 2) continue;
        if (lane == j) { my_gid = ng; my_first = n_items; my_rows0 = rows; }
        n_items += cj;
        rows += mj;
        ++ng;
      }
      if (my_gid >= 0) {
        grp_id[bb] = my_gid;
        g_leader[my_gid] = bb; g_kv[my_gid] = scan[bb]; g_first[my_gid] = my_first; g_tiles[my_gid] = order[bb];
        g_rows0[my_gid] = my_rows0; g_members[my_gid] = members;
      }
    }
    if (lane == 0) { n_groups = ng; n_rows = rows; n_shared_items = n_items; }
  }
  __syncthreads();
  // (3) members in batch order inside each group, then the ungrouped requests: a request's place is the number of
  // earlier requests of its kind.  (The kinds go through `scan`, dead since pass (2), so that the count is a row of independent
  // 16-byte reads: two dependent LDS hops a request were 3 of the kernel's 9 us at 64 requests.)
  for (int b = tid; b < batch; b += kPlanThreads) scan[b] = grp_id[leader[b]];
  __syncthreads();
  for (int b = tid; b < batch; b += kPlanThreads) {
    const int gi = scan[b];
    int rank = 0;                                      // gi < 0: all ungrouped count together
#pragma unroll 4
    for (int c = 0; c < b; c += 4) {
      const int4 v = *reinterpret_cast<const int4*>(scan + c);
      rank += (v.x == gi ? 1 : 0) + (c + 1 < b && v.y == gi ? 1 : 0) + (c + 2 < b && v.z == gi ? 1 : 0) + (c + 3 < b && v.w == gi ? 1 : 0);
    }
    order[gi >= 0 ? g_rows0[gi] + rank : n_rows + rank] = b;   // (`order` was scratch of passes (1) and (2) until the barrier)
  }
  __syncthreads();
  // ---- write-out, all threads ----
  const int ng = n_groups, rows = n_rows;
  for (int b = tid; b < batch; b += kPlanThreads) {
    const int gi = grp_id[leader[b]];
    pv.req_shared[b] = gi >= 0 ? g_kv[gi] : 0;
    pv.batch_order[b] = order[b];
    if (b < rows) pv.member_rows[b] = order[b];
  }
  for (int gi = tid; gi < ng; gi += kPlanThreads) {
    pv.group_pool_row[gi] = pool_row[g_leader[gi]];
    pv.group_kvlen[gi] = g_kv[gi];
    pv.group_qo[gi + 1] = g_rows0[gi] + g_members[gi];
  }
  for (int i = tid; i < n_shared_items; i += kPlanThreads) {
    int gi = 0;
    while (gi + 1 < ng && g_first[gi + 1] <= i) ++gi;
    const int rel = i - g_first[gi];
    const int c = rel / g_tiles[gi], t = rel - c * g_tiles[gi];
    const int left = g_members[gi] - t * tokens_per_tile;
    const int kvn = g_kv[gi] - c * chunk_tokens;
    int32_t* it = pv.items + 8 * i;
    it[0] = c;                                         // partial slot
    it[1] = c * chunk_tokens;                          // first kv token
    it[2] = kvn < chunk_tokens ? kvn : chunk_tokens;   // kv tokens
    it[3] = left < tokens_per_tile ? left : tokens_per_tile;   // members
    it[4] = g_rows0[gi] + t * tokens_per_tile;         // first entry of member_rows
    it[5] = 0;                                         // shared item
    it[6] = pool_row[g_leader[gi]];
    it[7] = gi;
  }
  if (tid == 0) {
    pv.group_qo[0] = 0;
    pv.header[1] = ng;
    pv.header[2] = rows;
    pv.header[3] = n_shared_items;
  }
  // (no word of a workgroup that looked)
  if (tid < kCheckers && tid >= static_cast<int>(gridDim.x) - 1) pv.meet[tid] = gridDim.x == 1 ? kPlanUntold : 0;
  // ---- private chunks of every request, appended behind the shared items (block-wide exclusive scan) ----
  int mine = 0, sh = 0, len = 0;
  if (tid < batch) {
    const int gi = grp_id[leader[tid]];
    sh = gi >= 0 ? g_kv[gi] : 0;
    len = len_s[tid];
    mine = len > sh ? (len - sh + chunk_tokens - 1) / chunk_tokens : 0;
  }
  const int my_tiles = len > sh ? (len - sh + 63) / 64 : 0;
  // inclusive scans of both: inside the wave by shuffles, across the 16 waves through LDS (one barrier, not twenty)
  int incl = mine, incl_t = my_tiles;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(incl, off, 64), u = __shfl_up(incl_t, off, 64);
    if (lane >= off) { incl += v; incl_t += u; }
  }
  if (lane == 63) { wave_tot[wid] = incl; wave_tiles[wid] = incl_t; }
  __syncthreads();
  int n_private = 0, n_tiles = 0;
#pragma unroll
  for (int w = 0; w < kPlanThreads / 64; ++w) {
    const int v = wave_tot[w], u = wave_tiles[w];
    n_private += v;
    n_tiles += u;
    if (w < wid) { incl += v; incl_t += u; }
  }
  const int base = n_shared_items + incl - mine;
  const int first_slot_p = (sh + chunk_tokens - 1) / chunk_tokens;
  for (int j = 0; j < mine; ++j) {
    if (base + j >= max_items) break;                // cannot happen when max_items is sized by the caller
    int32_t* it = pv.items + 8 * (base + j);
    const int kvb = sh + j * chunk_tokens;
    it[0] = first_slot_p + j;
    it[1] = kvb;
    it[2] = len - kvb < chunk_tokens ? len - kvb : chunk_tokens;
    it[4] = tid;                                     // the request itself
    it[5] = 1;                                       // private item
    it[6] = pool_row[tid];
    it[7] = kvb + chunk_tokens < len ? kOlder : kNewest;
    it[3] = 1;
  }
  // ---- spans: the private tokens of all requests, in 64-token tiles, as ONE line cut into equal parts ----
  // (runs of whole chunks of one request each, as many as fill the chip, left it half empty at their ends: 128 requests of 0.9 to 2.1 k tokens
  // 813 to 929 us against 709)
  const int total = n_shared_items + n_private;
  int want = span_units / num_kv_heads - n_shared_items;   // the shared items hold workgroups too
  if (want < 1) want = 1;
  const int span = span_units > 0 ? (n_tiles + want - 1) / want : 0;     // tiles of a span
  const bool spans = span >= kMinSpanTiles && static_cast<int64_t>(total) * num_kv_heads > kOneRoundUnits &&     // (uniform)
                     2 * static_cast<int64_t>(n_shared_items) * num_kv_heads <= span_units;
  if (tid == 0) {
    pv.header[0] = total < max_items ? total : max_items;
    pv.header[4] = spans ? span : 0;
    pv.header[5] = spans ? n_shared_items + (n_tiles + span - 1) / span : total < max_items ? total : max_items;
  }
  if (!spans) {
    if (tid < batch) pv.req_slots[tid] = first_slot_p + mine;
    return;
  }
  const int tile0 = incl_t - my_tiles;                 // this request's tiles are [tile0, incl_t) of the line
  const int first_span = tile0 / span, my_pieces = my_tiles > 0 ? (incl_t - 1) / span - first_span + 1 : 0;
  if (tid < batch) pv.req_slots[tid] = first_slot_p + my_pieces;
  incl = my_pieces;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int v = __shfl_up(incl, off, 64);
    if (lane >= off) incl += v;
  }
  __syncthreads();                                     // (wave_tot has been read by everybody)
  if (lane == 63) wave_tot[wid] = incl;
  __syncthreads();
  for (int w = 0; w < wid; ++w) incl += wave_tot[w];
  for (int j = 0; j < my_pieces; ++j) {                // at most one a span and one more a request
    const int k = first_span + j, i = incl - my_pieces + j;
    const int lo = k * span > tile0 ? k * span - tile0 : 0, hi = (k + 1) * span - tile0;     // tiles of the request
    if (k * span >= tile0) pv.span_first[k] = i;
    int32_t* it = pv.pieces + 8 * i;
    const int kvb = sh + lo * 64, kve = sh + hi * 64;
    it[0] = first_slot_p + j;
    it[1] = kvb;
    it[2] = (kve < len ? kve : len) - kvb;
    it[3] = 1;
    it[4] = tid;
    it[5] = 1;
    it[6] = pool_row[tid];
    it[7] = kve < len ? kOlder : kNewest;
  }
  if (tid == kPlanThreads - 1) pv.span_first[(n_tiles + span - 1) / span] = incl;
}

// ---- merge: slots [0, n_slots(b)) of every (request, head), in slot order ----------------------
// n_slots = shared chunks + private chunks (pieces, where the launch before walked spans) of the request; every one was written this step.
// Block = 256 / (D/4) heads x (D/4) lanes; a thread owns 4 consecutive output elements of one head.
constexpr int kMergeBlock = 16;  // slots loaded per round (all loads of a round are in flight together)

__global__ __launch_bounds__(256) void cascade_merge2_kernel(const float* __restrict__ ws_acc, const float* __restrict__ ws_ml,
                                                             const int32_t* __restrict__ plan, const int32_t* __restrict__ seq_lens, int walks_spans,
                                                             uint16_t* __restrict__ out, int64_t out_stride, int batch,
                                                             int max_items, int num_q_heads, int head_dim, int slots_total,
                                                             float out_scale) {
  const int tpd = head_dim >> 2;
  const int b = blockIdx.x;
  const int hq = blockIdx.y * (256 / tpd) + threadIdx.x / tpd;
  const int d = (threadIdx.x % tpd) * 4;
  if (hq >= num_q_heads) return;
  const CascadePlanView pv = cascade_plan_view(plan, batch, max_items);
  // (everything the partials' addresses follow from is asked for at once: one hop after another cost 0.3 us)
  const int span_slots = pv.req_slots[b], sh = pv.req_shared[b], len = seq_lens[b];
  int n = walks_spans ? span_slots : (sh + kChunk - 1) / kChunk + (len > sh ? (len - sh + kChunk - 1) / kChunk : 0);
  if (n > slots_total) n = slots_total;
  const int64_t base = (static_cast<int64_t>(b) * num_q_heads + hq) * slots_total;
  const float2* ml = reinterpret_cast<const float2*>(ws_ml) + base;
  const float* accp = ws_acc + base * head_dim + d;
  float m_run = kNegBig, l = 0.f;
  float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int s0 = 0; s0 < n; s0 += kMergeBlock) {
    float2 mlv[kMergeBlock];
    float4 av[kMergeBlock];
#pragma unroll
    for (int i = 0; i < kMergeBlock; ++i) {
      const int s = s0 + i < n ? s0 + i : n - 1;
      mlv[i] = ml[s];
      av[i] = *reinterpret_cast<const float4*>(accp + static_cast<int64_t>(s) * head_dim);
    }
    float m_new = m_run;
#pragma unroll
    for (int i = 0; i < kMergeBlock; ++i)
      if (s0 + i < n && mlv[i].y > 0.f) m_new = fmaxf(m_new, mlv[i].x);
    const float alpha = exp2f(m_run - m_new);
    l *= alpha; o.x *= alpha; o.y *= alpha; o.z *= alpha; o.w *= alpha;
    m_run = m_new;
#pragma unroll
    for (int i = 0; i < kMergeBlock; ++i) {
      if (s0 + i < n && mlv[i].y > 0.f) {
        const float sc = exp2f(mlv[i].x - m_run);
        l += mlv[i].y * sc;
        o.x += av[i].x * sc; o.y += av[i].y * sc; o.z += av[i].z * sc; o.w += av[i].w * sc;
      }
    }
  }
  const float inv = (l > 0.f) ? out_scale / l : 0.f;       // out_scale: v_scale of an fp8 pool, else 1
  uint2 w;
  w.x = pack_bf2(o.x * inv, o.y * inv);
  w.y = pack_bf2(o.z * inv, o.w * inv);
  *reinterpret_cast<uint2*>(out + static_cast<int64_t>(b) * out_stride + static_cast<int64_t>(hq) * head_dim + d) = w;
}

}  // namespace

extern "C" {

#ifdef CASC_TRACE
int sgl_amd_debug_casc_trace(void* buf) {
  uint64_t* p = static_cast<uint64_t*>(buf);
  return hipMemcpyToSymbol(HIP_SYMBOL(g_casc_trace), &p, sizeof(p)) == hipSuccess ? 0 : 1;
}
#endif

int sgl_amd_cascade_chunk_tokens(void) { return kChunk; }

int64_t sgl_amd_cascade_plan_ints(int64_t batch, int64_t max_items) { return cascade_plan_ints(batch, max_items); }

int sgl_amd_cascade_plan(const int32_t* req_to_token, int64_t req_to_token_stride, const int64_t* req_pool_indices,
                         const int32_t* seq_lens, int64_t batch, int num_q_heads, int num_kv_heads,
                         int min_shared_len, int64_t max_context_len, int32_t* plan, int64_t max_items, void* stream) {
  return sgl_amd_cascade_plan_new_rows(req_to_token, req_to_token_stride, req_pool_indices, seq_lens, nullptr, batch, num_q_heads, num_kv_heads, min_shared_len,
                                       max_context_len, plan, max_items, stream);
}

int sgl_amd_cascade_plan_new_rows(const int32_t* req_to_token, int64_t req_to_token_stride, const int64_t* req_pool_indices,
                                  const int32_t* seq_lens, const int64_t* new_loc, int64_t batch, int num_q_heads, int num_kv_heads,
                                  int min_shared_len, int64_t max_context_len, int32_t* plan, int64_t max_items, void* stream) {
  SGL_CLEAR_STALE_ERROR();
  SGL_CHECK_ARG(batch >= 1 && batch <= kPlanMaxBatch, "cascade_plan: batch=%lld (supported: 1..%d)", (long long)batch, kPlanMaxBatch);
  SGL_CHECK_ARG(num_kv_heads > 0 && num_q_heads % num_kv_heads == 0 && num_q_heads / num_kv_heads <= kRowsPerItem, "cascade_plan: bad head counts");
  SGL_CHECK_ARG(max_items >= 1 && plan && max_context_len >= 1, "cascade_plan: bad plan arguments");
  const int members_per_item = kRowsPerItem / (num_q_heads / num_kv_heads);
  const int chunks = static_cast<int>((max_context_len + kChunk - 1) / kChunk);
  // every request's private chunks must fit behind the shared items (which may use max_items / 2): a list that
  // silently dropped a chunk would drop its tokens from the attention
  SGL_CHECK_ARG(max_items >= 2 * batch * (chunks + 1),
                "cascade_plan: max_items=%lld too small for batch=%lld x %d chunks (need >= %lld)", (long long)max_items,
                (long long)batch, chunks + 1, (long long)(2 * batch * (chunks + 1)));
  const CascadePlanView pv = cascade_plan_view(plan, batch, max_items);
  const bool one = batch <= kPlanOneLaunch;
  if (!one)
    hipLaunchKernelGGL(cascade_plan_compare_kernel, dim3(static_cast<unsigned>((batch + kPlanThreads / 64 - 1) / (kPlanThreads / 64))),
                       dim3(kPlanThreads), 0, as_stream(stream), req_to_token, req_to_token_stride, req_pool_indices, seq_lens,
                       static_cast<int>(batch), pv.compare);
  const unsigned checkers = new_loc == nullptr ? 0 : static_cast<unsigned>(batch < kCheckers ? batch : kCheckers);
  hipLaunchKernelGGL(one ? cascade_plan_kernel<true> : cascade_plan_kernel<false>, dim3(1 + checkers), dim3(kPlanThreads), 0, as_stream(stream), req_to_token,
                     req_to_token_stride, req_pool_indices, seq_lens, new_loc, static_cast<int>(batch), min_shared_len,
                     kChunk, members_per_item, 64, chunks * kChunk, plan, static_cast<int>(max_items),
                     // end-of-list markers for every item a one-workgroup-per-unit launch of THIS batch can reach (the attention entry's
                     // own bound, batch x (chunks + 1)) whenever such a launch is possible at ANY setting of the launch-form switch --
                     // the switch may change between the plan and the attention launches, or after graphs were captured
                     static_cast<int>(batch * (chunks + 1) * num_kv_heads <= kSingleShotHardCap
                                          ? (batch * (chunks + 1) < max_items ? batch * (chunks + 1) : max_items) : 0),
                     num_kv_heads,
                     num_q_heads / num_kv_heads <= 8 && batch * (chunks + 1) * num_kv_heads > single_shot_most(chunks, true) ? kSpanUnits : 0);
  SGL_CHECK_LAUNCH("cascade_plan");
  return 0;
}

int sgl_amd_cascade_members_per_item(int num_q_heads, int num_kv_heads) {
  const int group = num_q_heads / (num_kv_heads > 0 ? num_kv_heads : 1);
  return group > 0 && group <= kRowsPerItem ? kRowsPerItem / group : 0;
}

int sgl_amd_cascade_decode_attention(const void* q, const void* k_cache, const void* v_cache, void* out,
                                     const int32_t* req_to_token, int64_t req_to_token_stride,
                                     const int64_t* req_pool_indices, const int32_t* seq_lens, const int32_t* plan,
                                     int64_t batch, int64_t max_items, int num_q_heads, int num_kv_heads, int head_dim,
                                     int64_t q_token_stride, int64_t out_token_stride, int64_t k_cache_row_stride,
                                     int64_t v_cache_row_stride, float sm_scale, int64_t max_context_len,
                                     int slots_total, void* ws_acc, void* ws_ml, void* stream) {
  return sgl_amd_cascade_decode_attention_ex(q, k_cache, v_cache, out, req_to_token, req_to_token_stride, req_pool_indices,
                                             seq_lens, plan, batch, max_items, num_q_heads, num_kv_heads, head_dim,
                                             q_token_stride, out_token_stride, k_cache_row_stride, v_cache_row_stride, sm_scale,
                                             max_context_len, slots_total, ws_acc, ws_ml, 0, 1.0f, 1.0f, 1, 0, stream);
}

int sgl_amd_cascade_decode_attention_ex(const void* q, const void* k_cache, const void* v_cache, void* out,
                                        const int32_t* req_to_token, int64_t req_to_token_stride,
                                        const int64_t* req_pool_indices, const int32_t* seq_lens, const int32_t* plan,
                                        int64_t batch, int64_t max_items, int num_q_heads, int num_kv_heads, int head_dim,
                                        int64_t q_token_stride, int64_t out_token_stride, int64_t k_cache_row_stride,
                                        int64_t v_cache_row_stride, float sm_scale, int64_t max_context_len,
                                        int slots_total, void* ws_acc, void* ws_ml, int kv_fp8, float k_scale, float v_scale,
                                        int page_size, int kv_layout_hnd, void* stream) {
  return sgl_amd_cascade_decode_attention_store(q, const_cast<void*>(k_cache), const_cast<void*>(v_cache), out, req_to_token, req_to_token_stride, req_pool_indices,
                                                seq_lens, plan, batch, max_items, num_q_heads, num_kv_heads, head_dim, q_token_stride, out_token_stride,
                                                k_cache_row_stride, v_cache_row_stride, sm_scale, max_context_len, slots_total, ws_acc, ws_ml, kv_fp8, k_scale,
                                                v_scale, page_size, kv_layout_hnd, nullptr, nullptr, nullptr, 0, 0, stream);
}

int sgl_amd_cascade_decode_attention_store(const void* q, void* k_cache, void* v_cache, void* out, const int32_t* req_to_token, int64_t req_to_token_stride,
                                           const int64_t* req_pool_indices, const int32_t* seq_lens, const int32_t* plan, int64_t batch, int64_t max_items,
                                           int num_q_heads, int num_kv_heads, int head_dim, int64_t q_token_stride, int64_t out_token_stride,
                                           int64_t k_cache_row_stride, int64_t v_cache_row_stride, float sm_scale, int64_t max_context_len, int slots_total,
                                           void* ws_acc, void* ws_ml, int kv_fp8, float k_scale, float v_scale, int page_size, int kv_layout_hnd,
                                           const void* k_new, const void* v_new, const int64_t* new_loc, int64_t k_new_stride, int64_t v_new_stride, void* stream) {
  SGL_CLEAR_STALE_ERROR();
  SGL_CHECK_ARG((k_new == nullptr) == (v_new == nullptr) && (k_new == nullptr) == (new_loc == nullptr), "cascade_decode_attention: new rows without a part");
  SGL_CHECK_ARG(((reinterpret_cast<uintptr_t>(k_new) | reinterpret_cast<uintptr_t>(v_new)) & 15) == 0 && k_new_stride % 8 == 0 && v_new_stride % 8 == 0,
                "cascade_decode_attention: new rows must be 16-byte aligned");
  SGL_CHECK_ARG(head_dim == 64 || head_dim == 128, "cascade_decode_attention: head_dim=%d not supported (64/128)", head_dim);
  SGL_CHECK_ARG(num_kv_heads > 0 && num_q_heads % num_kv_heads == 0 && num_q_heads / num_kv_heads <= kRowsPerItem,
                "cascade_decode_attention: bad head counts (%d / %d)", num_q_heads, num_kv_heads);
  SGL_CHECK_ARG(q_token_stride % 8 == 0 && k_cache_row_stride % 8 == 0 && v_cache_row_stride % 8 == 0 && out_token_stride % 4 == 0,
                "cascade_decode_attention: strides must keep 16-byte (q, k, v) / 8-byte (out) alignment");
  SGL_CHECK_ARG(k_cache_row_stride > 0 && k_cache_row_stride == v_cache_row_stride,
                "cascade_decode_attention: K and V pools must share a positive row stride");
  SGL_CHECK_ARG(!kv_fp8 || (k_scale > 0.f && v_scale > 0.f), "cascade_decode_attention: fp8 KV needs positive k_scale / v_scale");
  SGL_CHECK_ARG(batch >= 1 && batch <= 1024 && max_items >= 1 && plan && ws_acc && ws_ml, "cascade_decode_attention: bad batch / workspace");
  const int chunks = static_cast<int>((max_context_len + kChunk - 1) / kChunk);
  SGL_CHECK_ARG(slots_total >= chunks + 1, "cascade_decode_attention: slots_total=%d < %d (context chunks + 1)", slots_total, chunks + 1);
  hipStream_t st = as_stream(stream);
  ChunkParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.k_cache = static_cast<const uint16_t*>(k_cache);
  p.v_cache = static_cast<const uint16_t*>(v_cache);
  p.req_to_token = req_to_token; p.req_pool_indices = req_pool_indices; p.seq_lens = seq_lens; p.plan = plan;
  p.ws_acc = static_cast<float*>(ws_acc); p.ws_ml = static_cast<float*>(ws_ml);
  p.q_stride = q_token_stride; p.kc_stride = k_cache_row_stride; p.vc_stride = v_cache_row_stride; p.r2t_stride = req_to_token_stride;
  p.batch = static_cast<int>(batch); p.max_items = static_cast<int>(max_items); p.num_q_heads = num_q_heads;
  p.group = num_q_heads / num_kv_heads; p.members_per_item = kRowsPerItem / p.group;
  p.num_kv_heads = num_kv_heads;
  p.slots_total = slots_total;
  p.scale_log2 = sm_scale * 1.4426950408889634f * (kv_fp8 ? k_scale : 1.0f);
  SGL_CHECK_ARG(make_kv_format(&p.fmt, k_cache_row_stride, num_kv_heads, head_dim, page_size, kv_layout_hnd, kv_fp8),
                "cascade_decode_attention: HND pools need a power-of-two page_size (got %d); row / page strides below 4 GiB", page_size);
  // worst-case item count of this batch.  A request of len tokens whose first s are its group's shared part owns
  // ceil((len - s) / 128) private items and, as one of m members, 1 / m of the group's ceil(s / 128) x ceil(m / members_per_item)
  // shared items -- at most ceil(s / 128) of them: never more than chunks + 1 items per request (tests/test_cascade_plan_host.py
  // checks the bound on the host restatement of the plan).  Round 4 added member_tiles x chunks on top: 9552 instead of 5632
  // workgroups for the bench batch, i.e. 3.9 k more workgroups that leave after one load (~0.25 ns of dispatch each).
  int64_t units = batch * (chunks + 1);
  if (units > max_items) units = max_items;
  const int64_t worst = units * num_kv_heads;
  // (the plan may hold spans: the single-shot form works on its items all the same, and the merge goes by the form launched here)
  p.walks_spans = walks_spans(p.group, head_dim, kv_fp8 != 0) ? 1 : 0;
  const bool loop = worst > (g_cascade_single_shot_units > 0 ? g_cascade_single_shot_units : single_shot_most(chunks, p.walks_spans != 0));
  if (k_new && kv_layout_hnd) {
    // (a launch for the step's rows all the same: beside the addresses of head-major pages the looping form has no scalar registers left for theirs)
    const int rc = sgl_amd_store_kv_cache_ex(k_new, v_new, k_cache, v_cache, new_loc, batch, num_kv_heads, head_dim, k_new_stride, v_new_stride,
                                             k_cache_row_stride, kv_fp8, k_scale, v_scale, page_size, kv_layout_hnd, stream);
    if (rc != 0) return rc;
    k_new = nullptr;
  }
  const int64_t walkers = g_cascade_loop_grid > 0 ? g_cascade_loop_grid : kv_fp8 || head_dim == 64 ? kLoopGridSmallRows : kLoopGrid;
  dim3 grid(static_cast<unsigned>(loop && walkers < worst ? walkers : worst));
#define SGL_LAUNCH_CASC2(D_, KERNEL_)                                                                                 \
  do {                                                                                                       \
    if (kv_fp8 && kv_layout_hnd) hipLaunchKernelGGL((KERNEL_<D_, true, true>), grid, dim3(kThreads), 0, st, p);   \
    else if (kv_fp8) hipLaunchKernelGGL((KERNEL_<D_, true, false>), grid, dim3(kThreads), 0, st, p);             \
    else if (kv_layout_hnd) hipLaunchKernelGGL((KERNEL_<D_, false, true>), grid, dim3(kThreads), 0, st, p);      \
    else hipLaunchKernelGGL((KERNEL_<D_, false, false>), grid, dim3(kThreads), 0, st, p);                        \
  } while (0)
#define SGL_LAUNCH_CASC(D_)                                       \
  do {                                                            \
    if (loop) SGL_LAUNCH_CASC2(D_, cascade_chunk_loop_kernel);    \
    else SGL_LAUNCH_CASC2(D_, cascade_chunk_kernel);              \
  } while (0)
  if (k_new) {
    StoreParams sp;
    sp.chunk = p;
    sp.rows = NewRows{static_cast<const uint16_t*>(k_new), static_cast<const uint16_t*>(v_new), new_loc, k_new_stride, v_new_stride, 1.0f / k_scale, 1.0f / v_scale};
#define SGL_LAUNCH_STORE(KERNEL_)                                                                                                   \
  do {                                                                                                                              \
    if (kv_fp8) hipLaunchKernelGGL((head_dim == 128 ? KERNEL_<128, true> : KERNEL_<64, true>), grid, dim3(kThreads), 0, st, sp);    \
    else hipLaunchKernelGGL((head_dim == 128 ? KERNEL_<128, false> : KERNEL_<64, false>), grid, dim3(kThreads), 0, st, sp);         \
  } while (0)
    if (loop) SGL_LAUNCH_STORE(cascade_store_loop_kernel);
    else SGL_LAUNCH_STORE(cascade_store_kernel);
#undef SGL_LAUNCH_STORE
  } else if (head_dim == 128) SGL_LAUNCH_CASC(128);
  else SGL_LAUNCH_CASC(64);
#undef SGL_LAUNCH_CASC2
#undef SGL_LAUNCH_CASC
  const int hpb = 256 / (head_dim / 4);
  hipLaunchKernelGGL(cascade_merge2_kernel, dim3(static_cast<unsigned>(batch), (num_q_heads + hpb - 1) / hpb), dim3(256), 0, st,
                     p.ws_acc, p.ws_ml, plan, seq_lens, loop && p.walks_spans ? 1 : 0, static_cast<uint16_t*>(out), out_token_stride, p.batch, p.max_items,
                     num_q_heads, head_dim, slots_total, kv_fp8 ? v_scale : 1.0f);
  SGL_CHECK_LAUNCH("cascade_decode_attention");
  return 0;
}

int sgl_amd_debug_cascade_launch_form(int64_t single_shot_units, int64_t loop_grid) {
  SGL_CLEAR_STALE_ERROR();
  SGL_CHECK_ARG(single_shot_units >= 0 && single_shot_units <= kSingleShotHardCap && loop_grid >= 0 && loop_grid <= (1 << 20),
                "debug_cascade_launch_form: single_shot_units must be 0..%lld, loop_grid 0..2^20", (long long)kSingleShotHardCap);
  g_cascade_single_shot_units = single_shot_units;
  g_cascade_loop_grid = loop_grid;
  return 0;
}

}  // extern "C"
