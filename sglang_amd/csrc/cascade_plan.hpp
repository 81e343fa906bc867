// Layout of the shared-prefix (cascade) decode plan, an int32 array produced on the device by
// sgl_amd_cascade_plan and consumed by the cascade attention kernels (no host involvement, so
// the whole thing is recorded into the decode hipGraph).
//
//   header[8]            [0] n_items  [1] n_groups  [2] n_member_rows  [3] shared items  [4] 64-token tiles of a span (0: no spans)  [5] units of the looping kernel
//   req_shared[B]        kv tokens of request b that are covered by its group's shared part (0 = none)
//   member_rows[B]       batch indices sorted by group (the "query tokens" of a group)
//   group_qo[B + 1]      member_rows range of each group
//   group_pool_row[B]    req_to_token row of the group's leader
//   group_kvlen[B]       shared kv length of the group (multiple of the kv tile)
//   items[8 * max_items] self-contained records: (group, kv chunk, row tile, members, first member_rows
//                        index, kv tokens, req_to_token row of the leader, 0); members == 0: unused entry
//   batch_order[B]       permutation of the batch: grouped requests (group by group) first, then the rest
//   req_slots[B]         partial slots of request b: its shared chunks, then its private items or pieces
//   span_first[kSpanUnits + 1], pieces[8 * (B + kSpanUnits)]   (header[4] > 0) span k is pieces span_first[k] .. span_first[k + 1] - 1, records like
//                        the items'; they stand in the place of the private items for the looping attention kernel
//   compare[2 B]         scratch between the plan's two launches: leader of request b, its common prefix with the leader
//   new_slots[B]         the slots that the plan was told the step's rows go to (if it was)
//   meet[kCheckers]      what was found of them, a word of PlanFound bits a workgroup that looked (it was not told: kPlanUntold)
//   met_rows[kCheckers * 32]  the rows of the step that such a workgroup found something of, a bit each, where its word is not 0
#pragma once
#include <stdint.h>

namespace sgl_amd {

struct CascadePlanView {
  int32_t* header;
  int32_t* req_shared;
  int32_t* member_rows;
  int32_t* group_qo;
  int32_t* group_pool_row;
  int32_t* group_kvlen;
  int32_t* items;
  int32_t* batch_order;
  int32_t* compare;
  int32_t* req_slots;
  int32_t* span_first;
  int32_t* pieces;
  int32_t* new_slots;
  int32_t* meet;
  int32_t* met_rows;
};

// (span, kv head) units that a plan of spans aims at, the shared items taken off: three a compute unit.  The looping kernel's registers would
// let four run, but the chip starts about 740 of a thousand workgroups at once and the rest only as those end, a second round of a fifth of
// the work (us for four layers at 1024 / 768 units: 37 requests of 0.9 to 5.1 k tokens in e4m3 278 / 268, 16 of 4 k in bf16 297 / 280, 64
// behind shared prefixes, eight layers, 255 / 234; 640 and 896 units lose 4 to 8 %; with 32 kv heads of one row, where a workgroup waits
// for its instructions more than for memory, 321 / 345; the items are behind both there, 16 requests of 2 k 530 / 470 in 768 spans, 32 of 400
// 280 / 241, 37 of 1 k 601 / 530).  Below three 64-token tiles a span the items' single burst is quicker
// (32 requests of 190 tokens behind a shared prefix 93 us, 100 in spans of two).
// Nor where the items are no more than run in one round (7 requests of 585 tokens, 32 kv heads: 896 items 123 us, 768 spans 125), nor where the
// shared items take more than half of these units: the spans left are long and few, and the last of them begin when shared items end (us for
// four layers, spans / items: 128 requests of 100 tokens behind one prefix of 2 k 254 / 188, 128 of 130 in 16 groups behind 1 k 301 / 228, 100
// of 190 behind 1 k 191 / 176, 32 kv heads, 64 of 100 behind 2 k 260 / 224; at exactly half 64 in 4 groups, 1.5 k and 300, 176 / 185).
constexpr int kSpanUnits = 768;
constexpr int kOneRoundUnits = 1024;
constexpr int kMinSpanTiles = 3;
constexpr int kCheckers = 64;        // workgroups that look through the request tables for the new slots, one word each
enum PlanFound { kPlanMeet = 1, kPlanUnread = 2, kPlanUntold = 4 };   // a request reads a new slot that is not its own newest token's, or two rows have one; a request has no tokens

__host__ __device__ inline int64_t cascade_plan_ints(int64_t batch, int64_t max_items) {
  return 8 + batch + batch + (batch + 1) + batch + batch + 8 * max_items + batch + 2 * batch + batch + (kSpanUnits + 1) + 8 * (batch + kSpanUnits) + 3 + batch +
         kCheckers + kCheckers * 32;
}

__host__ __device__ inline CascadePlanView cascade_plan_view(const int32_t* plan, int64_t batch, int64_t max_items) {
  CascadePlanView v;
  int32_t* p = const_cast<int32_t*>(plan);
  v.header = p; p += 8;
  v.req_shared = p; p += batch;
  v.member_rows = p; p += batch;
  v.group_qo = p; p += batch + 1;
  v.group_pool_row = p; p += batch;
  v.group_kvlen = p; p += batch;
  v.items = p; p += 8 * max_items;
  v.batch_order = p; p += batch;
  v.compare = p; p += 2 * batch;
  v.req_slots = p; p += batch;
  v.span_first = p; p += kSpanUnits + 1;
  v.pieces = v.header + ((p - v.header + 3) & ~static_cast<int64_t>(3));   // 16-byte records
  v.new_slots = v.pieces + 8 * (batch + kSpanUnits);
  v.meet = v.new_slots + batch;
  v.met_rows = v.meet + kCheckers;
  return v;
}

}  // namespace sgl_amd
