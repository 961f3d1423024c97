// What the format-generic attention kernels and the decode kernel of head dimensions 64 and 128 take.
#pragma once

#include "kvx_device.h"

namespace kvx {

// One tile = row_capacity query rows x `group` query heads of one KV head
// (M fused rows) over the pages of one split.
struct AttendLane {
  const uint64_t *table;
  uint32_t committed, entries, split_count, active_rows;
  uint64_t row_base;   // first fused row of this lane's slots in the workspace
  uint64_t q_offset;   // element offset of the lane's queries / output
  uint32_t mask_offset;
  float score_scale;
};
struct AttendArgs {
  AttendLane lane[KVX_LANES_PER_LAUNCH];
  uint32_t n_lanes;
  uint32_t kv_heads, group, head_dim;
  uint32_t row_capacity;
  uint32_t row_stride;  // rows between KV heads in queries / output
  kvx_kv_layer kv;
  // The merge's second output (see Epilogue), from the launch's first lane on.
  uint16_t *hidden;
  const uint16_t *packed_qkv;
};
__device__ inline bool attend_contract(const AttendLane &l, const AttendArgs &a) {
  return l.active_rows > 0 && l.active_rows <= a.row_capacity &&
         l.entries >= (uint64_t(l.committed) + l.active_rows + KVX_PAGE_TOKENS - 1) / KVX_PAGE_TOKENS &&
         a.kv.extent_pages > 0 &&
         uint64_t(l.committed) + l.active_rows <= uint64_t(KVX_MAX_PHYSICAL_TOKENS) &&
         l.split_count > 0 &&
         l.split_count <= (a.row_capacity == 1 ? KVX_DECODE_MAX_SPLITS : KVX_VERIFY_MAX_SPLITS);
}

}  // namespace kvx
