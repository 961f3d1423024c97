// Verify lanes of 33 to 128 fused query rows on e4m3 and int8 pages and of 33 to 96 on bf16 pages for
// gfx950 (more on bf16 are group_wide_kernel's), and the shared prefix, up to 128 rows, of bf16 and int8
// pages: the rows of one (lane, split, KV head) share every page through LDS (head dimension 256).
//
// A workgroup is R waves of 32 fused rows each and S waves that bring the pages: a page comes in
// once, is expanded once into 16-bit MFMA operands in LDS (two copies, a barrier a page) and is
// multiplied by every wave that has rows with 32x32x16 MFMAs (kvx_page_share.h: the same page against the
// same 32 rows as in chunked prefill).
//
// Why waves apart: what a lane of few rows waits for is the one wave that a SIMD has for it, whose
// products, softmax and share of the staging come one after the other (of 1.9 us a page of int8, 96 rows,
// 1.2 were its own rows, the rest conversion, LDS writes and the wait for memory).  Waves that only stage
// do that beside it: trees of 16 nodes for a group of 6 over 4 x 32 768 tokens, int8 141 -> 98 us (the
// four waves of 24 rows of group_wide_kernel; 146 with these rows and every wave staging), e4m3 133 -> 99,
// bf16 126 -> 108; chains of 8 over 32 x 256 .. 8192 tokens 109 -> 78, 97 -> 78, 113 -> 106; over 30 random
// batches of 33 to 112 rows 1.39, 1.31 and 1.29 times as fast, 1.15 at the least.  Which is what a page costs:
// its bytes (16.6 KiB, e4m3) take 0.7 us at a CU's share of the memory's rate, the 96 rows' MFMAs 0.45.
#include "kvx_page_share.h"

namespace kvx {
namespace {

// QL: the queries of the last QL steps stay in LDS, so that two workgroups of four waves fit a CU (bytes:
// 64 KiB of pages and 14 of queries), or registers are left for the operands AHEAD reads of them.
template <uint32_t FMT, uint32_t R, uint32_t S, uint32_t QL, uint32_t AHEAD>
__global__ __launch_bounds__(64 * (R + S)) __attribute__((amdgpu_waves_per_eu(2, 2))) void verify_lane_kernel(
    const uint16_t *__restrict__ queries, uint16_t *__restrict__ output, float *__restrict__ partials,
    float *__restrict__ statistics, DecodeArgs a) {
  constexpr uint32_t D = kD;
  using Page = Staged<FMT, D>;
  constexpr bool kQuant = FMT != KVX_FMT_BF16;
  constexpr uint32_t kSteps = Page::kSteps, kQueryRegs = kSteps - QL;
  static_assert(FMT != KVX_FMT_INT4, "int4 lanes expand their pages in registers (kvx_decode_int4.hip)");
  __shared__ __align__(16) uint8_t staged[2][Page::kBytes];
  __shared__ __align__(16) float scale_lds[2][2 * kPage];
  __shared__ __align__(16) u32x4 query_lds[QL ? QL : 1][R][64];

  const uint32_t item = blockIdx.x, head = blockIdx.y;
  uint32_t li;
  const DecodeLane l = lane_of_item(a, item, li);
  // Every thread of the workgroup takes the same way out.
  const uint32_t split = item - l.first_item;
  if (split >= l.split_count) return;
  const uint32_t visible = l.committed + l.active_rows;
  const uint32_t pages = (visible + kPage - 1) / kPage;
  const uint32_t per = (pages + l.split_count - 1) / l.split_count;
  const uint32_t written = (pages + per - 1) / per;
  const uint32_t begin = split * per;
  if (begin >= pages) return;
  const uint32_t end = min(pages, begin + per);

  const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 31u, h = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t H = a.kv_heads, G = a.group, M = a.fused_rows;
  const float score_scale = default_score_scale(D, l.score_scale);
  const uint64_t *const entries = l.table + begin;
  const uint32_t count = end - begin, last_slot = count - 1;
  const auto slab_at = [&](uint32_t slot) {
    return slab_of(FMT, H, D, a.kv, head, scalar_entry(entries, min(slot, last_slot)));
  };
  // Two staged copies: while slot i is multiplied, slot i + 1 is staged into the other one.  Past the
  // end the last page is staged again into a copy nobody reads.  A wave's LDS operations (and direct
  // loads) are complete before it comes to the barrier; every wave comes to count + 1 of them.
  const auto barrier = [] {
    if constexpr (kQuant) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
  };
  if (wave >= R) {
    const uint32_t staging = tid - 64 * R;
    PageShare<FMT, D, S> raw;
    if constexpr (kQuant) {
      fetch_share<false>(raw, slab_at(0), staging);
      stage_share(staged[0], scale_lds[0], raw, staging, score_scale);
      fetch_share<false>(raw, slab_at(1), staging);
    } else {
      direct_page<D, S, false>(staged[0], slab_at(0), wave - R, lane);
    }
    barrier();
    for (uint32_t slot = 0; slot < count; ++slot) {
      const uint32_t next = (slot + 1) & 1;
      if constexpr (kQuant) {
        stage_share(staged[next], scale_lds[next], raw, staging, score_scale);
        fetch_share<false>(raw, slab_at(slot + 2), staging);
      } else {
        direct_page<D, S, false>(staged[next], slab_at(slot + 1), wave - R, lane);
      }
      barrier();
    }
    return;
  }

  const uint32_t first_row = 32 * wave, live_rows = l.active_rows * G;
  const bool computes = first_row < live_rows, chain = !l.masks && !a.committed_only;
  const uint32_t fused = first_row + n, row = fused / G;
  const bool live = fused < live_rows;
  // All of the wave's rows see the tokens before whole_to.
  const uint32_t whole_to = l.committed + (chain ? min(first_row / G, l.active_rows - 1) + 1 : 0u);
  const uint64_t head_at = l.q_offset + uint64_t(head) * a.row_stride * G * D;
  const uint16_t *q_row = queries + head_at + (live ? query_at(a, G, row, fused) : 0u);
  u32x4 q[kQueryRegs];
#pragma unroll
  for (uint32_t kb = 0; kb < kSteps; ++kb) {
    u32x4 x = load_global<u32x4>(q_row + 16 * kb + 8 * h);
    if (!live) x = u32x4{0u, 0u, 0u, 0u};
    x = query_operand<FMT>(x);
    if (kb < kQueryRegs) q[kb < kQueryRegs ? kb : 0] = x;
    else query_lds[kb - kQueryRegs][wave][lane] = x;  // (the wave's own: no barrier)
  }
  RowState<D> st;
  st.row_max = -INFINITY;
  st.row_sum = st.weight_sum = 0.0f;
#pragma unroll
  for (uint32_t mb = 0; mb < Page::kBlocks; ++mb)
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) st.acc[mb][i] = 0.0f;

  barrier();
  for (uint32_t slot = 0; slot < count; ++slot) {
    if (computes) {
      const uint8_t *const copy = staged[slot & 1];
      const uint32_t first_token = (begin + slot) * kPage, at = opaque(lane);
      f32x16 s;
      staged_scores<FMT, D, AHEAD>(s, copy, q, [&](uint32_t step, uint32_t at) { return query_lds[step][wave][at]; }, at);
      u32x4 weights[2];
      staged_weights<FMT, D>(
          weights, s, scale_lds[slot & 1], st, score_scale, at, first_token + kPage > whole_to, [&](uint32_t n) {
            const uint32_t fused = first_row + n, row = fused / G;
            const bool live = fused < live_rows;  // (columns without a row see everything, and count for nothing)
            // tokens before `from` are seen, those from `visible` on are not, in between the mask has a bit
            const uint32_t from = !live ? UINT32_MAX : chain ? l.committed + row + 1 : l.committed;
            const uint32_t mask = live && l.masks ? l.masks[row] : 0u;
            return [=](uint32_t place) {
              const uint32_t token = first_token + place;
              return token >= from && (token >= visible || !((mask >> ((token - from) & 31u)) & 1u));
            };
          });
      staged_products<FMT, D, AHEAD>(st, copy, weights, at);
    }
    barrier();
  }

  if (first_row >= M) return;
  const uint32_t at = opaque(lane), half = at >> 5, own = first_row + (at & 31u);
  const bool own_live = own < live_rows;
  const float sum = st.row_sum + other_half(st.row_sum);
  constexpr uint32_t kQuads = D / 8;
  if (written == 1 && !a.all_partials) {  // one split: the merge's weight is exp(0) = 1
    if (own >= M) return;
    const RowQuotient divided(own_live ? sum : 0.0f);  // rows past the live ones read as zeros
    uint16_t *out_row = output + head_at + uint64_t(own) * D;
#pragma unroll
    for (uint32_t k = 0; k < kQuads; ++k) {
      uint32_t dim;
      const f32x4 v = row_quad<FMT, D>(st, k, half, 0.0f, dim);
      u32x2 packed;
#pragma unroll
      for (uint32_t i = 0; i < 2; ++i) {
        const f32x2 pair = {divided(v[2 * i]), divided(v[2 * i + 1])};
        packed[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(pair, bf16x2));
      }
      *reinterpret_cast<u32x2 *>(out_row + dim) = packed;
    }
    return;
  }
  if (!own_live) return;
  const uint64_t slot_row = l.row_base + (uint64_t(head) * l.split_count + split) * M + own;
  float *part = partials + slot_row * D;
#pragma unroll
  for (uint32_t k = 0; k < kQuads; ++k) {
    uint32_t dim;
    const f32x4 v = row_quad<FMT, D>(st, k, half, 0.0f, dim);
    *reinterpret_cast<f32x4 *>(part + dim) = v;
  }
  if (half == 0) *reinterpret_cast<f32x2 *>(statistics + slot_row * 2) = f32x2{st.row_max, sum};
}

}  // namespace
}  // namespace kvx

using namespace kvx;

// Lanes of up to 128 fused rows on bf16, e4m3 and int8 pages of head dimension 256; arguments as
// kvx_attend_wide_launch, which has checked the shape.  Up to 64 rows in two waves, two workgroups of four
// waves to a CU; on bf16 pages up to 96 in three beside one that loads; else four and four, one workgroup to
// a CU (int8, 96 rows, 4 x 32 768 tokens: three waves and one 133 us, four and four 97).
int kvx_verify_lane_launch(const kvx_storage *s, kvx_kv_layer kv, uint32_t query_heads, const void *queries,
                           void *output, const uint64_t *const *page_tables, const kvx_verify_params *lanes,
                           uint32_t n_lanes, const uint32_t *row_masks, uint32_t row_stride, uint64_t lane_stride,
                           void *workspace, uint64_t workspace_bytes, hipStream_t stream, const Epilogue *epilogue) {
  const kvx_layout &l = s->layout;
  const uint32_t M = lanes[0].row_capacity * (query_heads / l.kv_heads);
  const auto launch = [&](auto kernel, uint32_t waves) {
    return launch_matrix_attention(kernel, "verify_lane_kernel", 128, 64 * waves, s, kv, query_heads, queries, output,
                                   page_tables, lanes, n_lanes, row_masks, row_stride, lane_stride, workspace,
                                   workspace_bytes, stream, nullptr, 0, epilogue);
  };
  if (l.format == KVX_FMT_BF16)
    return M <= 64   ? launch(verify_lane_kernel<KVX_FMT_BF16, 2, 2, 0, 3>, 4)
           : M <= 96 ? launch(verify_lane_kernel<KVX_FMT_BF16, 3, 1, 0, 3>, 4)
                     : launch(verify_lane_kernel<KVX_FMT_BF16, 4, 4, 0, 3>, 8);
  if (l.format == KVX_FMT_INT8)
    return M <= 64 ? launch(verify_lane_kernel<KVX_FMT_INT8, 2, 2, 7, 3>, 4)
                   : launch(verify_lane_kernel<KVX_FMT_INT8, 4, 4, 3, 2>, 8);
  return M <= 64 ? launch(verify_lane_kernel<KVX_FMT_FP8E4M3, 2, 2, 7, 3>, 4)
                 : launch(verify_lane_kernel<KVX_FMT_FP8E4M3, 4, 4, 3, 2>, 8);
}
