// Chunked prefill attention for gfx950: 256 consecutive fused query rows of a chunk (row x
// query head of the group) share every page through LDS, head dimensions 64, 128 and 256,
// every page format.
//
// A workgroup is eight waves, two to a SIMD, of 32 fused rows each, on one (sequence, KV head,
// split).  Each page is fetched once for the workgroup, expanded once into 16-bit MFMA operands
// (four copies in LDS, a barrier every second page) and multiplied by every wave with
// 32x32x16 MFMAs: keys x queries gives a lane 16 of its column's 32 scores (a column is a fused
// row), whose weights are then the other operand of values x weights as they lie in registers.
//
// Nothing but the fused row number ties a row to its workgroup, whose rows need not end with a tile.
// The tiles of 8 chunk rows that end in the same page have the same pages [begin, end) of every
// split, and a wave's rows are all of such tiles: four tiles are whole waves whatever the group, and
// where the first page's tiles are fewer than four, the rows start up to 24 columns into the first
// wave.  So a wave takes the pages of its rows' own tiles and no others, and the result of a row is a
// function of the row's own tile, split count and pages (reference:
// prefill/paged_attention.metal:7-206, common/paged_attention_tile.h:85-349,
// common/paged_attention_fp8_tile.h:34-265).  (With waves across such tiles an element that is no
// number, on bf16 or e4m3 pages, reached rows whose tiles end a page before it: weight 0 times NaN.)
//
// Why this shape: every LDS read feeds one 32x32x16 MFMA, so eight waves of 32 rows, each of which
// reads the whole staged page (32 KiB at head dimension 256), ask the LDS for its 128 bytes a
// cycle at the rate the matrix cores take them, and 32 rows are what leaves room for
// two waves a SIMD at head dimension 256 (128 accumulators, 64 queries): one wave's softmax runs
// under the other's MFMAs.  One wave a SIMD of 48 rows (four to a workgroup) had to take them in
// turn: 777 bf16 rows after 8192 tokens 632 -> 216 us a layer, of which 129 were the rows left
// over from whole groups of tiles; two fp8 chunks of 256 rows at 2 x 8 x 128 in one launch 144 ->
// 124 us.  Raised wave priority for half of the waves changed nothing, four waves to a workgroup
// lost 10 to 20 % on small calls.
#include "kvx_page_share.h"

namespace kvx {
namespace {

constexpr uint32_t W = 8, kThreads = 64 * W;              // waves and threads of a workgroup
constexpr uint32_t kWaveRows = 32, kRows = W * kWaveRows;  // fused rows

struct ChunkLane {
  const uint64_t *table;
  uint32_t committed;
  float score_scale;
  uint32_t at;  // the sequence's place in queries and output, in sequence strides
};
struct ChunkArgs {
  ChunkLane lane[kLanes];
  uint32_t sequences, rows, stride, splits;
  uint32_t kv_heads, group;
  uint64_t sequence_stride;  // elements between the sequences' queries and output rows
  uint64_t sequence_rows;    // workspace rows of a sequence
  kvx_kv_layer kv;
};

template <uint32_t FMT, uint32_t D>
__global__ __launch_bounds__(kThreads) __attribute__((amdgpu_waves_per_eu(D == 64 ? 4 : 2, D == 64 ? 4 : 2))) void chunk_attend_kernel(
    const uint16_t *__restrict__ queries, uint16_t *__restrict__ output, float *__restrict__ partials,
    float *__restrict__ statistics, ChunkArgs a) {
  using Page = Staged<FMT, D>;
  constexpr bool kQuant = FMT != KVX_FMT_BF16, kInt4 = FMT == KVX_FMT_INT4;
  constexpr uint32_t kSteps = Page::kSteps, kBlocks = Page::kBlocks;
  constexpr uint32_t T = KVX_PREFILL_TILE_ROWS;
  constexpr uint32_t kCopies = 4;
  __shared__ __align__(16) uint8_t staged[kCopies][Page::kBytes];
  __shared__ __align__(16) float scale_lds[kCopies][2 * kPage];
  // At head dimension 256 accumulators and queries take 192 of a wave's 256 registers; where raw
  // page bytes and scales have to live beside them, the last query blocks stay in LDS.
  constexpr uint32_t kQueryLds = kQuant && D == 256 ? 3 : 0, kQueryRegs = kSteps - kQueryLds;
  __shared__ __align__(16) u32x4 query_lds[kQueryLds ? kQueryLds : 1][W][64];

  // x: (sequence, split, KV head), so that the workgroups that walk the same pages follow one
  // another at a distance and tend to meet on the same XCD; y: 256 columns (fused rows), the last
  // first (they see the most pages).
  const uint32_t H = a.kv_heads, G = a.group;
  const uint32_t head = blockIdx.x % H, split = blockIdx.x / H % a.splits, sequence = blockIdx.x / (H * a.splits);
  const uint64_t *const table = a.lane[sequence].table;
  const uint32_t committed = a.lane[sequence].committed;
  const float score_scale = default_score_scale(D, a.lane[sequence].score_scale);

  const uint32_t tiles = (a.rows + T - 1) / T, fused_rows = tiles * T * G;
  const uint32_t lead = prefill_chunk_lead(committed, G);  // column 0 of the launch is fused row -lead

  // The pages of a tile under this split.
  struct Cut {
    uint32_t begin, end, written;
  };
  const auto cut_of = [&](uint32_t tile) {
    Cut c;
    const uint32_t visible = committed + min(a.rows, (tile + 1) * T);
    const uint32_t pages = (visible + kPage - 1) / kPage, per = (pages + a.splits - 1) / a.splits;
    c.begin = min(pages, split * per);
    c.end = min(pages, c.begin + per);
    c.written = (pages + per - 1) / per;
    return c;
  };
  // The fused rows of columns first_column .. first_column + columns - 1: [first, last], empty when
  // first > last.
  const uint32_t first_column = (gridDim.y - 1 - blockIdx.y) * kRows;
  const auto first_row_of = [&](uint32_t column) { return max(column, lead) - lead; };
  const auto last_row_of = [&](uint32_t column) { return int32_t(min(column, lead + fused_rows - 1)) - int32_t(lead); };
  // The workgroup's pages: from the first tile's first to the last tile's last.  Every thread
  // takes the same way out.
  if (first_column >= lead + fused_rows) return;
  const uint32_t begin = cut_of(first_row_of(first_column) / (T * G)).begin;
  const uint32_t end = cut_of(last_row_of(first_column + kRows - 1) / (T * G)).end;
  if (begin >= end) return;

  const uint32_t tid = threadIdx.x, lane = tid & 63u, n = lane & 31u, h = lane >> 5;
  const uint32_t wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  // Where column n of the wave lies.
  const uint32_t wave_column = first_column + wave * kWaveRows;
  struct Column {
    uint32_t fused, row;
    bool in_tile, live;
  };
  const auto column_of = [&](uint32_t n) {
    Column c;
    c.fused = wave_column + n - lead;  // (wraps below row 0)
    c.row = c.fused / G;
    c.in_tile = c.fused < fused_rows;
    c.live = c.in_tile && c.row < a.rows;
    return c;
  };
  const Column column = column_of(n);
  const bool live = column.live;
  // The wave's pages: none when none of its rows is live.  All of its rows see the tokens before
  // whole_to.
  const uint32_t wave_row = first_row_of(wave_column) / G;
  const int32_t wave_last = last_row_of(wave_column + kWaveRows - 1);
  const bool wave_live = wave_column < lead + fused_rows && wave_last >= 0 && wave_row < a.rows;
  const Cut cut = cut_of(wave_live ? uint32_t(wave_last) / (T * G) : 0);
  const uint32_t wave_first = cut.begin - begin, wave_pages = wave_live ? cut.end - cut.begin : 0u;  // slots
  const uint32_t whole_to = committed + wave_row + 1;

  // Queries: a lane holds 8 dims of every 16 of its column.
  const uint64_t head_row = (uint64_t(head) * a.stride) * G;
  const uint16_t *q_row = queries + a.lane[sequence].at * a.sequence_stride + (head_row + (live ? column.fused : 0u)) * D;
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
  for (uint32_t mb = 0; mb < kBlocks; ++mb)
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) st.acc[mb][i] = 0.0f;

  const uint64_t *const entries = table + begin;
  const uint32_t count = end - begin, last_slot = count - 1;
  const auto slab_at = [&](uint32_t slot) {
    return slab_of(FMT, H, D, a.kv, head, scalar_entry(entries, min(slot, last_slot)));
  };
  PageShare<FMT, D, W> raw;
  // What goes into the key scales: the score scale, but for head dimension 128, whose default is no
  // power of two.
  const float key_unit = D == 128 ? 1.0f : score_scale;

  // A staged page against the wave's rows.
  const auto attend_page = [&](const uint8_t *copy, const float *scales, uint32_t page) __attribute__((always_inline)) {
    constexpr uint32_t kAhead = kQuant ? 2 : 3;
    const uint32_t first_token = page * kPage, at = opaque(lane);
    f32x16 s;
    staged_scores<FMT, D, kAhead>(s, copy, q, [&](uint32_t step, uint32_t at) { return query_lds[step][wave][at]; }, at);
    u32x4 weights[2];
    staged_weights<FMT, D>(weights, s, scales, st, score_scale, at, first_token + kPage > whole_to, [&](uint32_t n) {
      const Column own = column_of(n);  // found again on the few such pages rather than kept
      // (columns without a row see everything, and count for nothing)
      const uint32_t to = own.live ? committed + own.row + 1 : UINT32_MAX;
      return [=](uint32_t place) { return first_token + place >= to; };
    });
    staged_products<FMT, D, kAhead>(st, copy, weights, at);
  };

  // Four staged copies, a barrier every second page: while slots i and i + 1 are multiplied,
  // slots i + 2 and i + 3 are staged into the other pair.  Past the end the last page is
  // staged again into copies nobody reads.  One page a turn of the loop: written out for two,
  // its code was twice as long, and a short launch is the time its instructions take to arrive.
  const auto barrier = [] {
    if constexpr (kQuant) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");  // direct loads have landed
  };
  const uint32_t mine = wave / (W / 2);  // int4: the slots this wave stages, even or odd
  if constexpr (!kQuant) {
    direct_page<D, W>(staged[0], slab_at(0), wave, lane);
    direct_page<D, W>(staged[1], slab_at(1), wave, lane);
  } else if constexpr (kInt4) {
    fetch_share(raw, slab_at(mine), tid);
    stage_share(staged[mine], scale_lds[mine], raw, tid, key_unit);
    fetch_share(raw, slab_at(2 + mine), tid);
  } else {
    for (uint32_t slot = 0; slot < 2; ++slot) {
      fetch_share(raw, slab_at(slot), tid);
      stage_share(staged[slot], scale_lds[slot], raw, tid, key_unit);
    }
    fetch_share(raw, slab_at(2), tid);
  }
  barrier();
  for (uint32_t slot = 0; slot < count; ++slot) {
    const uint32_t now = slot & 3, next = (slot + 2) & 3;
    if constexpr (!kQuant) {
      direct_page<D, W>(staged[next], slab_at(slot + 2), wave, opaque(lane));
    } else if (!kInt4 || (slot & 1) == mine) {
      stage_share(staged[next], scale_lds[next], raw, opaque(tid), key_unit);
      fetch_share(raw, slab_at(slot + (kInt4 ? 4 : 3)), opaque(tid));
    }
    if (slot - wave_first < wave_pages) attend_page(staged[now], scale_lds[now], begin + slot);
    if (slot & 1) barrier();
  }
  if constexpr (!kQuant) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS outlives the wave

  const uint32_t at = opaque(lane), half = at >> 5;
  const float sum = st.row_sum + other_half(st.row_sum);
  const float bias = kInt4 ? kNibbleBias * (st.weight_sum + other_half(st.weight_sum)) : 0.0f;
  constexpr uint32_t kQuads = D / 8;
  const auto quad = [&](uint32_t k, uint32_t &dim) { return row_quad<FMT, D>(st, k, half, bias, dim); };
  const Column place = column_of(at & 31u);  // found again rather than kept through the loop
  if (!place.in_tile) return;
  uint16_t *out_row = output + a.lane[sequence].at * a.sequence_stride + (head_row + place.fused) * D;
  if (!place.live) {  // rows of the last tile past the live ones read as zeros
    if (split == 0)
#pragma unroll
      for (uint32_t k = 0; k < kQuads; ++k) *reinterpret_cast<u32x2 *>(out_row + 8 * k + 4 * half) = u32x2{0u, 0u};
    return;
  }
  if (cut.begin >= cut.end) return;
  if (cut.written == 1) {  // one split: the merge's weight is exp(0) = 1
    const RowQuotient divided(sum);
#pragma unroll
    for (uint32_t k = 0; k < kQuads; ++k) {
      uint32_t dim;
      const f32x4 v = quad(k, dim);
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
  const uint32_t tile = place.row / T;
  const uint64_t slot_row = sequence * a.sequence_rows + ((uint64_t(tile) * H + head) * a.splits + split) * (T * G) +
                            (place.fused - tile * T * G);
  float *part = partials + slot_row * D;
#pragma unroll
  for (uint32_t k = 0; k < kQuads; ++k) {
    uint32_t dim;
    const f32x4 v = quad(k, dim);
    *reinterpret_cast<f32x4 *>(part + dim) = v;
  }
  if (half == 0) *reinterpret_cast<f32x2 *>(statistics + slot_row * 2) = f32x2{st.row_max, sum};
}

// Merge of the rows whose tile has more than one split, in split order (reference:
// common/paged_attention_tile.h:362-417): D / 4 lanes to a row.  The statistics of all splits
// (at most 32) are asked for at once, the partial rows kAhead at a time.
template <uint32_t D>
__global__ __launch_bounds__(256) void chunk_merge_kernel(uint16_t *__restrict__ output,
                                                          const float *__restrict__ partials,
                                                          const float *__restrict__ statistics, ChunkArgs a) {
  constexpr uint32_t T = KVX_PREFILL_TILE_ROWS, kRowLanes = D / 4, kAhead = 8;
  const uint32_t G = a.group, H = a.kv_heads;
  const uint32_t head = blockIdx.y, sequence = blockIdx.z;
  const uint32_t fused = blockIdx.x * (256 / kRowLanes) + threadIdx.x / kRowLanes, lane = threadIdx.x % kRowLanes;
  const uint32_t row = fused / G, tile = row / T;
  if (row >= a.rows) return;
  const uint32_t visible = a.lane[sequence].committed + min(a.rows, (tile + 1) * T);
  const uint32_t pages = (visible + kPage - 1) / kPage, per = (pages + a.splits - 1) / a.splits;
  const uint32_t written = (pages + per - 1) / per;
  if (written == 1) return;
  const uint64_t first = sequence * a.sequence_rows + (uint64_t(tile) * H + head) * a.splits * (T * G) + (fused - tile * T * G);
  const auto part = [&](uint32_t s) {
    return load_global<f32x4>(partials + (first + uint64_t(s) * (T * G)) * D + 4 * lane);
  };
  f32x4 early[kAhead];
#pragma unroll
  for (uint32_t u = 0; u < kAhead; ++u) early[u] = part(min(u, written - 1));
  // lane i of the row's lanes holds the statistics of splits i, i + kRowLanes, ..
  constexpr uint32_t kHeld = kRowLanes >= KVX_PREFILL_MAX_SPLITS ? 1 : KVX_PREFILL_MAX_SPLITS / kRowLanes;
  f32x2 stat[kHeld];
  float maximum = -INFINITY;
#pragma unroll
  for (uint32_t i = 0; i < kHeld; ++i) {
    const uint32_t s = lane + i * kRowLanes;
    stat[i] = s < written ? load_global<f32x2>(statistics + (first + uint64_t(s) * (T * G)) * 2) : f32x2{-INFINITY, 0.0f};
    maximum = fmaxf(maximum, stat[i][0]);
  }
#pragma unroll
  for (uint32_t offset = kRowLanes / 2; offset; offset >>= 1) maximum = fmaxf(maximum, __shfl_xor(maximum, offset));
  float weight[kHeld], term[kHeld];
#pragma unroll
  for (uint32_t i = 0; i < kHeld; ++i) {
    weight[i] = expf(__fsub_rn(stat[i][0], maximum));
    term[i] = __fmul_rn(weight[i], stat[i][1]);
  }
  f32x4 numerator = {0.0f, 0.0f, 0.0f, 0.0f};
  float denominator = 0.0f;
  for (uint32_t base = 0; base < written; base += kAhead) {
    f32x4 p[kAhead];
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) p[u] = base ? part(min(base + u, written - 1)) : early[u];
    const uint32_t held = kHeld == 1 ? 0 : base / kRowLanes;
#pragma unroll
    for (uint32_t u = 0; u < kAhead; ++u) {
      const uint32_t s = base + u;
      const float w = __shfl(held ? weight[kHeld - 1] : weight[0], int(s % kRowLanes), kRowLanes);
      const float t = __shfl(held ? term[kHeld - 1] : term[0], int(s % kRowLanes), kRowLanes);
      if (s < written) {
#pragma unroll
        for (uint32_t c = 0; c < 4; ++c) numerator[c] = __fadd_rn(numerator[c], __fmul_rn(w, p[u][c]));
        denominator = __fadd_rn(denominator, t);
      }
    }
  }
  u32x2 packed;
#pragma unroll
  for (uint32_t i = 0; i < 2; ++i)
    packed[i] = uint32_t(f32_to_bf16(denominator > 0.0f ? __fdiv_rn(numerator[2 * i], denominator) : 0.0f)) |
                uint32_t(f32_to_bf16(denominator > 0.0f ? __fdiv_rn(numerator[2 * i + 1], denominator) : 0.0f)) << 16;
  *reinterpret_cast<u32x2 *>(output + a.lane[sequence].at * a.sequence_stride + ((uint64_t(head) * a.stride) * G + fused) * D + 4 * lane) = packed;
}

}  // namespace
}  // namespace kvx

using namespace kvx;

// The chunks of up to 32 sequences (equal rows, stride and split count) in one launch of each
// kernel: sequences at[0], at[1], .. of the caller's arrays.  0 when enqueued, or a negative status.
// The caller has checked the parameters, that prefill_by_chunk takes them, and the workspace's
// size (rows x D + 2 floats per workspace row).
int kvx_prefill_chunk_launch(const kvx_storage *s, kvx_kv_layer kv, uint32_t query_heads, const void *queries,
                             void *output, const uint64_t *const *page_tables, const kvx_prefill_params *params,
                             const uint32_t *at, uint32_t sequences, uint64_t sequence_stride, void *workspace,
                             hipStream_t stream) {
  const kvx_layout &l = s->layout;
  const uint32_t H = l.kv_heads, G = query_heads / H, D = l.head_dim, T = KVX_PREFILL_TILE_ROWS;
  const kvx_prefill_params &first = params[at[0]];
  const uint32_t rows = first.rows, splits = first.split_count, tiles = (rows + T - 1) / T;
  ChunkArgs a{};
  for (uint32_t i = 0; i < sequences; ++i) {
    const kvx_prefill_params &p = params[at[i]];
    a.lane[i] = {page_tables[at[i]], p.committed_tokens, p.score_scale != 0.0f ? p.score_scale : l.score_scale, at[i]};
  }
  a.sequences = sequences;
  a.rows = rows;
  a.stride = first.chunk_stride;
  a.splits = splits;
  a.kv_heads = H;
  a.group = G;
  a.sequence_stride = sequence_stride;
  a.sequence_rows = uint64_t(tiles) * H * splits * T * G;
  a.kv = kv;
  float *partials = static_cast<float *>(workspace);
  float *statistics = partials + sequences * a.sequence_rows * D;
  // columns: the fused rows behind the kernel's `lead`
  uint32_t lead = 0;
  for (uint32_t i = 0; i < sequences; ++i)
    lead = std::max(lead, prefill_chunk_lead(a.lane[i].committed, G));
  const uint32_t columns = lead + tiles * T * G;
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(H * splits * sequences, (columns + kRows - 1) / kRows),
                       dim3(kThreads), 0, stream, static_cast<const uint16_t *>(queries),
                       static_cast<uint16_t *>(output), partials, statistics, a);
  };
#define KVX_CHUNK(D_)                                                                    \
  (l.format == KVX_FMT_INT4   ? launch(chunk_attend_kernel<KVX_FMT_INT4, D_>)              \
   : l.format == KVX_FMT_INT8 ? launch(chunk_attend_kernel<KVX_FMT_INT8, D_>)              \
   : l.format == KVX_FMT_BF16 ? launch(chunk_attend_kernel<KVX_FMT_BF16, D_>)              \
                              : launch(chunk_attend_kernel<KVX_FMT_FP8E4M3, D_>))
  if (D == 256) KVX_CHUNK(256);
  else if (D == 128) KVX_CHUNK(128);
  else KVX_CHUNK(64);
#undef KVX_CHUNK
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return hip_fail(e, "chunk_attend_kernel");
  if (splits == 1) return 0;
  const uint32_t to_a_group = 1024 / D;  // rows
  const dim3 grid((rows * G + to_a_group - 1) / to_a_group, H, sequences);
  if (D == 256) hipLaunchKernelGGL(chunk_merge_kernel<256>, grid, dim3(256), 0, stream, static_cast<uint16_t *>(output), partials, statistics, a);
  else if (D == 128) hipLaunchKernelGGL(chunk_merge_kernel<128>, grid, dim3(256), 0, stream, static_cast<uint16_t *>(output), partials, statistics, a);
  else hipLaunchKernelGGL(chunk_merge_kernel<64>, grid, dim3(256), 0, stream, static_cast<uint16_t *>(output), partials, statistics, a);
  if (const hipError_t e = hipGetLastError(); e != hipSuccess) return hip_fail(e, "chunk_merge_kernel");
  return 0;
}
