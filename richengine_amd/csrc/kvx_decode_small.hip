// One-row decode at head dimensions 64 and 128 for gfx950, every page format: a wave per (lane, split, group of
// P KV heads, one or two) streams the split's pages once, in registers.
//
// The P heads' query rows are the columns of one 16-wide MFMA block: keys (16 tokens x 32 dims) x queries
// gives every column its products with every head's keys, head by head, and a lane keeps those of its own
// column's head; the page's softmax is then taken once for all P heads, and values (16 dims x 32
// tokens) x weights go to accumulators of each head, of which a column's own head counts.  No product of
// one head reaches a row of another, so an element that is no number stays in its head.
//
// Why this form: a wave per head over a staged copy of its values (attend_split_small_wave_kernel) took the
// softmax of a page for the 4 or 8 columns a head has, and passed every value through LDS two or
// four bytes at a time.  With the step's token stored here too, a layer at 8 x 4 x 64: 32 int8 sequences of 700 ..
// 8192 tokens 62.0 -> 40.0 us, int4 63.0 -> 37.4, bf16 of half the length 49.6 -> 37.1, one of 500 int8 tokens 15.5 ->
// 12.9; at 2 x 8 x 128, int4, 40.0 -> 31.3 and 18.8 -> 13.8, bf16 33.4 -> 29.9 and 15.3 -> 12.8.  Bound by the memory:
// 32 x 8192 int8 tokens, slabs of 2 KiB, take 49.3 us in this kernel, 5.8 TB/s, and 61.7 a layer with the merge.
//
// Lane geometry (t = lane & 15, g = lane >> 4): key operand row t of token block tb is token 8 (t / 4) + 4 tb +
// t % 4, so that lane (t, g) holds column t's scores of tokens 8g .. 8g + 7; the value operands' k-slots are
// the same eight tokens, and the rounded weights the other operand as they are.
#include "kvx_page_share.h"
#include "kvx_small_args.h"

namespace kvx {
namespace {

template <uint32_t FMT>
__device__ __forceinline__ f32x4 mfma16(u32x4 a, u32x4 b, f32x4 c) {
  if constexpr (kHalfOperands<FMT>)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// The step's token, to be stored by the wave that owns a sequence's last page (keys null: it is stored).
struct SmallToken {
  const uint16_t *keys, *values;
  uint64_t lane_stride;
  uint32_t stride;
};

// The token's key and value row of one head: the arithmetic of append_kernel (reference:
// common/paged_store_row.h:47-147, paged_store_row_fp8.h:28-78), D / 64 consecutive dims to a lane.
template <uint32_t FMT, uint32_t D>
__device__ __forceinline__ void append_small_token(const SmallToken &a, const AttendLane &l, uint32_t li, uint32_t H,
                                                   kvx_kv_layer kv, uint32_t head, uint32_t lane) {
  constexpr uint32_t E = D / 64;
  const uint32_t slot = l.committed % kPage;
  const Slab slab = slab_of(FMT, H, D, kv, head, l.table[l.committed / kPage]);
  const uint16_t *key_row = a.keys + li * a.lane_stride + uint64_t(head) * a.stride * D + E * lane;
  const uint16_t *value_column = a.values + li * a.lane_stride + (uint64_t(head) * D + E * lane) * a.stride;
  uint16_t row[2][E];
#pragma unroll
  for (uint32_t i = 0; i < E; ++i) {
    row[0][i] = load_global<uint16_t>(key_row + i);
    row[1][i] = load_global<uint16_t>(value_column + uint64_t(i) * a.stride);
  }
#pragma unroll
  for (uint32_t tensor = 0; tensor < 2; ++tensor) {
    uint8_t *data = tensor ? slab.values : slab.keys;
    // element of dim d: token-major keys (and int4 values), dimension-major values
    const auto at = [&](uint32_t d) { return tensor && FMT != KVX_FMT_INT4 ? d * kPage + slot : slot * D + d; };
    if constexpr (FMT == KVX_FMT_BF16) {
#pragma unroll
      for (uint32_t i = 0; i < E; ++i) store_global<uint16_t>(data + 2 * at(E * lane + i), row[tensor][i]);
    } else {
      float maximum = fabsf(bf16_to_f32(row[tensor][0]));  // (not from 0: a row of nothing but NaN has no maximum)
#pragma unroll
      for (uint32_t i = 1; i < E; ++i) maximum = fmaxf(maximum, fabsf(bf16_to_f32(row[tensor][i])));
      for (int offset = 32; offset; offset >>= 1) maximum = fmaxf(maximum, __shfl_xor(maximum, offset));
      constexpr float kMost = FMT == KVX_FMT_INT4 ? 7.0f : FMT == KVX_FMT_INT8 ? 127.0f : 448.0f;
      constexpr int kLimit = FMT == KVX_FMT_INT4 ? 7 : 127;
      uint32_t code[E];
#pragma unroll
      for (uint32_t i = 0; i < E; ++i) {
        const float scaled = maximum == 0.0f ? 0.0f : __fdiv_rn(__fmul_rn(bf16_to_f32(row[tensor][i]), kMost), maximum);
        if constexpr (FMT == KVX_FMT_FP8E4M3) {
          code[i] = f32_to_e4m3(scaled);
        } else {
          const int c = int(rintf(scaled));
          code[i] = uint32_t(c < -kLimit ? -kLimit : c > kLimit ? kLimit : c);
        }
        if (maximum == 0.0f) code[i] = 0;
      }
      if constexpr (FMT != KVX_FMT_INT4) {
#pragma unroll
        for (uint32_t i = 0; i < E; ++i) store_global<uint8_t>(data + at(E * lane + i), uint8_t(code[i]));
      } else if constexpr (E == 2) {
        store_global<uint8_t>(data + at(2 * lane) / 2, uint8_t((code[0] & 0xfu) | (code[1] & 0xfu) << 4));
      } else {
        const uint32_t next = __shfl_xor(code[0], 1);
        if (!(lane & 1)) store_global<uint8_t>(data + at(lane) / 2, uint8_t((code[0] & 0xfu) | (next & 0xfu) << 4));
      }
      if (lane == 0)
        store_global<float>((tensor ? slab.value_scales : slab.key_scales) + slot,
                            maximum == 0.0f ? 0.0f : __fdiv_rn(maximum, kMost));
    }
  }
}

// A page's keys and values as they lie, for P heads; read by columns of 16 lanes.
template <uint32_t FMT, uint32_t D, uint32_t P>
struct SmallPage {
  static constexpr bool kInt4 = FMT == KVX_FMT_INT4, kBf16 = FMT == KVX_FMT_BF16;
  static constexpr uint32_t kSteps = D / 32;  // of 32 dims
  static constexpr uint32_t kRow = kInt4 ? D / 2 : kBf16 ? 2 * D : D, kSlab = kPage * kRow;
  // int4 at head dimension 64: the 32 bytes of a token are eight lanes, so a load takes two heads
  static constexpr bool kPairs = kInt4 && D == 64;
  static constexpr uint32_t kGroups = kPairs ? (P + 1) / 2 : P;          // accumulator groups
  static constexpr uint32_t kTiles = kInt4 ? 8 : D / 16;                 // of 16 rows, to a group
  static constexpr uint32_t kKeyWords = kRow / 16;                       // dwords of a token block to a lane and head
  static constexpr uint32_t kValueWords = kInt4 ? 8 : kBf16 ? D / 4 : D / 8;
  uint32_t k[P][2][kKeyWords];
  uint32_t v[kGroups][kValueWords];

  // N dwords to places i, i + 1, .. of an array.
  template <uint32_t N, uint32_t L>
  __device__ __forceinline__ static void load(uint32_t (&to)[L], uint32_t i, const uint8_t *from) {
    if constexpr (N == 4) {
      const u32x4 x = load_streaming<u32x4>(from);
      to[i] = x[0], to[i + 1] = x[1], to[i + 2] = x[2], to[i + 3] = x[3];
    } else if constexpr (N == 2) {
      const u32x2 x = load_streaming<u32x2>(from);
      to[i] = x[0], to[i + 1] = x[1];
    } else {
      to[i] = load_streaming<uint32_t>(from);
    }
  }
  // Dims of step kb that lane group g multiplies: eight from here on.
  __device__ __forceinline__ static uint32_t dims(uint32_t kb, uint32_t g) {
    if constexpr (kBf16) return 32 * kb + 8 * g;
    else if constexpr (kInt4) return D / 4 * g + 8 * kb;
    else return 64 * (kb >> 1) + 16 * g + 8 * (kb & 1);
  }
  __device__ __forceinline__ void load_keys(const uint8_t *keys, uint32_t t, uint32_t g) {
#pragma unroll
    for (uint32_t p = 0; p < P; ++p)
#pragma unroll
      for (uint32_t tb = 0; tb < 2; ++tb) {
        const uint8_t *row = keys + p * kSlab + (8 * (t >> 2) + 4 * tb + (t & 3)) * kRow;
        if constexpr (kInt4) {
          load<kKeyWords>(k[p][tb], 0, row + 4 * kKeyWords * g);
        } else {
          constexpr uint32_t kLoads = kKeyWords / 4;  // 64 bytes of a token each
#pragma unroll
          for (uint32_t j = 0; j < kLoads; ++j) load<4>(k[p][tb], 4 * j, row + 64 * j + 16 * g);
        }
      }
  }
  __device__ __forceinline__ void load_values(const uint8_t *values, uint32_t t, uint32_t g) {
#pragma unroll
    for (uint32_t c = 0; c < kGroups; ++c) {
      if constexpr (kPairs) {
        const uint8_t *from = values + (P == 1 ? 0u : 2 * c + (t >> 3)) * kSlab + 8 * g * kRow + 4 * (t & 7);
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) load<1>(v[c], i, from + i * kRow);
      } else if constexpr (kInt4) {
        const uint8_t *from = values + c * kSlab + 8 * g * kRow + 4 * t;
#pragma unroll
        for (uint32_t i = 0; i < 8; ++i) load<1>(v[c], i, from + i * kRow);
      } else {
        constexpr uint32_t B = kBf16 ? 2 : 1;
#pragma unroll
        for (uint32_t mb = 0; mb < kTiles; ++mb)
          load<2 * B>(v[c], 2 * B * mb, values + c * kSlab + ((16 * mb + t) * kPage + 8 * g) * B);
      }
    }
  }
  __device__ __forceinline__ u32x4 key_operand(uint32_t p, uint32_t tb, uint32_t kb) const {
    const uint32_t (&w)[kKeyWords] = k[p][tb];
    if constexpr (kBf16) {
      return u32x4{w[4 * kb], w[4 * kb + 1], w[4 * kb + 2], w[4 * kb + 3]};
    } else if constexpr (kInt4) {  // dims 0, 2, 4, 6, 1, 3, 5, 7 of the eight
      const uint32_t lo = signed_nibbles(w[kb]), hi = signed_nibbles(w[kb] >> 4);
      return u32x4{nibble_pair<false>(lo), nibble_pair<true>(lo), nibble_pair<false>(hi), nibble_pair<true>(hi)};
    } else {
      return byte_operand<FMT>(w[2 * kb], w[2 * kb + 1]);
    }
  }
  // The products of a group's values and the weights: tile by tile.
  template <class Product>
  __device__ __forceinline__ void each_value(uint32_t c, Product product) const {
    if constexpr (kInt4) {
      uint32_t w[8];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) w[i] = v[c][i] ^ 0x88888888u;  // code + 8
#pragma unroll
      for (uint32_t b = 0; b < 4; ++b) {  // byte b of every token: dims 2 b (low nibble) and 2 b + 1 of its eight
        const uint32_t select = 0x0c0c0400u + 0x0101u * b;
        const uint32_t first = __builtin_amdgcn_perm(w[1], w[0], select) | (__builtin_amdgcn_perm(w[3], w[2], select) << 16);
        const uint32_t second = __builtin_amdgcn_perm(w[5], w[4], select) | (__builtin_amdgcn_perm(w[7], w[6], select) << 16);
#pragma unroll
        for (uint32_t n = 0; n < 2; ++n) {
          const uint32_t lo = (n ? first >> 4 : first) & 0x0f0f0f0fu, hi = (n ? second >> 4 : second) & 0x0f0f0f0fu;
          product(2 * b + n, u32x4{nibble_pair<false>(lo), nibble_pair<true>(lo), nibble_pair<false>(hi), nibble_pair<true>(hi)});
        }
      }
    } else {
#pragma unroll
      for (uint32_t mb = 0; mb < kTiles; ++mb) {
        if constexpr (kBf16) product(mb, u32x4{v[c][4 * mb], v[c][4 * mb + 1], v[c][4 * mb + 2], v[c][4 * mb + 3]});
        else product(mb, byte_operand<FMT>(v[c][2 * mb], v[c][2 * mb + 1]));
      }
    }
  }
};

// WAVES: to a SIMD.
template <uint32_t FMT, uint32_t D, uint32_t P, uint32_t WAVES>
__global__ __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(WAVES, WAVES))) void decode_small_kernel(
    const uint16_t *__restrict__ queries, float *__restrict__ partials, float *__restrict__ statistics, AttendArgs a,
    SmallToken token) {
  using Page = SmallPage<FMT, D, P>;
  constexpr bool kQuant = FMT != KVX_FMT_BF16, kInt4 = FMT == KVX_FMT_INT4;
  constexpr uint32_t kSteps = Page::kSteps;
  // (split, group of heads) pairs, the groups fastest: the heads of a page lie side by side.
  const uint32_t flat = blockIdx.x, groups = a.kv_heads / P;
  const uint32_t split = flat / groups, head0 = P * (flat - split * groups), li = blockIdx.y;
  const AttendLane &l = a.lane[li];
  if (!attend_contract(l, a) || split >= l.split_count) return;
  const uint32_t H = a.kv_heads, G = a.group;
  const uint32_t visible = l.committed + 1, pages = (visible + kPage - 1) / kPage;
  const uint32_t per = (pages + l.split_count - 1) / l.split_count, begin = split * per;
  if (begin >= pages) return;
  const uint32_t end = min(pages, begin + per);
  const uint32_t lane = threadIdx.x & 63u, t = lane & 15u, g = lane >> 4;
  // Column t: query head `own_row` of the group's head `own`.
  const uint32_t own = min(t / G, P - 1), own_row = min(t - own * G, G - 1);
  const bool live = t < P * G;
  const float score_scale = default_score_scale(D, l.score_scale);

  const uint64_t *const entries = l.table + begin;
  const uint32_t last_slot = end - begin - 1;
  // One register set of pages (with two, twelve of sixteen batches were slower, by up to 13 %): the keys of the
  // next page are asked for when this page has multiplied its last key, its values when the page is done.
  Page page;
  f32x4 ks[2], vs[2];  // scales of the column's head, tokens 8g ..
  const auto fetch_keys = [&](const Slab &s) {
    asm volatile("");
    page.load_keys(s.keys, t, g);
    if constexpr (kQuant) {
      ks[0] = load_global<f32x4>(s.key_scales + own * kPage + 8 * g);
      ks[1] = load_global<f32x4>(s.key_scales + own * kPage + 8 * g + 4);
    }
    asm volatile("");
  };
  const auto fetch_values = [&](const Slab &s) {
    asm volatile("");
    page.load_values(s.values, t, g);
    if constexpr (kQuant) {
      vs[0] = load_global<f32x4>(s.value_scales + own * kPage + 8 * g);
      vs[1] = load_global<f32x4>(s.value_scales + own * kPage + 8 * g + 4);
    }
    asm volatile("");
  };
  const auto slab_at = [&](uint64_t entry) { return slab_of(FMT, H, D, a.kv, head0, entry); };
  // The wave that owns the sequence's last page stores the step's token: before anything else when that
  // page is the first it loads, otherwise behind the first loads.
  const bool appends = token.keys != nullptr && end == pages, appends_first = appends && end - begin == 1;
  const auto append = [&] {
#pragma unroll 1
    for (uint32_t p = 0; p < P; ++p) append_small_token<FMT, D>(token, l, li, H, a.kv, head0 + p, lane);
    __builtin_amdgcn_s_waitcnt(0x0F70);  // vmcnt(0): the page is loaded after them
  };
  if (appends_first) append();
  uint64_t upcoming = scalar_entry(entries, 0);  // the entry of the next page
  {
    const Slab first = slab_at(upcoming);
    fetch_keys(first);
    fetch_values(first);
    upcoming = scalar_entry(entries, min(1u, last_slot));
  }
  if (appends && !appends_first) append();

  const uint16_t *q_row = queries + l.q_offset + (uint64_t(head0 + own) * a.row_stride * G + own_row) * D;
  u32x4 q[kSteps];
#pragma unroll
  for (uint32_t kb = 0; kb < kSteps; ++kb) {
    u32x4 x = load_global<u32x4>(q_row + Page::dims(kb, g));
    if (!live) x = u32x4{0u, 0u, 0u, 0u};
    q[kb] = query_operand<FMT>(x);
  }
  f32x4 acc[Page::kGroups][Page::kTiles];
#pragma unroll
  for (uint32_t c = 0; c < Page::kGroups; ++c)
#pragma unroll
    for (uint32_t i = 0; i < Page::kTiles; ++i) acc[c][i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float row_max = -INFINITY, row_sum = 0.0f, weight_sum = 0.0f;

  // A page of the split; kLast: its last, the only one that can hold slots past the visible tokens, behind which
  // nothing is asked for.  (With the last page asked for once more, so that one copy of the code serves all, splits
  // of two to four pages took a quarter to a half more of the memory: bf16, 8 x 4000 tokens at 8 x 8 x 128 in 64
  // splits 51.7 us a layer, now 42.1; 11 sequences of 2938 .. 5876 at 3 x 16 x 128 under the plan 32.2, now 30.0;
  // int8, 32 x 700 .. 8192 at 8 x 4 x 64 42.1, now 40.9.)
  const auto attend = [&](uint32_t at, auto last) __attribute__((always_inline)) {
    constexpr bool kLast = decltype(last)::value;
    f32x4 s[2];
#pragma unroll
    for (uint32_t p = 0; p < P; ++p)
#pragma unroll
      for (uint32_t tb = 0; tb < 2; ++tb) {
        f32x4 mine = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (uint32_t kb = 0; kb < kSteps; ++kb) mine = mfma16<FMT>(page.key_operand(p, tb, kb), q[kb], mine);
#pragma unroll
        for (uint32_t i = 0; i < 4; ++i) s[tb][i] = p == 0 || own == p ? mine[i] : s[tb][i];
      }
    const f32x4 page_ks[2] = {ks[0], ks[1]}, page_vs[2] = {vs[0], vs[1]};
    const Slab next = slab_at(upcoming);
    if constexpr (!kLast) {
      fetch_keys(next);
      upcoming = scalar_entry(entries, min(at + 2 - begin, last_slot));
    }
    const uint32_t first_token = at * kPage + 8 * g;
    const bool whole = !kLast || (at + 1) * kPage <= visible;
    float score[8], local_max = -INFINITY;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      float x = s[i >> 2][i & 3];
      if constexpr (kQuant) x = __fmul_rn(x, page_ks[i >> 2][i & 3]);
      score[i] = __fmul_rn(x, score_scale);
    }
    if (!whole) {
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i)
        if (first_token + i >= visible) score[i] = -INFINITY;
    }
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) local_max = fmaxf(local_max, score[i]);
    local_max = fmaxf(local_max, __shfl_xor(local_max, 16));
    local_max = fmaxf(local_max, __shfl_xor(local_max, 32));
    const float next_max = fmaxf(row_max, local_max);
    const bool grows = next_max != row_max && next_max != -INFINITY;
    const float rescale = grows ? expf(__fsub_rn(row_max, next_max)) : 1.0f;
    // A row that has seen nothing yet measures from 0: -inf - -inf is no number.
    const float reference = next_max == -INFINITY ? 0.0f : next_max;
    float weight[8], page_sum = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      const float p = expf(__fsub_rn(score[i], reference));
      page_sum = __fadd_rn(page_sum, p);
      weight[i] = kQuant ? __fmul_rn(p, page_vs[i >> 2][i & 3]) : p;
    }
    // What an earlier sequence left in an unseen slot may have an infinite scale, or none.
    if (!whole) {
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i)
        if (first_token + i >= visible) weight[i] = 0.0f;
    }
    row_sum = __fadd_rn(__fmul_rn(row_sum, rescale), page_sum);
    row_max = next_max;
    u32x4 weights;
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      if constexpr (kHalfOperands<FMT>) {
        const f16x2 pair = {_Float16(weight[2 * i]), _Float16(weight[2 * i + 1])};
        weights[i] = __builtin_bit_cast(uint32_t, pair);
      } else {
        weights[i] = __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{weight[2 * i], weight[2 * i + 1]}, bf16x2));
      }
    }
    if (__builtin_amdgcn_ballot_w64(grows)) {
      if constexpr (kInt4) weight_sum *= rescale;
#pragma unroll
      for (uint32_t c = 0; c < Page::kGroups; ++c)
#pragma unroll
        for (uint32_t i = 0; i < Page::kTiles; ++i) acc[c][i] *= rescale;
    }
    if constexpr (kInt4) {
      const bf16x2 ones = {__bf16(1.0f), __bf16(1.0f)};
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t pair = weights[i];
        weight_sum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), ones, weight_sum, false);
      }
    }
#pragma unroll
    for (uint32_t c = 0; c < Page::kGroups; ++c)
      page.each_value(c, [&](uint32_t i, u32x4 v) { acc[c][i] = mfma16<FMT>(v, weights, acc[c][i]); });
    if constexpr (!kLast) fetch_values(next);
  };
  for (uint32_t at = begin; at + 1 < end; ++at) attend(at, std::false_type{});
  attend(end - 1, std::true_type{});

  // The lanes of a column hold disjoint tokens.
  float sum = row_sum, bias = 0.0f;
  sum = __fadd_rn(sum, __shfl_xor(sum, 16));
  sum = __fadd_rn(sum, __shfl_xor(sum, 32));
  if constexpr (kInt4) {
    weight_sum += __shfl_xor(weight_sum, 16);
    bias = kNibbleBias * (weight_sum + __shfl_xor(weight_sum, 32));
  }
  if (!live) return;
  const uint64_t slot_row = l.row_base + (uint64_t(head0 + own) * l.split_count + split) * G + own_row;
  float *out = partials + slot_row * D;
  const auto of_own = [&](uint32_t tile, uint32_t r) {
    const uint32_t group = Page::kPairs ? own >> 1 : own;
    float x = acc[0][tile][r];
#pragma unroll
    for (uint32_t c = 1; c < Page::kGroups; ++c) x = group == c ? acc[c][tile][r] : x;
    return x - bias;
  };
  if constexpr (kInt4) {
    // tile m's row 4g + r: dim 8 (4g + r) + m; at head dimension 64 the rows 8 .. 15 are the pair's second head's
    if (!Page::kPairs || (g >> 1) == (own & 1)) {
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r)
#pragma unroll
        for (uint32_t m4 = 0; m4 < 2; ++m4) {
          f32x4 x;
#pragma unroll
          for (uint32_t i = 0; i < 4; ++i) x[i] = of_own(4 * m4 + i, r);
          *reinterpret_cast<f32x4 *>(out + 8 * (4 * (Page::kPairs ? g & 1 : g) + r) + 4 * m4) = x;
        }
    }
  } else {
#pragma unroll
    for (uint32_t mb = 0; mb < Page::kTiles; ++mb) {
      f32x4 x;
#pragma unroll
      for (uint32_t r = 0; r < 4; ++r) x[r] = of_own(mb, r);
      *reinterpret_cast<f32x4 *>(out + 16 * mb + 4 * g) = x;
    }
  }
  if (g == 0) {
    statistics[slot_row * 2] = row_max;
    statistics[slot_row * 2 + 1] = sum;
  }
}

}  // namespace
}  // namespace kvx

using namespace kvx;

// The lanes of kvx_decode_small_launch: one MFMA block of query rows a head.
bool kvx_decode_small_covers(uint32_t format, uint32_t head_dim, uint32_t group) {
  return group <= 16 && (head_dim == 64 || head_dim == 128);
}

// The split kernel of one-row decode lanes at head dimensions 64 and 128; the lanes' token rows are stored first
// where `fused` brings them.
int kvx_decode_small_launch(uint32_t format, const void *queries, float *partials, float *statistics, const AttendArgs &a,
                            uint32_t max_splits, const FusedAppend *fused, hipStream_t stream) {
  const uint32_t D = a.head_dim, G = a.group, H = a.kv_heads;
  if (!kvx_decode_small_covers(format, D, G)) return KVX_EINVAL;
  // Two heads to a wave for int4 pages of head dimension 64 (1 KiB of keys a head) once there are more waves of one
  // head than a round of 3072: 8 x 8192 tokens (3328 waves) 27.8 -> 25.4 us, 32 x 8192 60.4 -> 48.8, 32 x 700 .. 8192
  // 42.9 -> 39.1; 24 x 2000 (3072) 20.2 -> 20.7, 8 x 2000 (1024) 14.4 -> 16.0.  Other pages gain nothing or little
  // (int8, 32 x 700 .. 8192 tokens 42.8 / 43.8 us, 32 x 8192 62 / 58).
  uint64_t waves = 0;  // of one head each
  for (uint32_t i = 0; i < a.n_lanes; ++i) waves += uint64_t(a.lane[i].split_count) * H;
  const uint32_t P = format == KVX_FMT_INT4 && D == 64 && H % 2 == 0 && 2 * G <= 16 && waves > 3072 ? 2 : 1;
  SmallToken token{};
  if (fused)
    token = {static_cast<const uint16_t *>(fused->keys), static_cast<const uint16_t *>(fused->values), fused->lane_stride,
             fused->stride};
  // One wave to a workgroup, so that a ragged batch fills the chip evenly: in workgroups of four, bf16, 16 x 100 ..
  // 1500 tokens 17.1 -> 19.5 us, 64 x 200 .. 2000 53.5 -> 68, 8 x 15000 49.3 -> 50.1.
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, dim3(max_splits * (H / P), a.n_lanes), dim3(64), 0, stream,
                       static_cast<const uint16_t *>(queries), partials, statistics, a, token);
    const hipError_t e = hipGetLastError();
    return e == hipSuccess ? KVX_OK : hip_fail(e, "decode_small_kernel");
  };
#define KVX_SMALL(FMT) (D == 64 ? launch(decode_small_kernel<FMT, 64, 1, 4>) : launch(decode_small_kernel<FMT, 128, 1, 3>))
  switch (format) {
  case KVX_FMT_INT4: return P == 2 ? launch(decode_small_kernel<KVX_FMT_INT4, 64, 2, 3>) : KVX_SMALL(KVX_FMT_INT4);
  case KVX_FMT_INT8: return KVX_SMALL(KVX_FMT_INT8);
  case KVX_FMT_BF16: return KVX_SMALL(KVX_FMT_BF16);
  default: return KVX_SMALL(KVX_FMT_FP8E4M3);
  }
#undef KVX_SMALL
}
