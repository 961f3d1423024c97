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
#include "kvx_attend_common.h"

namespace kvx {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

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

// Operands are bf16, on e4m3 pages fp16 (each holds the codes exactly).  int8 codes as fp16 would
// need the weights as fp16 too, whose places run out below 2^-14: a weight carries its token's value
// scale, so values of standard deviation 1e-3 would move a row by 1.4e-2.
template <uint32_t FMT>
constexpr bool kHalfOperands = FMT == KVX_FMT_FP8E4M3;

template <uint32_t FMT>
__device__ __forceinline__ f32x16 mfma(u32x4 a, u32x4 b, f32x16 c) {
  if constexpr (kHalfOperands<FMT>)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b),
                                                  c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a),
                                                   __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
}

// ---- bytes of a page to operand elements -----------------------------------------------
// int4 codes become bf16 numbers through e4m3, whose bytes 0 .. 8 are 0 .. 8 / 512 (the subnormals
// and the first normal) and so on up to 15: one conversion takes two of them, and its scale the
// 512.  (As code / 512 the rest went into the key scales, which overflow at keys of 2e37 and more.)
// Keys take the codes themselves, sign and magnitude.  Values take u = code + 8, which is one
// instruction for eight codes; the 8 an element they carry too much are taken off the finished
// row as 8 times the sum of its rounded weights.  (Keys' scores would lose their last bits to
// such a bias where keys have outlier channels.)
constexpr float kNibbleUnit = 512.0f, kNibbleBias = 8.0f;
// Four codes, a byte each (two's complement nibbles), to e4m3 bytes of sign and magnitude.
__device__ __forceinline__ uint32_t signed_nibbles(uint32_t x) {
  const uint32_t low = x & 0x07070707u, negative = (x >> 3) & 0x01010101u;
  return ((low ^ ((negative << 3) - negative)) + negative) | (negative << 7);  // 8 - low = (low ^ 7) + 1
}
template <bool HIGH>
__device__ __forceinline__ uint32_t nibble_pair(uint32_t bytes) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(bytes, kNibbleUnit, HIGH));
}
// Two int8 codes: a small integer's float, cut to its upper half, is exact.
template <bool HIGH>
__device__ __forceinline__ uint32_t int8_pair(uint32_t x) {
  const int lo = __builtin_amdgcn_sbfe(int(x), HIGH ? 16 : 0, 8), hi = __builtin_amdgcn_sbfe(int(x), HIGH ? 24 : 8, 8);
  return __builtin_amdgcn_perm(__float_as_uint(float(hi)), __float_as_uint(float(lo)), 0x07060302u);
}
// Eight one-byte elements in order.
template <uint32_t FMT>
__device__ __forceinline__ u32x4 byte_operand(uint32_t first, uint32_t second) {
  if constexpr (FMT == KVX_FMT_FP8E4M3) {
    return u32x4{fp8_pair<false>(first), fp8_pair<true>(first), fp8_pair<false>(second), fp8_pair<true>(second)};
  } else {
    return u32x4{int8_pair<false>(first), int8_pair<true>(first), int8_pair<false>(second), int8_pair<true>(second)};
  }
}

// ---- a staged page -----------------------------------------------------------------------
// Keys: operand block kb holds dims 16 kb .. 16 kb + 15, a piece of 8 dims (16 bytes) for
// (operand row, half).  Operand row r is token key_token(r), so that the 16 scores a lane of
// half h gets are those of tokens 8h .. 8h+7 and 16 + 8h .. 16 + 8h + 7, in order.
// Values: operand (mb, s) holds 32 dims by tokens 16 s + 8 h .. + 7; the dim of row r of block
// mb is 32 mb + r, for int4,
// whose values lie token by token, 8 dims to a thread, place 32 mb + r holds dim
// 8 (place % (D / 8)) + place / (D / 8).
// Where a piece lies inside its block is a matter of LDS banks: eight consecutive lanes of a
// wave, storing as well as loading, shall touch all of them.
template <uint32_t FMT, uint32_t D>
struct Staged {
  static constexpr uint32_t kSteps = D / 16, kBlocks = D / 32;
  static constexpr uint32_t kKeyBytes = kPage * D * 2, kBytes = 2 * kKeyBytes;
  static constexpr bool kBf16 = FMT == KVX_FMT_BF16, kInt4 = FMT == KVX_FMT_INT4;

  __device__ __forceinline__ static uint32_t key_token(uint32_t r) {  // its own inverse
    return (r & 0x13u) | ((r & 4u) << 1) | ((r & 8u) >> 1);
  }
  __device__ __forceinline__ static uint32_t key_place(uint32_t kb, uint32_t h, uint32_t r) {
    if constexpr (kBf16)  // blocks of 16 rows x 4 pieces, as a direct load lays them down
      return ((kb >> 1) * 2 + (r >> 4)) * 1024 + (4 * (r & 15) + ((2 * (kb & 1) + h) ^ ((r >> 1) & 3))) * 16;
    const uint32_t turn = kInt4 ? 2 * ((kb >> 1) & 3) : 2 * (kb & 3);
    return kb * 1024 + (32 * h + (r ^ turn)) * 16;
  }
  __device__ __forceinline__ static uint32_t value_place(uint32_t mb, uint32_t s, uint32_t h, uint32_t r) {
    if constexpr (kBf16)
      return kKeyBytes + (2 * mb + (r >> 4)) * 1024 + (4 * (r & 15) + ((2 * s + h) ^ ((r >> 1) & 3))) * 16;
    const uint32_t turn = kInt4 ? 0 : 4 * s;
    return kKeyBytes + (2 * mb + s) * 1024 + (32 * h + (r ^ turn)) * 16;
  }
};

typedef __attribute__((address_space(3))) uint8_t SharedByte;
__device__ __forceinline__ u32x4 lds_read(const uint8_t *at) { return *reinterpret_cast<const u32x4 *>(at); }
__device__ __forceinline__ void lds_write(uint8_t *at, u32x4 v) { *reinterpret_cast<u32x4 *>(at) = v; }

// What a thread holds of a page on its way: the raw bytes, not yet expanded, and a token's scale.
// int8 and e4m3: every wave holds a piece of every page, 16 bytes of keys or of values at a time,
// four lanes to 64 bytes of a token's keys.  int4: the first four waves hold the even pages, the
// others the odd ones, so that a page is on its way for the time of two: D / 2 threads 8 tokens
// of 8 dims of values each, as many threads two 16-byte pieces of keys.
template <uint32_t FMT, uint32_t D>
struct PageShare {
  static constexpr bool kInt4 = FMT == KVX_FMT_INT4;
  static constexpr uint32_t kPageThreads = kInt4 ? kThreads / 2 : kThreads;  // that hold a page
  static constexpr uint32_t kTensor = kPage * D / 16;  // 16-byte pieces of a one-byte tensor
  static constexpr uint32_t kPieces = (2 * kTensor + kThreads - 1) / kThreads;
  // int4 keys, piece by piece: 16 bytes of a token, four lanes (two at head dimension 64) a run
  static constexpr uint32_t kRun = D == 64 ? 2 : 4;
  __device__ __forceinline__ static uint32_t nibble_token(uint32_t piece) { return piece / kRun % kPage; }
  __device__ __forceinline__ static uint32_t nibble_chunk(uint32_t piece) {
    return piece % kRun + kRun * (piece / (kRun * kPage));
  }
  u32x4 raw[kInt4 ? 2 : kPieces];
  float scale;
};
template <uint32_t FMT, uint32_t D>
__device__ __forceinline__ void fetch_share(PageShare<FMT, D> &r, const Slab &page, uint32_t tid) {
  using Share = PageShare<FMT, D>;
  if constexpr (FMT == KVX_FMT_INT4) {
    tid %= Share::kPageThreads;
    if (tid < D / 2) {
      const uint8_t *from = page.values + 8 * (tid / (D / 8)) * (D / 2) + 4 * (tid % (D / 8));
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) r.raw[i / 4][i % 4] = load_global<uint32_t>(from + i * (D / 2));
    } else if (tid < D) {
#pragma unroll
      for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t piece = tid - D / 2 + i * (D / 2);
        r.raw[i] = load_global<u32x4>(page.keys + Share::nibble_token(piece) * (D / 2) + 16 * Share::nibble_chunk(piece));
      }
    }
  } else {
#pragma unroll
    for (uint32_t i = 0; i < Share::kPieces; ++i) {
      const uint32_t piece = tid + i * kThreads;
      const uint32_t chunk = piece % 4 + 4 * (piece / (4 * kPage)), token = piece / 4 % kPage;
      const uint8_t *from = piece < Share::kTensor ? page.keys + token * D + 16 * chunk
                                                   : page.values + 16 * (piece - Share::kTensor);
      if (2 * Share::kTensor % kThreads == 0 || piece < 2 * Share::kTensor) r.raw[i] = load_global<u32x4>(from);
    }
  }
  if (tid < 2 * kPage) r.scale = load_global<float>(tid < kPage ? page.key_scales + tid : page.value_scales + (tid - kPage));
}

// The share's elements into the staged copy; `key_unit` goes into the key scales.
template <uint32_t FMT, uint32_t D>
__device__ __forceinline__ void stage_share(uint8_t *copy, float *scales, const PageShare<FMT, D> &r,
                                            uint32_t tid, float key_unit) {
  using Share = PageShare<FMT, D>;
  using Page = Staged<FMT, D>;
  if constexpr (FMT == KVX_FMT_INT4) {
    tid %= Share::kPageThreads;
    if (tid < D / 2) {
      const uint32_t dg = tid % (D / 8), sh = tid / (D / 8);
      uint32_t w[8];
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) w[i] = r.raw[i / 4][i % 4] ^ 0x88888888u;
#pragma unroll
      for (uint32_t b = 0; b < 4; ++b) {  // byte b of every token: dims 8 dg + 2 b (low nibble) and + 1
        const uint32_t select = 0x0c0c0400u + 0x0101u * b;  // that byte of two tokens
        const uint32_t first = __builtin_amdgcn_perm(w[1], w[0], select) | (__builtin_amdgcn_perm(w[3], w[2], select) << 16);
        const uint32_t second = __builtin_amdgcn_perm(w[5], w[4], select) | (__builtin_amdgcn_perm(w[7], w[6], select) << 16);
#pragma unroll
        for (uint32_t n = 0; n < 2; ++n) {
          const uint32_t lo = (n ? first >> 4 : first) & 0x0f0f0f0fu, hi = (n ? second >> 4 : second) & 0x0f0f0f0fu;
          const uint32_t place = (2 * b + n) * (D / 8) + dg;
          lds_write(copy + Page::value_place(place / 32, sh >> 1, sh & 1, place % 32),
                    u32x4{nibble_pair<false>(lo), nibble_pair<true>(lo), nibble_pair<false>(hi), nibble_pair<true>(hi)});
        }
      }
    } else if (tid < D) {
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) {  // dims 0, 2, 4, 6, 1, 3, 5, 7 of each eight
        const uint32_t piece = tid - D / 2 + (i / 4) * (D / 2), x = r.raw[i / 4][i % 4];
        const uint32_t lo = signed_nibbles(x), hi = signed_nibbles(x >> 4);
        lds_write(copy + Page::key_place(2 * Share::nibble_chunk(piece) + (i % 4) / 2, i & 1, Page::key_token(Share::nibble_token(piece))),
                  u32x4{nibble_pair<false>(lo), nibble_pair<true>(lo), nibble_pair<false>(hi), nibble_pair<true>(hi)});
      }
    }
  } else {
#pragma unroll
    for (uint32_t i = 0; i < Share::kPieces; ++i) {
      const uint32_t piece = tid + i * kThreads;
      if (2 * Share::kTensor % kThreads == 0 || piece < 2 * Share::kTensor) {
        const u32x4 first = byte_operand<FMT>(r.raw[i][0], r.raw[i][1]), second = byte_operand<FMT>(r.raw[i][2], r.raw[i][3]);
        const bool keys = piece < Share::kTensor;
        const uint32_t kb = piece % 4 + 4 * (piece / (4 * kPage)), row = Page::key_token(piece / 4 % kPage);
        const uint32_t dim = (piece - Share::kTensor) / 2, s = piece & 1;
        lds_write(copy + (keys ? Page::key_place(kb, 0, row) : Page::value_place(dim / 32, s, 0, dim % 32)), first);
        lds_write(copy + (keys ? Page::key_place(kb, 1, row) : Page::value_place(dim / 32, s, 1, dim % 32)), second);
      }
    }
  }
  if (tid < 2 * kPage) scales[tid] = tid < kPage ? r.scale * key_unit : r.scale;
}

// bf16 pages need no expansion: they go from global memory into the staged copy directly,
// 16 bytes per lane and instruction, 1 KiB of LDS per instruction in lane order.
template <uint32_t D>
__device__ __forceinline__ void direct_page(uint8_t *copy, const Slab &page, uint32_t wave, uint32_t lane) {
  typedef __attribute__((address_space(1))) const void GlobalBytes;
  typedef __attribute__((address_space(3))) void SharedBytes;
  const uint32_t r = lane >> 2, piece = (lane & 3) ^ ((r >> 1) & 3);  // row of the block, 16 bytes of its 64
#pragma unroll
  for (uint32_t i = 0; i < D / 8 / W; ++i) {  // D / 16 instructions of keys, as many of values
    constexpr uint32_t kPerTensor = D / 16;
    const uint32_t block = wave + i * W;
    const uint8_t *from;
    uint32_t to;
    if (block < kPerTensor) {
      const uint32_t token = Staged<KVX_FMT_BF16, D>::key_token(16 * (block & 1) + r);
      from = page.keys + token * (2 * D) + (block >> 1) * 64 + 16 * piece;
      to = block * 1024;
    } else {
      from = page.values + (16 * (block - kPerTensor) + r) * 64 + 16 * piece;
      to = Staged<KVX_FMT_BF16, D>::kKeyBytes + (block - kPerTensor) * 1024;
    }
    __builtin_amdgcn_global_load_lds((GlobalBytes *)(reinterpret_cast<uintptr_t>(from)),
                                     (SharedBytes *)(copy + to), 16, 0, 0);
  }
}

// A thread's number as a value the compiler cannot see through: what is computed from it inside
// the page loop is computed there (a few integer instructions) instead of being kept in
// registers, of which accumulators and queries leave 64.
__device__ __forceinline__ uint32_t opaque(uint32_t x) {
  asm volatile("" : "+v"(x));
  return x;
}
// exp(x), x <= 0: 2^(x log2 e) with the product's rounding error put back, but not that of log2 e:
// within 1.2 ulp (and those of the instruction) to -1, 3 to -10, 5 to -20, 20 to -87, where 2^y
// alone is 1.3, 8, 16 and 63 off.
__device__ __forceinline__ float corrected_exp(float x) {
  const float y = x * kLog2e, e = __builtin_amdgcn_exp2f(y);
  // Of -inf the rounding error is no number, which the median takes for its lower bound: what is 0
  // stays 0, and of an x that is no number e is none either.
  const float rest = __builtin_amdgcn_fmed3f(fmaf(x, kLog2e, -y), -1.0f, 1.0f);
  return fmaf(e, rest * 0.693147180559945309f, e);
}
__device__ __forceinline__ float other_half(float x) { return __shfl_xor(x, 32); }
__device__ __forceinline__ float halves_max(float x) {
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
  return fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
}

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
  // The difference first, so that the heaviest tokens' weights carry the scores' own rounding and
  // no more; at head dimensions 64 and 128 a row is short enough that the error of a product
  // with log2 e in the lighter ones shows as well (against the oracle's expf).
  const auto weight_of = [](float difference) {
    return D == 256 ? __builtin_amdgcn_exp2f(difference * kLog2e) : corrected_exp(difference);
  };

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
    if constexpr (kInt4) {
      x = u32x4{__builtin_amdgcn_perm(x[1], x[0], 0x05040100u), __builtin_amdgcn_perm(x[3], x[2], 0x05040100u),
                __builtin_amdgcn_perm(x[1], x[0], 0x07060302u), __builtin_amdgcn_perm(x[3], x[2], 0x07060302u)};
    } else if constexpr (kHalfOperands<FMT>) {
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        const f16x2 pair = {_Float16(__uint_as_float(x[i] << 16)), _Float16(__uint_as_float(x[i] & 0xffff0000u))};
        x[i] = __builtin_bit_cast(uint32_t, pair);
      }
    }
    if (kb < kQueryRegs) q[kb < kQueryRegs ? kb : 0] = x;
    else query_lds[kb - kQueryRegs][wave][lane] = x;  // (the wave's own: no barrier)
  }
  f32x16 acc[kBlocks];
  float row_max = -INFINITY, row_sum = 0.0f, weight_sum = 0.0f;
#pragma unroll
  for (uint32_t mb = 0; mb < kBlocks; ++mb)
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) acc[mb][i] = 0.0f;

  const uint64_t *const entries = table + begin;
  const uint32_t count = end - begin, last_slot = count - 1;
  const auto slab_at = [&](uint32_t slot) {
    return slab_of(FMT, H, D, a.kv, head, scalar_entry(entries, min(slot, last_slot)));
  };
  PageShare<FMT, D> raw;
  // What goes into the key scales: the score scale, but for head dimension 128, whose default is no
  // power of two.
  const float key_unit = D == 128 ? 1.0f : score_scale;

  // A staged page against the wave's rows.
  const auto attend_page = [&](const uint8_t *copy, const float *scales, uint32_t page) __attribute__((always_inline)) {
    const uint32_t at = opaque(lane), n = at & 31u, h = at >> 5;
    const auto key_at = [&](uint32_t kb) { return lds_read(copy + Page::key_place(kb, h, n)); };
    const auto value_at = [&](uint32_t i) { return lds_read(copy + Page::value_place(i >> 1, i & 1, h, n)); };
    constexpr uint32_t kAhead = kQuant ? 2 : 3;
    u32x4 operand[kAhead];
    f32x16 s;
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) s[i] = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) operand[i] = key_at(i);
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t kb = 0; kb < kSteps; ++kb) {
      const u32x4 q_block = kb < kQueryRegs ? q[kb < kQueryRegs ? kb : 0] : query_lds[kb - kQueryRegs][wave][at];
      s = mfma<FMT>(operand[kb % kAhead], q_block, s);
      if (kb + kAhead < kSteps) operand[kb % kAhead] = key_at(kb + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
    // scores: lane element 8 t + j is token 16 t + 8 h + j
    if constexpr (kQuant) {
#pragma unroll
      for (uint32_t i = 0; i < 16; i += 4) {
        const f32x4 ks = *reinterpret_cast<const f32x4 *>(scales + 16 * (i >> 3) + 8 * h + (i & 7));
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) s[i + j] = D == 128 ? s[i + j] * ks[j] * score_scale : s[i + j] * ks[j];
      }
      __builtin_amdgcn_sched_barrier(0);
    } else {
#pragma unroll
      for (uint32_t i = 0; i < 16; ++i) s[i] *= score_scale;
    }
    const uint32_t first_token = page * kPage;
    const bool masked = first_token + kPage > whole_to;
    uint32_t unseen = 0;  // (of a masked page) bit i: score i
    if (masked) {
      const Column own = column_of(n);  // found again on the few such pages rather than kept
      // (columns without a row see everything, and count for nothing)
      const uint32_t to = own.live ? committed + own.row + 1 : UINT32_MAX;
#pragma unroll
      for (uint32_t i = 0; i < 16; ++i) {
        const uint32_t token = first_token + 16 * (i >> 3) + 8 * h + (i & 7);
        if (token >= to) s[i] = -INFINITY;
        if constexpr (kQuant) unseen |= token >= to ? 1u << i : 0u;
      }
    }
    float local_max = fmaxf(s[0], s[1]);
#pragma unroll
    for (uint32_t i = 2; i < 16; i += 2) local_max = fmaxf(fmaxf(local_max, s[i]), s[i + 1]);
    const float next_max = fmaxf(row_max, halves_max(local_max));
    const bool grows = next_max != row_max;
    const float rescale = grows ? weight_of(row_max - next_max) : 1.0f;
    // A row that has seen nothing yet measures from 0: -inf - -inf is no number.
    const float reference = next_max == -INFINITY ? 0.0f : next_max;
    float page_sum = 0.0f;
    u32x4 weights[2];
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t i = 0; i < 16; i += 4) {
      float p[4];
#pragma unroll
      for (uint32_t j = 0; j < 4; ++j) {
        p[j] = weight_of(s[i + j] - reference);
        page_sum += p[j];
      }
      if constexpr (kQuant) {
        const f32x4 vs = *reinterpret_cast<const f32x4 *>(scales + kPage + 16 * (i >> 3) + 8 * h + (i & 7));
#pragma unroll
        for (uint32_t j = 0; j < 4; ++j) p[j] *= vs[j];
      }
#pragma unroll
      for (uint32_t j = 0; j < 4; j += 2) {
        uint32_t bits;
        if constexpr (FMT == KVX_FMT_FP8E4M3) {
          const f16x2 pair = {_Float16(p[j]), _Float16(p[j + 1])};
          bits = __builtin_bit_cast(uint32_t, pair);
        } else {
          const f32x2 wide = {p[j], p[j + 1]};
          bits = __builtin_bit_cast(uint32_t, __builtin_convertvector(wide, bf16x2));
        }
        weights[i >> 3][(i & 7) / 2 + j / 2] = bits;
      }
    }
    // An unseen token's weight is 0 whatever its scale: what an earlier sequence left in the page may be
    // infinite, or no number.  (On the rounded weights, all at once: tests between the products above
    // took 10 % of a one-wave-a-SIMD chunk's time.)
    if constexpr (kQuant)
      if (masked) {
#pragma unroll
        for (uint32_t i = 0; i < 16; i += 2) {
          const uint32_t first = __builtin_amdgcn_sbfe(unseen, i, 1), second = __builtin_amdgcn_sbfe(unseen, i + 1, 1);
          weights[i >> 3][(i & 7) / 2] &= ~((first & 0xffffu) | (second & 0xffff0000u));
        }
      }
    row_sum = fmaf(row_sum, rescale, page_sum);
    row_max = next_max;
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (uint32_t i = 0; i < kAhead; ++i) operand[i] = value_at(i);
    __builtin_amdgcn_sched_barrier(0);
    if (__builtin_amdgcn_ballot_w64(grows)) {
      if constexpr (kInt4) weight_sum *= rescale;
#pragma unroll
      for (uint32_t mb = 0; mb < kBlocks; ++mb) acc[mb] *= rescale;
    }
    if constexpr (kInt4) {
      const bf16x2 ones = {__bf16(1.0f), __bf16(1.0f)};
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) {
        const uint32_t pair = weights[i >> 2][i & 3];  // (a copy: bit_cast of a vector's element takes element 0)
        weight_sum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), ones, weight_sum, false);
      }
    }
#pragma unroll
    for (uint32_t i = 0; i < 2 * kBlocks; ++i) {
      acc[i >> 1] = mfma<FMT>(operand[i % kAhead], weights[i & 1], acc[i >> 1]);
      if (i + kAhead < 2 * kBlocks) operand[i % kAhead] = value_at(i + kAhead);
      __builtin_amdgcn_sched_barrier(0);
    }
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
    direct_page<D>(staged[0], slab_at(0), wave, lane);
    direct_page<D>(staged[1], slab_at(1), wave, lane);
  } else if constexpr (kInt4) {
    fetch_share<FMT, D>(raw, slab_at(mine), tid);
    stage_share<FMT, D>(staged[mine], scale_lds[mine], raw, tid, key_unit);
    fetch_share<FMT, D>(raw, slab_at(2 + mine), tid);
  } else {
    for (uint32_t slot = 0; slot < 2; ++slot) {
      fetch_share<FMT, D>(raw, slab_at(slot), tid);
      stage_share<FMT, D>(staged[slot], scale_lds[slot], raw, tid, key_unit);
    }
    fetch_share<FMT, D>(raw, slab_at(2), tid);
  }
  barrier();
  for (uint32_t slot = 0; slot < count; ++slot) {
    const uint32_t now = slot & 3, next = (slot + 2) & 3;
    if constexpr (!kQuant) {
      direct_page<D>(staged[next], slab_at(slot + 2), wave, opaque(lane));
    } else if (!kInt4 || (slot & 1) == mine) {
      stage_share<FMT, D>(staged[next], scale_lds[next], raw, opaque(tid), key_unit);
      fetch_share<FMT, D>(raw, slab_at(slot + (kInt4 ? 4 : 3)), opaque(tid));
    }
    if (slot - wave_first < wave_pages) attend_page(staged[now], scale_lds[now], begin + slot);
    if (slot & 1) barrier();
  }
  if constexpr (!kQuant) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS outlives the wave

  // A lane's element i of block mb is row 8 (i / 4) + 4 h + i % 4 of the block; four dims that
  // follow one another, at `dim`.
  const uint32_t at = opaque(lane), half = at >> 5;
  const float sum = row_sum + other_half(row_sum);
  const float bias = kInt4 ? kNibbleBias * (weight_sum + other_half(weight_sum)) : 0.0f;
  constexpr uint32_t kQuads = D / 8;
  const auto quad = [&](uint32_t k, uint32_t &dim) {
    f32x4 v;
    if constexpr (kInt4) {  // dims 8 r .. 8 r + 7 are places r, r + D / 8, ..
      const uint32_t r = (k / 2) % 4 + 8 * (k / 8), first = 4 * (k & 1);  // (r + 4 half)
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) {
        const uint32_t place = r + (first + i) * (D / 8), in_block = place % 32;
        v[i] = acc[place / 32][(in_block & 3) + 4 * (in_block >> 3)] - bias;
      }
      dim = 8 * (r + 4 * half) + first;
    } else {
#pragma unroll
      for (uint32_t i = 0; i < 4; ++i) v[i] = acc[k / 4][4 * (k % 4) + i];
      dim = 8 * k + 4 * half;
    }
    return v;
  };
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
    // x / sum by the reciprocal, with the quotient's error put back: the divider's own result
    // but for its last bit, in a third of its instructions.
    const bool some = sum > 0.0f;  // a sum that is no number leaves no row, as in the merge
    const float reciprocal = some ? __fdiv_rn(1.0f, sum) : 0.0f;
    const auto divided = [&](float x) {
      if (!some) return 0.0f;
      const float quotient = x * reciprocal;
      const float better = fmaf(fmaf(-quotient, sum, x), reciprocal, quotient);
      return fabsf(quotient) < INFINITY ? better : quotient;  // (an infinite quotient has no error)
    };
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
  if (half == 0) *reinterpret_cast<f32x2 *>(statistics + slot_row * 2) = f32x2{row_max, sum};
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
