// Pages in LDS as finished 16-bit MFMA operands, shared by the waves of a workgroup, and a wave's
// 32 fused rows against such a page: chunked prefill (kvx_prefill.hip) and verify lanes of more
// than 32 fused rows (kvx_verify.hip).
#pragma once

#include "kvx_attend_common.h"

namespace kvx {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));

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

// Eight bf16 query elements of a lane as the operand that meets the staged keys: int4 in the
// order their dims are staged, e4m3 as fp16.
template <uint32_t FMT>
__device__ __forceinline__ u32x4 query_operand(u32x4 x) {
  if constexpr (FMT == KVX_FMT_INT4) {
    x = u32x4{__builtin_amdgcn_perm(x[1], x[0], 0x05040100u), __builtin_amdgcn_perm(x[3], x[2], 0x05040100u),
              __builtin_amdgcn_perm(x[1], x[0], 0x07060302u), __builtin_amdgcn_perm(x[3], x[2], 0x07060302u)};
  } else if constexpr (kHalfOperands<FMT>) {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      const f16x2 pair = {_Float16(__uint_as_float(x[i] << 16)), _Float16(__uint_as_float(x[i] & 0xffff0000u))};
      x[i] = __builtin_bit_cast(uint32_t, pair);
    }
  }
  return x;
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
// four lanes to 64 bytes of a token's keys.  int4, eight waves: the first four hold the even pages, the
// others the odd ones, so that a page is on its way for the time of two: D / 2 threads 8 tokens
// of 8 dims of values each, as many threads two 16-byte pieces of keys.
template <uint32_t FMT, uint32_t D, uint32_t W>
struct PageShare {
  static constexpr bool kInt4 = FMT == KVX_FMT_INT4;
  static constexpr uint32_t kThreads = 64 * W;
  static constexpr uint32_t kPageThreads = kInt4 && W == 8 ? kThreads / 2 : kThreads;  // that hold a page
  static_assert(!kInt4 || kPageThreads >= D, "int4: a page is held by D threads");
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
// REUSED: see load_streaming.
template <bool REUSED = true, uint32_t FMT, uint32_t D, uint32_t W>
__device__ __forceinline__ void fetch_share(PageShare<FMT, D, W> &r, const Slab &page, uint32_t tid) {
  using Share = PageShare<FMT, D, W>;
  constexpr uint32_t kThreads = Share::kThreads;
  if constexpr (FMT == KVX_FMT_INT4) {
    tid %= Share::kPageThreads;
    if (tid < D / 2) {
      const uint8_t *from = page.values + 8 * (tid / (D / 8)) * (D / 2) + 4 * (tid % (D / 8));
#pragma unroll
      for (uint32_t i = 0; i < 8; ++i) r.raw[i / 4][i % 4] = load_streaming<uint32_t, REUSED>(from + i * (D / 2));
    } else if (tid < D) {
#pragma unroll
      for (uint32_t i = 0; i < 2; ++i) {
        const uint32_t piece = tid - D / 2 + i * (D / 2);
        r.raw[i] = load_streaming<u32x4, REUSED>(page.keys + Share::nibble_token(piece) * (D / 2) + 16 * Share::nibble_chunk(piece));
      }
    }
  } else {
#pragma unroll
    for (uint32_t i = 0; i < Share::kPieces; ++i) {
      const uint32_t piece = tid + i * kThreads;
      const uint32_t chunk = piece % 4 + 4 * (piece / (4 * kPage)), token = piece / 4 % kPage;
      const uint8_t *from = piece < Share::kTensor ? page.keys + token * D + 16 * chunk
                                                   : page.values + 16 * (piece - Share::kTensor);
      if (2 * Share::kTensor % kThreads == 0 || piece < 2 * Share::kTensor) r.raw[i] = load_streaming<u32x4, REUSED>(from);
    }
  }
  if (tid < 2 * kPage) r.scale = load_global<float>(tid < kPage ? page.key_scales + tid : page.value_scales + (tid - kPage));
}

// The share's elements into the staged copy; `key_unit` goes into the key scales.
template <uint32_t FMT, uint32_t D, uint32_t W>
__device__ __forceinline__ void stage_share(uint8_t *copy, float *scales, const PageShare<FMT, D, W> &r,
                                            uint32_t tid, float key_unit) {
  using Share = PageShare<FMT, D, W>;
  using Page = Staged<FMT, D>;
  constexpr uint32_t kThreads = Share::kThreads;
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
template <uint32_t D, uint32_t W, bool REUSED = true>
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
                                     (SharedBytes *)(copy + to), 16, 0, REUSED ? 0 : 2);  // 2: non-temporal
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
// The difference first, so that the heaviest tokens' weights carry the scores' own rounding and
// no more; at head dimensions 64 and 128 a row is short enough that the error of a product
// with log2 e in the lighter ones shows as well (against the oracle's expf).
template <uint32_t D>
__device__ __forceinline__ float row_weight(float difference) {
  return D == 256 ? __builtin_amdgcn_exp2f(difference * kLog2e) : corrected_exp(difference);
}

// What a wave keeps of its 32 rows; a lane's share of row lane % 32.
template <uint32_t D>
struct RowState {
  f32x16 acc[D / 32];
  float row_max, row_sum;
  float weight_sum;  // int4: of the rounded weights
};

// Scores of a staged page's keys against the wave's 32 rows (raw products).  q: the queries of the
// first steps in registers, a lane's share of its row; late_query(step, lane): those of the others.
// Operands come out of LDS AHEAD reads before the MFMAs that take them.
template <uint32_t FMT, uint32_t D, uint32_t AHEAD, uint32_t QUERIES, class LateQuery>
__device__ __forceinline__ void staged_scores(f32x16 &s, const uint8_t *copy, const u32x4 (&q)[QUERIES],
                                              LateQuery late_query, uint32_t lane) {
  using Page = Staged<FMT, D>;
  constexpr uint32_t kSteps = Page::kSteps;
  const uint32_t n = lane & 31u, h = lane >> 5;
  u32x4 operand[AHEAD], late[AHEAD];
#pragma unroll
  for (uint32_t i = 0; i < 16; ++i) s[i] = 0.0f;
  const auto read_step = [&](uint32_t kb) {
    operand[kb % AHEAD] = lds_read(copy + Page::key_place(kb, h, n));
    if (kb >= QUERIES) late[kb % AHEAD] = late_query(kb - QUERIES, lane);
  };
#pragma unroll
  for (uint32_t i = 0; i < AHEAD; ++i) read_step(i);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (uint32_t kb = 0; kb < kSteps; ++kb) {
    s = mfma<FMT>(operand[kb % AHEAD], kb < QUERIES ? q[kb < QUERIES ? kb : 0] : late[kb % AHEAD], s);
    if (kb + AHEAD < kSteps) read_step(kb + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// The page's softmax: scores to rounded weights, the rows' sums and maxima, the accumulators rescaled
// where a row's maximum grew.  masked: some row does not see every token; sight_of(row) then tells
// which places of the page it does not.
template <uint32_t FMT, uint32_t D, class SightOf>
__device__ __forceinline__ void staged_weights(u32x4 (&weights)[2], f32x16 &s, const float *scales, RowState<D> &st,
                                               float score_scale, uint32_t lane, bool masked, SightOf sight_of) {
  constexpr bool kQuant = FMT != KVX_FMT_BF16, kInt4 = FMT == KVX_FMT_INT4;
  const uint32_t n = lane & 31u, h = lane >> 5;
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
  uint32_t unseen = 0;  // (of a masked page) bit i: score i
  if (masked) {
    const auto hides = sight_of(n);
#pragma unroll
    for (uint32_t i = 0; i < 16; ++i) {
      const bool hidden = hides(16 * (i >> 3) + 8 * h + (i & 7));
      if (hidden) s[i] = -INFINITY;
      if constexpr (kQuant) unseen |= hidden ? 1u << i : 0u;
    }
  }
  float local_max = fmaxf(s[0], s[1]);
#pragma unroll
  for (uint32_t i = 2; i < 16; i += 2) local_max = fmaxf(fmaxf(local_max, s[i]), s[i + 1]);
  const float next_max = fmaxf(st.row_max, halves_max(local_max));
  const bool grows = next_max != st.row_max;
  const float rescale = grows ? row_weight<D>(st.row_max - next_max) : 1.0f;
  // A row that has seen nothing yet measures from 0: -inf - -inf is no number.
  const float reference = next_max == -INFINITY ? 0.0f : next_max;
  float page_sum = 0.0f;
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (uint32_t i = 0; i < 16; i += 4) {
    float p[4];
#pragma unroll
    for (uint32_t j = 0; j < 4; ++j) {
      p[j] = row_weight<D>(s[i + j] - reference);
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
  st.row_sum = fmaf(st.row_sum, rescale, page_sum);
  st.row_max = next_max;
  if (__builtin_amdgcn_ballot_w64(grows)) {
    if constexpr (kInt4) st.weight_sum *= rescale;
#pragma unroll
    for (uint32_t mb = 0; mb < D / 32; ++mb) st.acc[mb] *= rescale;
  }
  if constexpr (kInt4) {
    const bf16x2 ones = {__bf16(1.0f), __bf16(1.0f)};
#pragma unroll
    for (uint32_t i = 0; i < 8; ++i) {
      const uint32_t pair = weights[i >> 2][i & 3];  // (a copy: bit_cast of a vector's element takes element 0)
      st.weight_sum = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, pair), ones, st.weight_sum, false);
    }
  }
}

// The page's values times the weights onto the accumulators.
template <uint32_t FMT, uint32_t D, uint32_t AHEAD>
__device__ __forceinline__ void staged_products(RowState<D> &st, const uint8_t *copy, const u32x4 (&weights)[2],
                                                uint32_t lane) {
  using Page = Staged<FMT, D>;
  constexpr uint32_t kOperands = 2 * Page::kBlocks;
  const uint32_t n = lane & 31u, h = lane >> 5;
  const auto value_at = [&](uint32_t i) { return lds_read(copy + Page::value_place(i >> 1, i & 1, h, n)); };
  u32x4 operand[AHEAD];
#pragma unroll
  for (uint32_t i = 0; i < AHEAD; ++i) operand[i] = value_at(i);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (uint32_t i = 0; i < kOperands; ++i) {
    st.acc[i >> 1] = mfma<FMT>(operand[i % AHEAD], weights[i & 1], st.acc[i >> 1]);
    if (i + AHEAD < kOperands) operand[i % AHEAD] = value_at(i + AHEAD);
    __builtin_amdgcn_sched_barrier(0);
  }
}

// A lane's element i of block mb is row 8 (i / 4) + 4 half + i % 4 of the block; four dims that
// follow one another (quad k of D / 8), from `dim` on.  bias: what int4 values carry too much.
template <uint32_t FMT, uint32_t D>
__device__ __forceinline__ f32x4 row_quad(const RowState<D> &st, uint32_t k, uint32_t half, float bias, uint32_t &dim) {
  f32x4 v;
  if constexpr (FMT == KVX_FMT_INT4) {  // dims 8 r .. 8 r + 7 are places r, r + D / 8, ..
    const uint32_t r = (k / 2) % 4 + 8 * (k / 8), first = 4 * (k & 1);  // (r + 4 half)
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) {
      const uint32_t place = r + (first + i) * (D / 8), in_block = place % 32;
      v[i] = st.acc[place / 32][(in_block & 3) + 4 * (in_block >> 3)] - bias;
    }
    dim = 8 * (r + 4 * half) + first;
  } else {
#pragma unroll
    for (uint32_t i = 0; i < 4; ++i) v[i] = st.acc[k / 4][4 * (k % 4) + i];
    dim = 8 * k + 4 * half;
  }
  return v;
}

// x / sum by the reciprocal, with the quotient's error put back: the divider's own result
// but for its last bit, in a third of its instructions.
struct RowQuotient {
  float sum, reciprocal;
  bool some;
  __device__ __forceinline__ explicit RowQuotient(float of)
      : sum(of), some(of > 0.0f) {  // a sum that is no number leaves no row, as in the merge
    reciprocal = some ? __fdiv_rn(1.0f, sum) : 0.0f;
  }
  __device__ __forceinline__ float operator()(float x) const {
    if (!some) return 0.0f;
    const float quotient = x * reciprocal;
    const float better = fmaf(fmaf(-quotient, sum, x), reciprocal, quotient);
    return fabsf(quotient) < INFINITY ? better : quotient;  // (an infinite quotient has no error)
  }
};

}  // namespace
}  // namespace kvx
