// Paged attention for many query rows per KV head (more than 16: prompt chunks, wide speculative verifies, the
// rows of a shared prefix) on the matrix cores, over a BF16, FP8 (e4m3fn) or INT8 paged cache.
//
// A tile is BM consecutive rows (row r = query r / G, head h G + r % G) of one (sequence, KV head); it walks the
// chunks of kRowsChunk tokens that its last row sees (causal: later tokens are never read for it). The tiles' chunks
// are laid end to end on a line that the workgroups cut into equal ranges, as in the decode kernels (decode_common.h):
// a tile held by one workgroup is written directly, the others go through partials that the last arriver combines or,
// where they are large, a second launch (rows_combine_kernel).
//
// One workgroup = NW waves = WM row blocks of 32 rows x WN token groups. Per chunk:
//  * all waves load the chunk's K and V codes (whole 16-token groups, one page lookup each), decode them once to
//    16 bits and store them to LDS: K as [token][channel], V transposed as [channel][token];
//  * every wave computes its 32 rows over its kRowsChunk / WN tokens with 32x32x16 MFMAs: S^T = K Q^T (A = K from
//    LDS, B = Q^T from registers), online softmax, O^T += V^T P^T. With n = lane % 32 and hf = lane / 32 a lane
//    holds row n's scores of tokens 8 a + 4 hf + b (a, b < 4) of each 32; the second product's contraction index
//    is mapped to exactly those tokens, so P^T is built in registers. V^T holds every 16 tokens in that order.
// The codes are exact in 16 bits (FP8 and INT8 in bf16 and f16, BF16 as it is). The weights are float32 numbers
// fed to the MFMAs as the vector kernel takes them: over BF16 and INT8 values whole, as three bf16 parts (24 bits, the
// range of float32: a per-token INT8 scale rides in them), over FP8 values as f16 plus f16 remainder (22 bits); an f16 q
// over a BF16 cache as bf16 plus bf16 remainder (exact). (INT8 in two f16 parts is faster, 512 new over 8192 cached tokens,
// 32 heads 154 us against 172, but drops bits that the vector kernel keeps, and scales past 2^64.)
//
// What bounds it: with many chunks the matrix cores (FP8: three products where two would do, for the weights' second
// part) and the vector units, mostly in turn (256-row tiles, 2048 queries x 16 heads over 4096 tokens: busy for 42 % and
// 51 % of the cycles); with few the first loads and the partials. Kernel times against the vector kernel's 4-row groups,
// which decode every chunk rows / 4 times (8 KV heads, us): FP8 prompt chunks of 2048 over 2048 cached tokens, 16 heads
// 1885 -> 129 (114 and 15 in the combine's launch); verifies of 5 queries, 32 heads, 16 sequences of 1024..3072 tokens
// 113 -> 34.
//
// LDS layouts (16-byte units; both spread the 8 lanes that one LDS cycle serves over all banks):
//  * K: token row of 16 units, unit u at u ^ (token % 8) ^ (u / 8). Operand reads take one unit of 8 consecutive
//    tokens; stores take two units of each of 8 lanes of a row.
//  * V: 64-token blocks of [channel][8 units], unit u of channel c at u ^ ((c + c / 8) % 8); unit 2 s + hf holds
//    tokens 16 s + 4 hf + 0..3 and 16 s + 8 + 4 hf + 0..3. Reads take one unit of 8 consecutive channels; an 8-byte
//    store takes one half unit of channels c, c + 8, ...: lanes of the upper 64 channels hold the other half.
//
// A token that a row does not see must add nothing to it, and the split weights must not turn an infinity into NaN, but
// the MFMAs multiply every value by every weight and by every part of it, zeros included. So values that are not finite
// (and per-token value scales that are not) are replaced by zeros on their way into LDS, and the rows that see them get
// them added one by one (rows_add_nonfinite), which finite data never pays for; the look at the values, one dot product
// with zero per two of them, costs BF16 caches 1 to 3 % (2048 + 2048 tokens, 16 heads 134 -> 137 us, 512 + 8192, 32 heads
// 169 -> 171, with an f16 q 191 -> 196) and the others nothing that shows (FP8 111 -> 110).
#pragma once

#include <type_traits>

#include "decode_common.h"

namespace bpt {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));

template <int KV_, int SK_, bool PU_, bool QF16_, int WM_, int NW_, int NBUF_>
struct RowsCfg {
  static constexpr int KV = KV_, SK = SK_, WM = WM_, NW = NW_, NBUF = NBUF_;
  static constexpr bool PU = PU_;
  static constexpr int NT = NW * 64;
  static constexpr int WN = NW / WM;   // token groups
  static constexpr int BM = 32 * WM;   // rows per tile
  static constexpr int CT = kRowsChunk;
  static constexpr int TW = CT / WN;               // tokens per wave and chunk
  static constexpr bool kBf16 = KV == kKvBf16;
  static constexpr bool kF16K = QF16_ && !kBf16;   // K and q operands in f16 (an f16 q over codes), else bf16
  static constexpr bool kQSplit = QF16_ && kBf16;  // an f16 q as two bf16 parts
  static constexpr bool kQF16 = QF16_;
  static constexpr bool kVF16 = KV == kKvFp8;      // values and weights in f16 (weights in two parts), else bf16 (three)
  // Whether values or value scales can be infinite or NaN (INT8 codes cannot).
  static constexpr bool kNonfinite = KV != kKvInt8 || SK == kScaleTokenHead;
  static constexpr bool kVBound = kVF16 && SK == kScaleTokenHead;  // the reference point tracks vscale_bound
  static constexpr int kQOps = kQSplit ? 16 : 8;
  static constexpr int kGroups = CT / 16 / NW;     // 16-token groups a wave loads per chunk
  static constexpr int kKLoads = kBf16 ? 4 : 2;    // 16-byte K loads per group
  static constexpr int kBuf = CT * 2 * kHeadDim * 2;  // bytes of one chunk in LDS: K, then V
  static constexpr int kMerge = (WN - 1) * WM * 64 * 66 * 4;
  static constexpr int kOut = BM * (kHeadDim + 4) * 4 + BM * 4;
  static constexpr int kSmem = NBUF * kBuf > kMerge ? (NBUF * kBuf > kOut ? NBUF * kBuf : kOut)
                                                    : (kMerge > kOut ? kMerge : kOut);
  // Whether pieces can be combined in the launch: two of the largest tiles' already call for a second one (rows_two_pass).
  static constexpr bool kInLaunch = 2 * BM * kHeadDim * 4 < kRowsTwoPassBytes;
  static_assert(NW % WM == 0 && TW % 32 == 0 && (CT / 16) % NW == 0, "tile shape");
};

// One chunk's codes of one thread, in flight.
template <typename C>
struct RowsStage {
  U4 k[C::kGroups][C::kKLoads];
  typename std::conditional<C::kBf16, U4, u32x2>::type v[C::kGroups][4];  // 8 channels of 4 tokens
  float sc;
  int page[C::kGroups];  // PU: the next chunk's page of each group
  int sc_page;           // per-token scales: the page of this thread's token of the next chunk
};

// ---- conversions ------------------------------------------------------------------------------------------

__device__ __forceinline__ u32x4 rows_fp8_to_bf16(uint32_t w0, uint32_t w1) {
  return u32x4{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w0, 1.0f, true)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w1, 1.0f, true))};
}
__device__ __forceinline__ u32x2 rows_fp8_to_f16(uint32_t w) {
  return u32x2{__builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, false)),
               __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(w, 1.0f, true))};
}
// Four int8 codes -> f16: the bits 0x6400 | (b ^ 0x80) are the f16 value 1152 + b.
__device__ __forceinline__ u32x2 rows_int8_to_f16(uint32_t w) {
  typedef _Float16 f16x2v __attribute__((ext_vector_type(2)));
  const f16x2v bias = {(_Float16)1152.0f, (_Float16)1152.0f};
  const f16x2v a = __builtin_bit_cast(f16x2v, __builtin_amdgcn_perm(0u, w, 0x0c010c00u) ^ 0x64806480u) - bias;
  const f16x2v b = __builtin_bit_cast(f16x2v, __builtin_amdgcn_perm(0u, w, 0x0c030c02u) ^ 0x64806480u) - bias;
  return u32x2{__builtin_bit_cast(uint32_t, a), __builtin_bit_cast(uint32_t, b)};
}
// Four int8 codes -> bf16, through float32 (exact: 8 significant bits).
__device__ __forceinline__ u32x2 rows_int8_to_bf16(uint32_t w) {
  float f[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) f[i] = (float)(int8_t)((w >> (8 * i)) & 0xffu);
  return u32x2{__builtin_amdgcn_perm(__float_as_uint(f[1]), __float_as_uint(f[0]), 0x07060302u),
               __builtin_amdgcn_perm(__float_as_uint(f[3]), __float_as_uint(f[2]), 0x07060302u)};
}
// Eight codes (two dwords) as the K operand's 16-bit type.
template <typename C>
__device__ __forceinline__ u32x4 rows_k_cvt(uint32_t w0, uint32_t w1) {
  if constexpr (C::KV == kKvFp8 && !C::kF16K) {
    return rows_fp8_to_bf16(w0, w1);
  } else {
    const u32x2 a = C::KV == kKvFp8 ? rows_fp8_to_f16(w0) : C::kF16K ? rows_int8_to_f16(w0) : rows_int8_to_bf16(w0);
    const u32x2 b = C::KV == kKvFp8 ? rows_fp8_to_f16(w1) : C::kF16K ? rows_int8_to_f16(w1) : rows_int8_to_bf16(w1);
    return u32x4{a.x, a.y, b.x, b.y};
  }
}
// 4 x 4 byte transpose: w[i] byte j -> out[j] byte i.
__device__ __forceinline__ void rows_transpose4(uint32_t w0, uint32_t w1, uint32_t w2, uint32_t w3, uint32_t* o) {
  const uint32_t t0 = __builtin_amdgcn_perm(w1, w0, 0x05010400u);
  const uint32_t t1 = __builtin_amdgcn_perm(w3, w2, 0x05010400u);
  const uint32_t t2 = __builtin_amdgcn_perm(w1, w0, 0x07030602u);
  const uint32_t t3 = __builtin_amdgcn_perm(w3, w2, 0x07030602u);
  o[0] = __builtin_amdgcn_perm(t1, t0, 0x05040100u);
  o[1] = __builtin_amdgcn_perm(t1, t0, 0x07060302u);
  o[2] = __builtin_amdgcn_perm(t3, t2, 0x05040100u);
  o[3] = __builtin_amdgcn_perm(t3, t2, 0x07060302u);
}

// ---- a chunk's way into LDS ---------------------------------------------------------------------------------

__device__ __forceinline__ int rows_clamp_page(const DecodeParams& p, int e) {
  return e < 0 ? 0 : (e >= p.num_blocks ? p.num_blocks - 1 : e);
}

// First token (of the chunk) of the wave's u-th 16-token group, and the token group a lane's V loads take.
template <typename C>
__device__ __forceinline__ int rows_group(int u, int wave) { return 16 * (u * C::NW + wave); }
__device__ __forceinline__ int rows_v_quad(int lane) { return (lane >> 4) ^ (((lane >> 3) & 1) << 1); }

// The page ids chunk kk's loads need: one per group (16 tokens lie in one page when page_size >= 16; smaller pages
// are looked up per token when the loads are issued), and one per thread for the per-token scales.
template <typename C>
__device__ __forceinline__ void rows_fetch_pages(const DecodeParams& p, int b, int kk, int len, int wave, int tid,
                                                 RowsStage<C>& s) {
  const int32_t* table = (const int32_t*)p.table;
  const int T0 = kk * C::CT;
  if constexpr (C::PU) {
#pragma unroll
    for (int u = 0; u < C::kGroups; ++u)
      s.page[u] = load_uniform(table + table_word(p, b, min(T0 + rows_group<C>(u, wave), len - 1) >> p.logP));
  }
  if constexpr (C::SK == kScaleTokenHead) {
    if (tid < 2 * C::CT) s.sc_page = table[table_word(p, b, min(T0 + (tid & (C::CT - 1)), len - 1) >> p.logP)];
  }
}

// Issue chunk kk's loads. Tokens at or past len read the sequence's last token instead (valid memory; masked).
template <typename C>
__device__ __forceinline__ void rows_issue(const DecodeParams& p, int b, int h, int kk, int len, int wave, int lane,
                                           int tid, RowsStage<C>& s) {
  constexpr int KR = C::kBf16 ? 4 : 8;         // tokens per K load instruction
  constexpr int VB = C::kBf16 ? 16 : 8;        // bytes of 8 channels
  const int T0 = kk * C::CT;
  const int kr = C::kBf16 ? lane >> 4 : lane >> 3;
  const int kofs = 16 * (C::kBf16 ? lane & 15 : lane & 7);
  const int vq = 4 * rows_v_quad(lane);
  const int vofs = VB * (lane & 15);
#pragma unroll
  for (int u = 0; u < C::kGroups; ++u) {
    const int tf = T0 + rows_group<C>(u, wave);
    if constexpr (C::PU) {
      const int tfc = min(tf, len - 1);
      const int rmax = max(len - 1 - tf, 0);
      const int e = rows_clamp_page(p, sread(s.page[u]));
      const int64_t base = (int64_t)e * p.kv_sblk + (int64_t)(tfc & (p.P - 1)) * p.kv_stok + (int64_t)h * p.kv_shead;
      const uint8_t* kb = p.k + base;
      const uint8_t* vb = p.v + base;
      const uint32_t stok = (uint32_t)p.kv_stok;
#pragma unroll
      for (int j = 0; j < C::kKLoads; ++j) s.k[u][j] = load16(kb + (uint32_t)(min(KR * j + kr, rmax) * stok + kofs));
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const uint8_t* src = vb + (uint32_t)(min(vq + i, rmax) * stok + vofs);
        if constexpr (C::kBf16) s.v[u][i] = load16(src);
        else s.v[u][i] = __builtin_nontemporal_load((const u32x2*)src);
      }
    } else {
      const int32_t* table = (const int32_t*)p.table;
      const int64_t head = (int64_t)h * p.kv_shead;
#pragma unroll
      for (int j = 0; j < C::kKLoads; ++j) {
        const int tok = min(tf + KR * j + kr, len - 1);
        const int e = rows_clamp_page(p, table[table_word(p, b, tok >> p.logP)]);
        s.k[u][j] = load16(p.k + (int64_t)e * p.kv_sblk + (int64_t)(tok & (p.P - 1)) * p.kv_stok + head + kofs);
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int tok = min(tf + vq + i, len - 1);
        const int e = rows_clamp_page(p, table[table_word(p, b, tok >> p.logP)]);
        const uint8_t* src = p.v + (int64_t)e * p.kv_sblk + (int64_t)(tok & (p.P - 1)) * p.kv_stok + head + vofs;
        if constexpr (C::kBf16) s.v[u][i] = load16(src);
        else s.v[u][i] = __builtin_nontemporal_load((const u32x2*)src);
      }
    }
  }
  if constexpr (C::SK == kScaleTokenHead) {
    if (tid < 2 * C::CT) {
      const int tok = min(T0 + (tid & (C::CT - 1)), len - 1);
      const int e = rows_clamp_page(p, s.sc_page);
      s.sc = (tid < C::CT ? p.ks : p.vs)[(int64_t)e * p.sc_sblk + (int64_t)(tok & (p.P - 1)) * p.sc_stok +
                                         (int64_t)h * p.sc_shead];
    }
  }
}

// Per-token scales of one chunk in LDS: K scales (times sm_scale log2 e), V scales, and (f16 weights) vscale_bound of
// the latter.
template <typename C>
using RowsScales = float[C::kVBound ? 3 : 2][C::SK == kScaleTokenHead ? C::CT : 1];

__device__ __forceinline__ bool rows_finite(float x) { return fabsf(x) <= __FLT_MAX__; }

// Chunk kk's codes and scales into LDS. partial: some row of the tile does not see all of its tokens. *bad becomes
// kk + 1 if values or value scales are not finite and were replaced by zeros: any of a BF16 chunk (whose infinities the
// split weights would turn into NaN), NaN codes of a partial FP8 chunk (in the others every row gets the NaN anyway).
template <typename C>
__device__ __forceinline__ void rows_store(const DecodeParams& p, const RowsStage<C>& s, uint8_t* buf,
                                           RowsScales<C>& ssc, int kk, bool partial, int* bad, int wave, int lane, int tid) {
  uint8_t* kbuf = buf;
  uint8_t* vbuf = buf + C::CT * kHeadDim * 2;
#pragma unroll
  for (int u = 0; u < C::kGroups; ++u) {
    const int t0 = rows_group<C>(u, wave);
#pragma unroll
    for (int j = 0; j < C::kKLoads; ++j) {
      const U4& w = s.k[u][j];
      if constexpr (C::kBf16) {
        const int tok = t0 + 4 * j + (lane >> 4);
        const int un = lane & 15;
        *(u32x4*)(kbuf + tok * 256 + 16 * (un ^ (tok & 7) ^ (un >> 3))) = u32x4{w.x, w.y, w.z, w.w};
      } else {
        const int tok = t0 + 8 * j + (lane >> 3);
        const int sg = lane & 7;
        const int sw = (tok & 7) ^ (sg >> 2);
        *(u32x4*)(kbuf + tok * 256 + 16 * ((2 * sg) ^ sw)) = rows_k_cvt<C>(w.x, w.y);
        *(u32x4*)(kbuf + tok * 256 + 16 * ((2 * sg + 1) ^ sw)) = rows_k_cvt<C>(w.z, w.w);
      }
    }
    const int cl = lane & 15;
    const int quad = rows_v_quad(lane);
    const int unit = 2 * ((t0 & 63) >> 4) + (quad & 1);
    uint8_t* vrow = vbuf + (t0 >> 6) * 16384 + 8 * cl * 128 + 8 * (quad >> 1);
    if constexpr (C::kBf16) {
      uint32_t w[4][4] = {{s.v[u][0].x, s.v[u][0].y, s.v[u][0].z, s.v[u][0].w},
                          {s.v[u][1].x, s.v[u][1].y, s.v[u][1].z, s.v[u][1].w},
                          {s.v[u][2].x, s.v[u][2].y, s.v[u][2].z, s.v[u][2].w},
                          {s.v[u][3].x, s.v[u][3].y, s.v[u][3].z, s.v[u][3].w}};
      const bf16x2 zero = {(__bf16)0.0f, (__bf16)0.0f};
      float nan = 0.0f;  // what 0 times an infinity or NaN leaves
#pragma unroll
      for (int i = 0; i < 16; ++i)
        nan = __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, w[i >> 2][i & 3]), zero, nan, false);
      if (__any(nan != 0.0f)) {
        *bad = kk + 1;
#pragma unroll
        for (int i = 0; i < 16; ++i) {
          uint32_t& x = w[i >> 2][i & 3];
          if ((x & 0x7f80u) == 0x7f80u) x &= 0xffff0000u;
          if ((x & 0x7f800000u) == 0x7f800000u) x &= 0xffffu;
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const uint32_t sel = (i & 1) ? 0x07060302u : 0x05040100u;
        const u32x2 x = {__builtin_amdgcn_perm(w[1][i >> 1], w[0][i >> 1], sel),
                         __builtin_amdgcn_perm(w[3][i >> 1], w[2][i >> 1], sel)};
        *(u32x2*)(vrow + i * 128 + 16 * (unit ^ ((i + cl) & 7))) = x;
      }
    } else {
      uint32_t o[8];
      rows_transpose4(s.v[u][0].x, s.v[u][1].x, s.v[u][2].x, s.v[u][3].x, o);
      rows_transpose4(s.v[u][0].y, s.v[u][1].y, s.v[u][2].y, s.v[u][3].y, o + 4);
      if constexpr (C::KV == kKvFp8) {
        if (partial) {
          uint32_t any = 0u;
#pragma unroll
          for (int i = 0; i < 8; ++i) {  // NaN: the code 0x7f with either sign
            const uint32_t nan = ((o[i] & 0x7f7f7f7fu) + 0x01010101u) & 0x80808080u;
            any |= nan;
            o[i] &= ~((nan >> 7) * 0xffu);
          }
          if (__any(any != 0u)) *bad = kk + 1;
        }
      }
#pragma unroll
      for (int i = 0; i < 8; ++i)
        *(u32x2*)(vrow + i * 128 + 16 * (unit ^ ((i + cl) & 7))) =
            C::KV == kKvFp8 ? rows_fp8_to_f16(o[i]) : rows_int8_to_bf16(o[i]);
    }
  }
  if constexpr (C::SK == kScaleTokenHead) {
    if (tid < C::CT) {
      ssc[0][tid] = s.sc * p.qscale;
    } else if (tid < 2 * C::CT) {
      const bool fin = rows_finite(s.sc);
      if (!fin) *bad = kk + 1;
      ssc[1][tid - C::CT] = fin ? s.sc : 0.0f;
      if constexpr (C::kVBound) ssc[2][tid - C::CT] = vscale_bound(s.sc);
    }
  }
}

// ---- the products ---------------------------------------------------------------------------------------------

template <typename C>
__device__ __forceinline__ f32x16 rows_mfma_k(u32x4 a, u32x4 q, f32x16 acc) {
  if constexpr (C::kF16K)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, q), acc, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, q), acc, 0, 0, 0);
}
template <typename C>
__device__ __forceinline__ f32x16 rows_mfma_v(u32x4 a, u32x4 w, f32x16 acc) {
  if constexpr (!C::kVF16)
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, w), acc, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, w), acc, 0, 0, 0);
}

// This lane's state of its row (n = lane % 32; the row's two lanes share m and add their l at the end) and its
// output channels 32 ct + 8 a + 4 hf + b, at o[ct][4 a + b].
struct RowsState {
  float m, l;
  f32x16 o[4];
};

// w0, w1 = f16 pairs hi + lo (22 bits): hi rounded to nearest, lo the rounded remainder. The remainders come from
// v_fma_mix_f32, which reads a half as a float (the compiler converts back and subtracts: two instructions more each).
__device__ __forceinline__ void rows_split_f16(float w0, float w1, uint32_t& hi, uint32_t& lo) {
  const f16x2 h = {(_Float16)w0, (_Float16)w1};
  hi = __builtin_bit_cast(uint32_t, h);
  float r0, r1;
  __asm__("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[0,0,0] op_sel_hi:[1,0,0]" : "=v"(r0) : "v"(hi), "v"(w0));
  __asm__("v_fma_mix_f32 %0, %1, -1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r1) : "v"(hi), "v"(w1));
  lo = __builtin_bit_cast(uint32_t, f16x2{(_Float16)r0, (_Float16)r1});
}

// The K operands (A) of 32 tokens from t0 on: one per 16 channels.
template <typename C>
__device__ __forceinline__ void rows_read_k(const uint8_t* buf, int t0, int lane, u32x4 (&ka)[8]) {
  const int n = lane & 31, hf = lane >> 5;
  const uint8_t* kbuf = buf + (t0 + n) * 256;
#pragma unroll
  for (int k = 0; k < 8; ++k) ka[k] = *(const u32x4*)(kbuf + 16 * ((2 * k + hf) ^ (n & 7) ^ (k >> 2)));
}
template <typename C>
__device__ __forceinline__ f32x16 rows_scores(const u32x4 (&ka)[8], const u32x4 (&qb)[C::kQOps]) {
  f32x16 s;
#pragma unroll
  for (int i = 0; i < 16; ++i) s[i] = 0.0f;
  // An f16 q's remainders go first, while the sum is small: they then cost it no rounding (float32 outputs 5.3e-7 from 64
  // bits at 512 + 2048 tokens, 16 heads, and 6.9e-7 with each after its high part; 512 + 8192, 32 heads 199 -> 203 us).
  if constexpr (C::kQSplit) {
#pragma unroll
    for (int k = 0; k < 8; ++k) s = rows_mfma_k<C>(ka[k], qb[8 + k], s);
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) s = rows_mfma_k<C>(ka[k], qb[k], s);
  return s;
}
// The V operands (A) of the 16 tokens from t0 on: one per 32 channels.
template <typename C>
__device__ __forceinline__ void rows_read_v(const uint8_t* buf, int t0, int lane, u32x4 (&va)[4]) {
  const int n = lane & 31, hf = lane >> 5;
  const uint8_t* vbuf = buf + C::CT * kHeadDim * 2 + (t0 >> 6) * 16384 + n * 128;
#pragma unroll
  for (int ct = 0; ct < 4; ++ct)
    va[ct] = *(const u32x4*)(vbuf + ct * 4096 + 16 * ((2 * ((t0 & 63) >> 4) + hf) ^ ((n + (n >> 3)) & 7) ^ (4 * (ct & 1))));
}

// The wave's tokens [t0, t0 + TW) of the chunk (T: their first token in the sequence) folded into the state, 32 at a
// time. qs: the score scale, not negative (SK token-head: in the per-token K scales instead). rlen: the tokens this
// lane's row sees; rlen_min: the fewest that a row of the wave sees.
//
// Two waves share a SIMD, so LDS latency is covered by the wave itself: a block's V operands and the next block's K
// operands are requested ahead of its softmax, and the next block's score products stand between its two halves.
template <typename C>
__device__ __forceinline__ void rows_compute(const uint8_t* buf, const RowsScales<C>& ssc, int t0, int T, int lane,
                                             const u32x4 (&qb)[C::kQOps], float qs, int rlen, int rlen_min, RowsState& st) {
  constexpr int NH = C::TW / 32;
  const int hf = lane >> 5;
  u32x4 ka[8];
  rows_read_k<C>(buf, t0, lane, ka);
  f32x16 s = rows_scores<C>(ka, qb);
#pragma unroll
  for (int half = 0; half < NH; ++half) {
    const int th = t0 + 32 * half;
    u32x4 va[2][4];
    rows_read_v<C>(buf, th, lane, va[0]);

    float mul = qs;
    float mx = kNegInf;
    if constexpr (C::SK == kScaleTokenHead) {
      mul = 1.0f;
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int at = th + 8 * a + 4 * hf;
        const f32x4 kq = *(const f32x4*)&ssc[0][at];
#pragma unroll
        for (int j = 0; j < 4; ++j) s[4 * a + j] *= kq[j];
      }
    }
    if (T + 32 * half + 32 > rlen_min) {  // some row of the wave does not see all of them
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int tok = T + 32 * half + 8 * (i >> 2) + 4 * hf + (i & 3);
        const float x = C::SK == kScaleTokenHead ? s[i] : s[i] * qs;
        s[i] = tok < rlen ? x : kNegInf;
      }
      mul = 1.0f;
    }
    if constexpr (C::kVBound) {
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const f32x4 vb = *(const f32x4*)&ssc[2][th + 8 * a + 4 * hf];
#pragma unroll
        for (int j = 0; j < 4; ++j) mx = fmaxf(mx, s[4 * a + j] + vb[j]);
      }
    } else {
#pragma unroll
      for (int i = 0; i < 16; ++i) mx = fmaxf(mx, s[i]);
    }
    mx = max_xor<32>(mx) * mul;
    const bool move = mx > st.m + kSlack;
    if (__any(move)) {
      const float mn = move ? mx : st.m;
      const float alpha = move ? fast_exp2(st.m - mn) : 1.0f;  // 0 when m was -inf
      st.l *= alpha;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) st.o[ct] *= alpha;
      st.m = mn;
    }
    const float base = (st.m == kNegInf ? 0.0f : st.m) - kBias;

    if (half + 1 < NH) rows_read_k<C>(buf, th + 32, lane, ka);
    rows_read_v<C>(buf, th + 16, lane, va[1]);
    f32x16 s_next = s;
    float l0 = 0.0f, l1 = 0.0f;
#pragma unroll
    for (int h2 = 0; h2 < 2; ++h2) {
      float w[8];
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        w[j] = fast_exp2(fmaf(s[8 * h2 + j], mul, -base));
        if (j & 1) l1 += w[j]; else l0 += w[j];
      }
      if constexpr (C::SK == kScaleTokenHead) {
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          const f32x4 vs = *(const f32x4*)&ssc[1][th + 16 * h2 + 8 * a + 4 * hf];
#pragma unroll
          for (int j = 0; j < 4; ++j) w[4 * a + j] *= vs[j];
        }
      }
      u32x4 part[3];
      if constexpr (!C::kVF16) {
#pragma unroll
        for (int q = 0; q < 3; ++q) {
#pragma unroll
          for (int j = 0; j < 4; ++j) {
            const bf16x2 x = pack_bf16(w[2 * j], w[2 * j + 1]);
            w[2 * j] -= (float)x.x;
            w[2 * j + 1] -= (float)x.y;
            part[q][j] = __builtin_bit_cast(uint32_t, x);
          }
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          uint32_t hi, lo;
          rows_split_f16(w[2 * j], w[2 * j + 1], hi, lo);
          part[0][j] = hi;
          part[1][j] = lo;
        }
      }
#pragma unroll
      for (int q = 0; q < (C::kVF16 ? 2 : 3); ++q) {
#pragma unroll
        for (int ct = 0; ct < 4; ++ct) st.o[ct] = rows_mfma_v<C>(va[h2][ct], part[q], st.o[ct]);
      }
      if (h2 == 0 && half + 1 < NH) s_next = rows_scores<C>(ka, qb);
    }
    st.l += l0 + l1;
    s = s_next;
  }
}

// The values of tokens T .. T + n - 1 that rows_store replaced by zeros, added for the rows that see them.
template <typename C>
__device__ __forceinline__ void rows_add_nonfinite(const DecodeParams& p, int b, int h, int T, int n, int lane, int rlen,
                                                   RowsState& st) {
  const int32_t* table = (const int32_t*)p.table;
  const int hf = lane >> 5;
#pragma unroll 1
  for (int tok = T; tok < T + n; ++tok) {
    const int e = rows_clamp_page(p, load_uniform(table + table_word(p, b, tok >> p.logP)));
    const int64_t in_page = tok & (p.P - 1);
    const uint8_t* src = p.v + (int64_t)e * p.kv_sblk + in_page * p.kv_stok + (int64_t)h * p.kv_shead;
    float mul = 1.0f;
    if constexpr (C::SK == kScaleTokenHead) {
      const float sc = p.vs[(int64_t)e * p.sc_sblk + in_page * p.sc_stok + (int64_t)h * p.sc_shead];
      if (!rows_finite(sc)) mul = sc;
    }
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
#pragma unroll
      for (int a = 0; a < 4; ++a) {
        const int ch = 32 * ct + 8 * a + 4 * hf;
        float x[4];
        if constexpr (C::kBf16) {
          const u32x2 w = *(const u32x2*)(src + 2 * ch);
          x[0] = __uint_as_float(w.x << 16);
          x[1] = __uint_as_float(w.x & 0xffff0000u);
          x[2] = __uint_as_float(w.y << 16);
          x[3] = __uint_as_float(w.y & 0xffff0000u);
        } else {
          const uint32_t w = *(const uint32_t*)(src + ch);
          if constexpr (C::KV == kKvFp8) {
            fp8x4_to_f32(w, x);
          } else {
#pragma unroll
            for (int j = 0; j < 4; ++j) x[j] = (float)(int8_t)((w >> (8 * j)) & 0xffu);
          }
        }
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float v = x[j] * mul;
          if (tok < rlen && !rows_finite(v)) st.o[ct][4 * a + j] += v;
        }
      }
    }
  }
}

// Row gr's q as the B operands of the score products (channels 16 k + 8 hf .. + 7); flip: negated.
template <typename C>
__device__ __forceinline__ void rows_load_q(const DecodeParams& p, int b, int h, int gr, int lane, bool flip,
                                            u32x4 (&qb)[C::kQOps]) {
  const int qi = gr / p.G;
  const int hq = h * p.G + (gr - qi * p.G);
  const uint16_t* src = (const uint16_t*)p.q + (int64_t)b * p.q_sb + (int64_t)qi * p.q_sq + (int64_t)hq * p.q_sh + 8 * (lane >> 5);
  const uint32_t sign = flip ? 0x80008000u : 0u;
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    u32x4 x = *(const u32x4*)(src + 16 * k);
    x ^= sign;
    if constexpr (C::kQSplit) {
      const f16x8 f = __builtin_bit_cast(f16x8, x);
      bf16x8 hi, lo;
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        hi[j] = (__bf16)(float)f[j];
        lo[j] = (__bf16)((float)f[j] - (float)hi[j]);
      }
      qb[k] = __builtin_bit_cast(u32x4, hi);
      qb[8 + k] = __builtin_bit_cast(u32x4, lo);
    } else {
      qb[k] = x;
    }
  }
}

// ---- the line of tiles ------------------------------------------------------------------------------------------

// Tokens that tile t of a sequence of len tokens reads: those its last row sees.
template <int BM>
__device__ __forceinline__ int rows_tile_chunks(const DecodeParams& p, int len, int t) {
  int vis = len;
  if (!p.noncausal) vis -= p.Q - 1 - (min((t + 1) * BM, p.Q * p.G) - 1) / p.G;
  return max((vis + kRowsChunk - 1) / kRowsChunk, 1);
}

// s_line[b T + t]: exclusive prefix sum of one KV head's tile costs (chunks + piece cost; 0 for empty sequences),
// s_line[B T] their sum; s_len: the clamped lengths.
template <int NW, int BM>
__device__ __forceinline__ void build_tile_line(const DecodeParams& p, int* s_line, int* s_len, int* s_wsum) {
  constexpr int NT = NW * 64;
  const int tid = threadIdx.x, lane = tid & 63;
  const int T = p.n_rg, N = p.B * T;
  for (int b = tid; b < p.B; b += NT) {
    const int len = (p.lens ? p.lens[b] : p.len_cap + p.len_offset) - p.len_offset;
    s_len[b] = len < 0 ? 0 : (len > p.len_cap ? p.len_cap : len);
  }
  __syncthreads();
  const int per_thread = (N + NT - 1) / NT;
  const int lo = min(tid * per_thread, N), hi = min(lo + per_thread, N);
  int sum = 0;
  for (int i = lo; i < hi; ++i) {
    const int b = i / T;
    const int len = s_len[b];
    const int cost = len > 0 ? rows_tile_chunks<BM>(p, len, i - b * T) + p.piece_cost : 0;
    s_line[i] = cost;
    sum += cost;
  }
  int x = sum;
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    const int y = __shfl_up(x, off, 64);
    if (lane >= off) x += y;
  }
  if (lane == 63) s_wsum[tid >> 6] = x;
  __syncthreads();
  int run = x - sum;
  for (int w = 0; w < (tid >> 6); ++w) run += s_wsum[w];
  for (int i = lo; i < hi; ++i) {
    const int cost = s_line[i];
    s_line[i] = run;
    run += cost;
  }
  if (tid == NT - 1) s_line[N] = run;
  __syncthreads();
}

// Four channels of a finished row, as write_out stores each.
__device__ __forceinline__ void rows_write4(const DecodeParams& p, int b, int qi, int hq, int ch, f32x4 o, float lse2,
                                            bool packed) {
  if (!packed) {
#pragma unroll
    for (int j = 0; j < 4; ++j) write_out(p, b, qi, hq, ch + j, o[j], lse2);
    return;
  }
  const int64_t at = (int64_t)b * p.o_sb + (int64_t)qi * p.o_sq + (int64_t)hq * p.o_sh + ch;
  u32x2 w;
  if (p.out_dtype == kFBf16) {
    w = u32x2{(uint32_t)f32_to_bf16_bits(o[0]) | ((uint32_t)f32_to_bf16_bits(o[1]) << 16),
              (uint32_t)f32_to_bf16_bits(o[2]) | ((uint32_t)f32_to_bf16_bits(o[3]) << 16)};
  } else {
    w = u32x2{__builtin_bit_cast(uint32_t, f16x2{(_Float16)o[0], (_Float16)o[1]}),
              __builtin_bit_cast(uint32_t, f16x2{(_Float16)o[2], (_Float16)o[3]})};
  }
  *(u32x2*)((uint16_t*)p.out + at) = w;
}

// The combine of one tile's n pieces by the whole workgroup: piece 0 (the tile's start) lies in slot 2 g_first + 1,
// piece j > 0 in slot 2 (g_first + j).
template <int BM, int NT>
__device__ __forceinline__ void rows_combine(const DecodeParams& p, int b, int h, int t, int64_t g_first, int n, int live,
                                             bool packed, int tid) {
  constexpr int D = kHeadDim;
  ws_acquire();
  for (int idx = tid; idx < live * (D / 4); idx += NT) {
    const int r = idx / (D / 4);
    const int ch = 4 * (idx - r * (D / 4));
    float M = kNegInf, W = 0.0f;
    f32x4 O = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int j0 = 0; j0 < n; j0 += 4) {
      float lv[4];
      f32x4 ov[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool in = j0 + j < n;
        const int64_t slot = 2 * (g_first + j0 + j) + (j0 + j == 0 ? 1 : 0);
        lv[j] = kNegInf;
        ov[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        if (in) {
          lv[j] = ws_load(p.ws_lse + slot * BM + r);
          float x, y, z, w;
          ws_load2(p.ws_out + (slot * BM + r) * D + ch, x, y);
          ws_load2(p.ws_out + (slot * BM + r) * D + ch + 2, z, w);
          ov[j] = f32x4{x, y, z, w};
        }
      }
      const float nm = fmaxf(fmaxf(fmaxf(lv[0], lv[1]), fmaxf(lv[2], lv[3])), M);
      const float mu = nm == kNegInf ? 0.0f : nm;
      const float alpha = W > 0.0f ? fast_exp2(M - mu) : 0.0f;
      W *= alpha;
      O *= alpha;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float e = fast_exp2(lv[j] - mu);  // 0 for pieces in which the row saw no token
        W += e;
        O += ov[j] * e;
      }
      M = nm;
    }
    const int gr = t * BM + r;
    const int qi = gr / p.G;
    const float inv = W > 0.0f ? 1.0f / W : 0.0f;
    const float lse2 = W > 0.0f ? M + __log2f(W) : kNegInf;
    rows_write4(p, b, qi, h * p.G + (gr - qi * p.G), ch, O * inv, lse2, packed);
  }
}

// The combine as a launch of its own (DecodeParams::two_pass): the workgroups take strips of kCombineRows rows of the
// tiles in turn, the pieces in the slots of rows_combine. The last arriver of a tile is one CU: 33 pieces of 128 rows
// (64 KiB each) took it about 25 us, some 85 GB/s. Spread over the chip they take 5.5 us: a call whose tiles have much to
// combine pays a second launch instead (rows_two_pass), and its pieces are plain stores.
constexpr int kCombineRows = 8, kCombineWaves = 4, kCombineGrid = 4 * kComputeUnits;
template <int BM>
__global__ __launch_bounds__(kCombineWaves * 64) void rows_combine_kernel(const DecodeParams p) {
  constexpr int D = kHeadDim, NT = kCombineWaves * 64, kJ = 8;
  static_assert(NT == kCombineRows * (D / 4), "one output of four channels per thread");
  extern __shared__ int s_dyn[];
  __shared__ int s_wsum[kCombineWaves];
  const int T = p.n_rg, X = p.piece_cost, tid = threadIdx.x;
  int* s_line = s_dyn;
  int* s_len = s_dyn + p.B * T + 1;
  build_tile_line<kCombineWaves, BM>(p, s_line, s_len, s_wsum);
  const int64_t total = (int64_t)p.Hkv * s_line[p.B * T];
  const int64_t per = p.per_forced > 0 ? p.per_forced : (total + p.grid - 1) / p.grid;
  const bool packed = !p.merge_out && !p.lse_out && p.out_dtype != kFF32 && ((uintptr_t)p.out & 7) == 0 &&
                      ((p.o_sb | p.o_sq | p.o_sh) & 3) == 0;
  constexpr int kStrips = BM / kCombineRows;
  const int ch = 4 * (tid % (D / 4));
  for (int64_t strip = blockIdx.x; strip < (int64_t)p.B * p.Hkv * T * kStrips; strip += gridDim.x) {
    const int tile = (int)(strip / kStrips);
    const int r = (int)(strip % kStrips) * kCombineRows + tid / (D / 4);
    const int t = tile % T, h = tile / T % p.Hkv, b = tile / (T * p.Hkv);
    const int gr = t * BM + r;
    if (s_len[b] == 0 || gr >= p.Q * p.G) continue;
    const int start = s_line[b * T + t], end = s_line[b * T + t + 1];
    const int64_t c0 = (int64_t)p.Hkv * s_line[b * T] + (int64_t)h * (s_line[(b + 1) * T] - s_line[b * T]) + (start - s_line[b * T]);
    const int64_t g_first = (c0 + X) / per;
    const int n = (int)((c0 + (end - start) - 1) / per - g_first) + 1;
    if (n == 1) continue;  // written by the workgroup that held it
    float M = kNegInf, W = 0.0f;
    f32x4 O = {0.0f, 0.0f, 0.0f, 0.0f};
    for (int j0 = 0; j0 < n; j0 += kJ) {
      float lv[kJ];
      f32x4 ov[kJ];
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        const int jj = min(j0 + j, n - 1);  // a piece past the last is read again, for nothing
        const int64_t row = (2 * (g_first + jj) + (jj == 0 ? 1 : 0)) * BM + r;
        lv[j] = p.ws_lse[row];
        ov[j] = *(const f32x4*)(p.ws_out + row * D + ch);
      }
      float nm = M;
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        if (j0 + j >= n) {
          lv[j] = kNegInf;
          ov[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
        nm = fmaxf(nm, lv[j]);
      }
      const float mu = nm == kNegInf ? 0.0f : nm;
      const float alpha = W > 0.0f ? fast_exp2(M - mu) : 0.0f;
      W *= alpha;
      O *= alpha;
#pragma unroll
      for (int j = 0; j < kJ; ++j) {
        const float e = fast_exp2(lv[j] - mu);  // 0 for pieces in which the row saw no token
        W += e;
        O += ov[j] * e;
      }
      M = nm;
    }
    const int qi = gr / p.G;
    const float inv = W > 0.0f ? 1.0f / W : 0.0f;
    rows_write4(p, b, qi, h * p.G + (gr - qi * p.G), ch, O * inv, W > 0.0f ? M + __log2f(W) : kNegInf, packed);
  }
}

template <int KV, int SK, bool PU, bool QF16, int WM, int NW, int NBUF>
__global__ __launch_bounds__(NW * 64, 2) void decode_rows_kernel(const DecodeParams p) {
  typedef RowsCfg<KV, SK, PU, QF16, WM, NW, NBUF> C;
  constexpr int NT = C::NT, BM = C::BM, D = kHeadDim;

  extern __shared__ int s_dyn[];  // [B T + 1] the tile line, then [B] lengths
  int* s_line = s_dyn;
  __shared__ int s_wsum[NW];
  __shared__ int s_last;
  __shared__ __attribute__((aligned(16))) uint8_t smem[C::kSmem];
  __shared__ __attribute__((aligned(16))) RowsScales<C> s_sc[NBUF];
  __shared__ int s_bad[NBUF];  // rows_store: 1 + the chunk in the buffer, if it holds values that are not finite

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = sread(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int B = p.B, T = p.n_rg, Hkv = p.Hkv, X = p.piece_cost;
  const int rows = p.Q * p.G;
  int* s_len = s_dyn + B * T + 1;

  if (tid < NBUF) s_bad[tid] = 0;
  build_tile_line<NW, BM>(p, s_line, s_len, s_wsum);
  // Sequences with no tokens: zero rows, or the caller's partial.
  for (int b = blockIdx.x; b < B; b += gridDim.x) {
    if (s_len[b] > 0) continue;
    for (int i = tid; i < p.Q * p.Hq * D; i += NT) write_out(p, b, i / (D * p.Hq), (i / D) % p.Hq, i % D, 0.0f, kNegInf);
  }

  const int64_t total = (int64_t)Hkv * s_line[B * T];
  if (total == 0) return;
  const int64_t per = p.per_forced > 0 ? p.per_forced : (total + gridDim.x - 1) / gridDim.x;
  const int64_t g = line_index(gridDim.x);
  const int64_t c_begin = g * per;
  if (c_begin >= total) return;
  const int64_t c_end = min(c_begin + per, total);

  // The piece at c_begin: sequence b, KV head h, tile t, from chunk k on.
  int b, h, t, k;
  {
    int lo = 0, hi = B - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if ((int64_t)Hkv * s_line[mid * T] <= c_begin) lo = mid; else hi = mid - 1;
    }
    b = sread(lo);
    const int head = sread(s_line[(b + 1) * T] - s_line[b * T]);  // one head's units
    const int64_t r = c_begin - (int64_t)Hkv * s_line[b * T];
    h = sread((int)(r / head));
    const int rt = sread((int)(r - (int64_t)h * head));
    lo = 0;
    hi = T - 1;
    while (lo < hi) {
      const int mid = (lo + hi + 1) >> 1;
      if (s_line[b * T + mid] - s_line[b * T] <= rt) lo = mid; else hi = mid - 1;
    }
    t = sread(lo);
    k = sread(max(rt - (s_line[b * T + t] - s_line[b * T]) - X, 0));
  }
  auto tile_start = [&](int sb, int sh, int stl) -> int64_t {
    const int head = s_line[(sb + 1) * T] - s_line[sb * T];
    return (int64_t)Hkv * s_line[sb * T] + (int64_t)sh * head + (s_line[sb * T + stl] - s_line[sb * T]);
  };
  auto tile_span = [&](int sb, int stl) { return sread(s_line[sb * T + stl + 1] - s_line[sb * T + stl]); };

  int span = tile_span(b, t);
  int64_t c0 = tile_start(b, h, t);
  int k_end = sread((int)(min(c_end, c0 + span) - c0 - X));
  if (k_end <= k) return;  // the range lies within one tile's piece cost
  int len = sread(s_len[b]);

  RowsStage<C> stage;
  u32x4 qb[C::kQOps];
  rows_fetch_pages<C>(p, b, k, len, wave, tid, stage);
  rows_issue<C>(p, b, h, k, len, wave, lane, tid, stage);
  rows_fetch_pages<C>(p, b, k + 1, len, wave, tid, stage);

  const bool packed = !p.merge_out && !p.lse_out && p.out_dtype != kFF32 && ((uintptr_t)p.out & 7) == 0 &&
                      ((p.o_sb | p.o_sq | p.o_sh) & 3) == 0;

  for (;;) {
    // This wave's rows: lane n has row r0 + n (rows past the last repeat it; they are not written).
    const int r0 = t * BM + 32 * wm;
    const int gr = min(r0 + (lane & 31), rows - 1);
    const float qscale = SK == kScaleTokenHead ? 0.0f : p.qscale * (SK == kScaleHead ? load_uniform(p.ks + h) : 1.0f);
    const float vscale = SK == kScaleHead ? load_uniform(p.vs + h) : 1.0f;
    rows_load_q<C>(p, b, h, gr, lane, qscale < 0.0f, qb);
    const int rlen = p.noncausal ? len : len - (p.Q - 1 - gr / p.G);
    const int rlen_min = sread(rlen);  // lane 0's row sees the fewest tokens, the last lane's the most
    const int rlen_max = __builtin_amdgcn_readlane(rlen, 31);

    // Chunks from this one on are not seen whole by the tile's first row.
    const int partial = (p.noncausal ? len : max(len - (p.Q - 1 - t * BM / p.G), 0)) / C::CT;

    // The next piece of the range, if it holds chunks of one.
    int nb_ = b, nh = h, nt = t + 1, n_end = 0, nlen = 0, nspan = 0;
    int64_t nc0 = c0 + span;
    if (nc0 < c_end) {
      if (nt == T) {
        nt = 0;
        if (++nh == Hkv) {
          nh = 0;
          do {
            ++nb_;
          } while (s_len[nb_] == 0);
          nb_ = sread(nb_);
        }
      }
      nspan = tile_span(nb_, nt);
      n_end = sread((int)(min(c_end, nc0 + nspan) - nc0 - X));
      nlen = sread(s_len[nb_]);
    }
    const bool more = n_end > 0;

    RowsState st;
    st.m = kNegInf;
    st.l = 0.0f;
#pragma unroll
    for (int ct = 0; ct < 4; ++ct) {
#pragma unroll
      for (int i = 0; i < 16; ++i) st.o[ct][i] = 0.0f;
    }

    int cur = 0;
    if constexpr (NBUF == 2) {
      rows_store<C>(p, stage, smem, s_sc[0], k, k >= partial, s_bad, wave, lane, tid);
      __syncthreads();
    }
    for (int kk = k; kk < k_end; ++kk) {
      // The lane's LDS and cache offsets are worked out again for every chunk (some 50 instructions): kept over the
      // loop they would take 40 registers that the operands in flight need.
      int ln = lane;
      __asm__ volatile("" : "+v"(ln));
      if constexpr (NBUF == 1) {
        if (kk > k) __syncthreads();  // every wave is done with the previous chunk
        rows_store<C>(p, stage, smem, s_sc[0], kk, kk >= partial, s_bad, wave, ln, tid);
        __syncthreads();
      }
      const bool last = kk + 1 == k_end;
      if (!last) {
        rows_issue<C>(p, b, h, kk + 1, len, wave, ln, tid, stage);
        rows_fetch_pages<C>(p, b, kk + 2, len, wave, tid, stage);
      } else if (more) {
        rows_fetch_pages<C>(p, nb_, 0, nlen, wave, tid, stage);
        rows_issue<C>(p, nb_, nh, 0, nlen, wave, ln, tid, stage);
        rows_fetch_pages<C>(p, nb_, 1, nlen, wave, tid, stage);
      }
      {
        const int t0 = wn * C::TW;
        const int tok = kk * C::CT + t0;
        if (tok < rlen_max) {
          rows_compute<C>(smem + cur * C::kBuf, s_sc[cur], t0, tok, ln, qb, fabsf(qscale), rlen, rlen_min, st);
          if (C::kNonfinite && sread(s_bad[cur]) == kk + 1)
            rows_add_nonfinite<C>(p, b, h, tok, min(C::TW, rlen_max - tok), ln, rlen, st);
        }
      }
      if constexpr (NBUF == 2) {
        if (!last) {
          cur ^= 1;
          rows_store<C>(p, stage, smem + cur * C::kBuf, s_sc[cur], kk + 1, kk + 1 >= partial, s_bad + cur, wave, ln, tid);
          __syncthreads();
        }
      }
    }

    // ---- merge the token groups; write the tile, or this piece's partial -------------------------------------
    __syncthreads();  // the chunk buffers become the merge buffers
    if (tid < NBUF) s_bad[tid] = 0;
    st.l = sum_xor<32>(st.l);
    float* mrg = (float*)smem;
    if (wn > 0) {
      float* dst = mrg + (((wn - 1) * WM + wm) * 66) * 64;
#pragma unroll
      for (int i = 0; i < 16; ++i)
        *(f32x4*)(dst + (i * 64 + lane) * 4) =
            f32x4{st.o[i >> 2][4 * (i & 3)], st.o[i >> 2][4 * (i & 3) + 1], st.o[i >> 2][4 * (i & 3) + 2], st.o[i >> 2][4 * (i & 3) + 3]};
      dst[64 * 64 + lane] = st.m;
      dst[65 * 64 + lane] = st.l;
    }
    if constexpr (C::WN > 1) __syncthreads();
    float lse2 = kNegInf;
    if (wn == 0) {
      float M = st.m;
#pragma unroll
      for (int w = 1; w < C::WN; ++w) M = fmaxf(M, mrg[(((w - 1) * WM + wm) * 66 + 64) * 64 + lane]);
      const float mu = M == kNegInf ? 0.0f : M;
      const float e0 = st.l > 0.0f ? fast_exp2(st.m - mu) : 0.0f;
      float L = st.l * e0;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
#pragma unroll
        for (int i = 0; i < 16; ++i) st.o[ct][i] = st.l > 0.0f ? st.o[ct][i] * e0 : 0.0f;
      }
#pragma unroll
      for (int w = 1; w < C::WN; ++w) {
        const float* src = mrg + (((w - 1) * WM + wm) * 66) * 64;
        const float lw = src[65 * 64 + lane];
        const float e = lw > 0.0f ? fast_exp2(src[64 * 64 + lane] - mu) : 0.0f;
        L += lw * e;
        if (lw > 0.0f) {
#pragma unroll
          for (int i = 0; i < 16; ++i) {
            const f32x4 x = *(const f32x4*)(src + (i * 64 + lane) * 4);
#pragma unroll
            for (int j = 0; j < 4; ++j) st.o[i >> 2][4 * (i & 3) + j] += x[j] * e;
          }
        }
      }
      const float f = L > 0.0f ? vscale / L : 0.0f;
      lse2 = L > 0.0f ? M - kBias + __log2f(L) : kNegInf;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) st.o[ct] *= f;
    }
    if constexpr (C::WN > 1) __syncthreads();
    float* s_o = (float*)smem;
    float* s_lse = s_o + BM * (D + 4);
    if (wn == 0) {
      const int r = 32 * wm + (lane & 31), hf = lane >> 5;
#pragma unroll
      for (int ct = 0; ct < 4; ++ct) {
#pragma unroll
        for (int a = 0; a < 4; ++a)
          *(f32x4*)(s_o + r * (D + 4) + 32 * ct + 8 * a + 4 * hf) =
              f32x4{st.o[ct][4 * a], st.o[ct][4 * a + 1], st.o[ct][4 * a + 2], st.o[ct][4 * a + 3]};
      }
      if (hf == 0) s_lse[r] = lse2;
    }
    __syncthreads();

    const int nchunks = span - X;
    const int64_t g_first = (c0 + X) / per;  // the workgroups holding the tile's first and last chunks
    const int64_t g_last = (c0 + X + nchunks - 1) / per;
    const int live = min(BM, rows - t * BM);
    const bool whole = g_first == g_last;
    const int64_t slot = 2 * g + (k == 0 ? 1 : 0);
    for (int idx = tid; idx < live * (D / 4); idx += NT) {
      const int r = idx / (D / 4);
      const int ch = 4 * (idx - r * (D / 4));
      const f32x4 o = *(const f32x4*)(s_o + r * (D + 4) + ch);
      if (whole) {
        const int row = t * BM + r;
        const int qi = row / p.G;
        rows_write4(p, b, qi, h * p.G + (row - qi * p.G), ch, o, s_lse[r], packed);
      } else if (!C::kInLaunch || p.two_pass) {
        *(f32x4*)(p.ws_out + (slot * BM + r) * D + ch) = o;
        if (ch == 0) p.ws_lse[slot * BM + r] = s_lse[r];
      } else {
        ws_store2(p.ws_out + (slot * BM + r) * D + ch, o[0], o[1]);
        ws_store2(p.ws_out + (slot * BM + r) * D + ch + 2, o[2], o[3]);
        if (ch == 0) ws_store(p.ws_lse + slot * BM + r, s_lse[r]);
      }
    }
    if constexpr (C::kInLaunch) {
      if (!whole && !p.two_pass) {
        const int seg = (b * Hkv + h) * T + t;
        const int n = (int)(g_last - g_first + 1);
        ws_publish();
        __syncthreads();
        if (tid == 0) s_last = ws_arrive(p.counters + seg) == (unsigned)n - 1u;
        __syncthreads();
        if (s_last) {
          rows_combine<BM, NT>(p, b, h, t, g_first, n, live, packed, tid);
          if (tid == 0) __hip_atomic_store(p.counters + seg, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    }
    if (!more) break;
    __syncthreads();  // the merge buffers become chunk buffers again
    b = nb_;
    h = nh;
    t = nt;
    k = 0;
    k_end = n_end;
    len = nlen;
    span = nspan;
    c0 = nc0;
  }
}

template <int KV, int SK, int WM, int NW, int NBUF>
static hipError_t launch_rows_t(const DecodeParams& p, hipStream_t stream, const LaunchEvents& events) {
  dim3 grid(p.grid), block(NW * 64);
  const size_t lds = (size_t)(p.B * p.n_rg + 1 + p.B) * sizeof(int);
  const bool pu = p.P >= 16, f16 = p.q_dtype == kFF16;
  LaunchEvents ev = events;  // the interval of a call spans both of its launches
  if (p.two_pass) ev.stop = nullptr;
  if (pu && !f16) launch_kernel(decode_rows_kernel<KV, SK, true, false, WM, NW, NBUF>, grid, block, lds, stream, ev, p);
  else if (pu) launch_kernel(decode_rows_kernel<KV, SK, true, true, WM, NW, NBUF>, grid, block, lds, stream, ev, p);
  else if (!f16) launch_kernel(decode_rows_kernel<KV, SK, false, false, WM, NW, NBUF>, grid, block, lds, stream, ev, p);
  else launch_kernel(decode_rows_kernel<KV, SK, false, true, WM, NW, NBUF>, grid, block, lds, stream, ev, p);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !p.two_pass) return e;
  constexpr int BM = 32 * WM;
  const int64_t strips = (int64_t)p.B * p.Hkv * p.n_rg * (BM / kCombineRows);
  dim3 cgrid((unsigned)(strips < kCombineGrid ? strips : kCombineGrid)), cblock(kCombineWaves * 64);
  if (events.start) hipExtLaunchKernelGGL((rows_combine_kernel<BM>), cgrid, cblock, (uint32_t)lds, stream, nullptr, events.stop, 0u, p);
  else hipLaunchKernelGGL((rows_combine_kernel<BM>), cgrid, cblock, lds, stream, p);
  return hipGetLastError();
}

template <int WM, int NW, int NBUF>
static hipError_t launch_rows_cfg(const DecodeParams& p, int kv_dtype, int scale_kind, hipStream_t stream, const LaunchEvents& ev) {
  if (kv_dtype == kKvBf16) return launch_rows_t<kKvBf16, kScaleNone, WM, NW, NBUF>(p, stream, ev);
  if (kv_dtype == kKvFp8 && scale_kind == kScaleHead) return launch_rows_t<kKvFp8, kScaleHead, WM, NW, NBUF>(p, stream, ev);
  if (kv_dtype == kKvFp8) return launch_rows_t<kKvFp8, kScaleTokenHead, WM, NW, NBUF>(p, stream, ev);
  if (kv_dtype == kKvInt8 && scale_kind == kScaleHead) return launch_rows_t<kKvInt8, kScaleHead, WM, NW, NBUF>(p, stream, ev);
  if (kv_dtype == kKvInt8) return launch_rows_t<kKvInt8, kScaleTokenHead, WM, NW, NBUF>(p, stream, ev);
  return hipErrorInvalidValue;
}

}  // namespace bpt
