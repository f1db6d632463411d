// Single-token decode over segments of any kind in 16-bit caches (gfx950,
// wave64): the general form of the page kernels.
//
// Scope: bf16 or fp16 cache and query of the same type, head_dim 64 or 128, 1
// to 16 query heads per KV head, segments of any token count whose keys are
// dense, uniform (2, 4, 8 bits) or Dart pages with any promoted count, in key
// groups that divide the 128-token tile or are a multiple of it (at most four
// per tile), and whose values are dense or uniform (2, 4, 8 bits) in at most
// four groups; fp16 metadata.  The page kernels (decode_fast.hip,
// decode_uniform.hip) take the runs they are made for; this kernel takes the
// rest: other head ratios, key groups and head_dims, partial pages, and dense
// pieces beside them.  What it does not take (fp32 and float64 caches, other
// metadata, odd group sizes) stays with decode_split_general.
//
// One wave owns one split, a contiguous range of segments of one (batch, kv
// head), and walks it in tiles of TILE tokens (128, or 64 with 8-bit codes,
// whose registers a larger tile would not leave room for).
//
// Bound by VALU issue and by the latency between a tile's steps at two waves
// per SIMD (200-255 VGPRs), not by memory.  Against decode_split_general, which
// spent about 100 VALU per element on scalar index arithmetic (one layer,
// MI355X): 8 sequences x 4,096 tokens, 2-bit pages in groups of 64, fp16: 572
// -> 23.6 µs; 8 x 8,011 tokens of Dart pages, six heads per KV head: 1,453 ->
// 36.8 µs; 16 x 4,000 tokens of head_dim 64: 841 -> 31.8 µs.
//
// Layout.  Both products run on v_mfma_f32_16x16x32 with the query heads in
// the 16 rows.  Codes are packed along tokens for keys and along channels for
// values, so the column index takes the packed direction: in Q K, lane (n, kq)
// holds the TILE / 16 tokens NJ n .. NJ n + NJ - 1 of channels 32 kb + 8 kq +
// i, one load of 1 to 8 bytes per channel, straight from memory into
// registers (no staging: every byte is read by one lane); in P V it holds the
// D / 16 channels NC n .. of tokens 32 kb + 8 kq + i.  A pair of K indices
// and a position j then give one dword of a B operand:
//   2-bit codes: the dequantized values of the four codes are tabulated per
//   (channel, group) or (token, group) in LDS, as byte planes, and looked up
//   with v_perm_b32, two tables per permute: 1.5 VALU per element;
//   4- and 8-bit codes: code to fp16 (the e4m3 pattern of a code below 16 is
//   code x 2^-9), then the rounding chain in packed fp16, then bf16: 2 to 3.75
//   VALU per element.
// Promoted channels have zero 2-bit tables and take a pass of their own over
// their slots, 32 to a block.
//
// Arithmetic.  K and V hold the reference's dequantized values exactly (its
// rounding chain), the query is exact in the operand type, and the softmax
// weights stay fp32: a weight is the exact sum of three 16-bit parts (8 + 8 +
// 8 bits for bf16; 11 + 11 + 2 for fp16), the parts of 4 heads fill the 16
// rows of one MFMA (those of 8 heads two MFMAs, of 16 heads three), and their
// products meet in the fp32 accumulators when the split ends.
#include <hip/hip_runtime.h>
#include <math.h>

#include <algorithm>

#include "dkv_capi_util.h"
#include "dkv_decode.h"
#include "dkv_device.h"
#include "dkv_page_common.h"

using namespace dkv;

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

constexpr int kTileWaves = 4;
constexpr int kMaxGroups = 4;       // key groups per tile, value groups per token
constexpr float kTileSlack = 5.5f;  // natural-log headroom before the running max moves (e^5.5 = 245)

struct TileParams {
  // This kernel's segments are numbered packed first: index i < n_packed is
  // rest entry packed_first + i, then come the dense entries in order (rest
  // entries: the descriptors outside the page kernels' run, then the tail).
  DecodeParams d;
  int packed_first, n_packed, splits;
  // what every packed segment shares
  int key_group, value_group, promoted;
  // LDS of one wave (bytes): key tables, value tables, weights, then what Dart
  // pages need (scale/zero pairs by channel, the query rows)
  int kt, vt, pw, sz, q, wave_bytes;
};

__device__ __forceinline__ int uni(int x) { return __builtin_amdgcn_readfirstlane(x); }

// Rest entry i of the decode call (a descriptor outside the page kernels' run).
__device__ __forceinline__ const_segment& rest_entry(const DecodeParams& p, int i) {
  return descriptor(p.a.segments, i < p.skip_first ? i : i + p.skip_count);
}

// Global loads from a wave-uniform base and a 32-bit lane offset (the
// addresses come out of memory, so without the address space they would be
// flat loads, which also count as LDS traffic).
template <class T>
__device__ __forceinline__ T gload(const void* base, uint32_t off) {
  typedef __attribute__((address_space(1))) const uint8_t gbyte;
  typedef __attribute__((address_space(1))) const T gtype;
  return *(gtype*)((gbyte*)(uintptr_t)base + off);
}

// A packed segment's fields, moved to this (batch, kv head).  Wave-uniform.
struct Packed {
  int tokens;
  const uint8_t *k, *kh, *v;
  const int32_t* ki;
  const uint16_t *ks, *kz, *vs, *vz;
};

__device__ __forceinline__ Packed packed_segment(const_segment& s, int64_t bh) {
  const PageAddr a = page_addr(s, bh);
  Packed t;
  t.tokens = uni(s.tokens);
  t.k = a.kl; t.kh = a.kh; t.ki = a.ki; t.ks = a.ks; t.kz = a.kz;
  t.v = a.vc; t.vs = a.vs; t.vz = a.vz;
  return t;
}

__device__ __forceinline__ int groups_of(int n, int group) { return (n + group - 1) / group; }

// fp16 pair -> the pair in the operand type.
template <bool BF>
__device__ __forceinline__ uint32_t to_operand(half2v h) {
  if (!BF) return __builtin_bit_cast(uint32_t, h);
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){(float)h[0], (float)h[1]}, bf16x2));
}

template <bool BF>
__device__ __forceinline__ float4v mfma(u32x4 a, u32x4 b, float4v c) {
  if constexpr (BF)
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8, a), __builtin_bit_cast(half8, b), c, 0, 0,
                                                  0);
}

// Byte-plane table of the dequantized values of codes 0..3 (x = low bytes, y =
// high bytes).  0 s and 1 s are exact, so one fused multiply-add rounds once
// there, as the chain's add does; codes 2 and 3 multiply and add separately.
template <bool BF>
__device__ __forceinline__ uint2 table4(uint32_t sz) {
  const half2v s = splat_h(sz & 0xffffu), z = splat_h(sz >> 16);
  const half2v h01 = __builtin_elementwise_fma(half2v{0.0f16, 1.0f16}, s, z);
  const half2v p23 = half2v{2.0f16, 3.0f16} * s;
  const uint32_t v01 = to_operand<BF>(h01), v23 = to_operand<BF>(p23 + z);
  return make_uint2(perm(v23, v01, 0x06040200u), perm(v23, v01, 0x07050301u));
}

// ---- codes: NP consecutive positions (tokens of a key channel, channels of a
// value row) of K index k are one load of NP * BITS / 8 bytes ----

template <int BITS, int NP>
struct Codes {
  static constexpr int kBytes = NP * BITS / 8;                     // 1, 2, 4 or 8
  static constexpr int kPairRegs = kBytes <= 2 ? 1 : kBytes / 2;   // registers of two K indices
};

// Codes of K indices 0 .. NK - 1 of the lane into regs, two per pair: index k's
// are at base(k) (wave-uniform) + off(k) bytes.
template <int BITS, int NP, int NK, int N, class Base, class Off>
__device__ __forceinline__ void load_codes(uint32_t (&regs)[N], Base base, Off off) {
  typedef Codes<BITS, NP> C;
  static_assert(N == NK / 2 * C::kPairRegs, "one tile's codes");
#pragma unroll
  for (int p = 0; p < NK / 2; ++p) {
    const uint8_t *a = base(2 * p), *b = base(2 * p + 1);
    const uint32_t oa = off(2 * p), ob = off(2 * p + 1);
    if constexpr (C::kBytes == 1) {
      regs[p] = (uint32_t)gload<uint8_t>(a, oa) | ((uint32_t)gload<uint8_t>(b, ob) << 16);
    } else if constexpr (C::kBytes == 2) {
      regs[p] = (uint32_t)gload<uint16_t>(a, oa) | ((uint32_t)gload<uint16_t>(b, ob) << 16);
    } else if constexpr (C::kBytes == 4) {
      regs[2 * p] = gload<uint32_t>(a, oa);
      regs[2 * p + 1] = gload<uint32_t>(b, ob);
    } else {
      const u32x2 x = gload<u32x2>(a, oa), y = gload<u32x2>(b, ob);
      regs[4 * p] = x.x; regs[4 * p + 1] = x.y;
      regs[4 * p + 2] = y.x; regs[4 * p + 3] = y.y;
    }
  }
}

// Operand dwords of a pair of K indices at every position j, from 2-bit codes
// in byte planes: y's bytes are (k0, k1, k0, k1) at positions j and j + NP / 2.
template <int NP>
__device__ __forceinline__ void lookup_pair(uint32_t codes, uint32_t lo0, uint32_t hi0, uint32_t lo1, uint32_t hi1,
                                            uint32_t m3, uint32_t sel2, uint32_t (&op)[NP]) {
  const uint32_t y = NP == 8 ? perm(0u, codes, 0x03010200u) : perm(codes >> 4, codes, 0x06040200u);
#pragma unroll
  for (int j = 0; j < NP / 2; ++j) {
    const uint32_t e = ((y >> (2 * j)) & m3) | sel2;
    const uint32_t l = perm(lo1, lo0, e), h = perm(hi1, hi0, e);
    op[j] = perm(h, l, 0x05010400u);
    op[j + NP / 2] = perm(h, l, 0x07030602u);
  }
}

// Two code bytes (values below 16) of word half W as an fp16 pair.
template <bool HI>
__device__ __forceinline__ half2v codes16(uint32_t e) {
  return __builtin_bit_cast(half2v, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(e, 512.f, HI));
}

// The same from 4- or 8-bit codes by the arithmetic chain; s, z hold the two
// indices' scales and zero points.
template <bool BF, int BITS, int NP>
__device__ __forceinline__ void chain_pair(const uint32_t* codes, uint32_t s, uint32_t z, uint32_t (&op)[NP]) {
  const half2v sv = __builtin_bit_cast(half2v, s), zv = __builtin_bit_cast(half2v, z);
  auto value = [&](half2v c) {
    const half2v prod = c * sv;  // -ffp-contract=off: one rounding each
    return to_operand<BF>(prod + zv);
  };
  if constexpr (BITS == 4) {
#pragma unroll
    for (int q = 0; q < NP / 4; ++q) {  // four positions: bytes (k0, k1, k0, k1), two positions per byte
      const uint32_t y = NP == 8 ? perm(codes[1], codes[0], q ? 0x07030602u : 0x05010400u) : perm(0u, codes[0], 0x03010200u);
      const uint32_t even = y & 0x0f0f0f0fu, odd = (y >> 4) & 0x0f0f0f0fu;
      op[4 * q] = value(codes16<false>(even));
      op[4 * q + 1] = value(codes16<false>(odd));
      op[4 * q + 2] = value(codes16<true>(even));
      op[4 * q + 3] = value(codes16<true>(odd));
    }
  } else {
    static_assert(BITS == 8, "2-bit codes take the tables");
#pragma unroll
    for (int q = 0; q < NP / 4; ++q) {
      const uint32_t a = codes[q], b = codes[NP / 4 + q];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        // bytes (a_j, 0x64, b_j, 0x64): 1024 + code in fp16
        const uint32_t y = perm(b, a, j == 0 ? 0x0c040c00u : j == 1 ? 0x0c050c01u : j == 2 ? 0x0c060c02u : 0x0c070c03u);
        const half2v c = __builtin_bit_cast(half2v, y | 0x64006400u) - half2v{1024.0f16, 1024.0f16};
        op[4 * q + j] = value(c);
      }
    }
  }
}

// Scale (low half) and zero point (high half) of item lane_at + at.
__device__ __forceinline__ uint32_t load_sz(const uint16_t* s, const uint16_t* z, uint32_t lane_at, int at) {
  return (uint32_t)gload<uint16_t>(s + at, 2 * lane_at) | ((uint32_t)gload<uint16_t>(z + at, 2 * lane_at) << 16);
}

// Item `i` of a table region: a byte-plane table (2-bit codes) or its place in
// the pair (s0, s1), (z0, z1) of the arithmetic chain.
template <bool BF>
__device__ __forceinline__ void put_table(uint8_t* region, int i, uint32_t sz, bool two_bit) {
  if (two_bit) {
    *(uint2*)(region + 8 * i) = table4<BF>(sz);
  } else {
    uint8_t* at = region + 8 * (i >> 1) + 2 * (i & 1);
    *(uint16_t*)at = (uint16_t)sz;
    *(uint16_t*)(at + 4) = (uint16_t)(sz >> 16);
  }
}

// The softmax state and accumulators of a wave, and the steps both kinds of
// tile share.  GP: query rows per KV head rounded up to 4, 8 or 16.  S[j] row 4
// kq + i = head (4 kq + i) % GP, column n = token NJ n + j; O[j] row 4 kq + i =
// weight part and head of that row (head % GP), column n = channel NC n + j.
template <int D, bool BF, int GP, int TILE>
struct TileState {
  static constexpr int NJ = TILE / 16;          // tokens of a lane
  static constexpr int NC = D / 16;             // channels of a lane
  static constexpr int KB = D / 32;             // 32-channel blocks of Q K
  static constexpr int VB = TILE / 32;          // 32-token blocks of P V
  static constexpr int PASSES = GP == 4 ? 1 : GP == 8 ? 2 : 3;  // MFMAs that take the three weight parts
  static constexpr int U = NJ * GP / 16;        // a lane's own positions in the softmax
  static constexpr int kPRow = TILE * 2 + 16;   // bytes of a weight row
  u32x4 qa[KB];
  float m_run[4], l_part[4];
  float4v O[NC];
  uint8_t* pw;  // weight rows in LDS
  float scale;
  int n, kq;

  __device__ __forceinline__ void q_products(int kb, const uint32_t (&op)[4][NJ], float4v (&S)[NJ]) const {
#pragma unroll
    for (int j = 0; j < NJ; ++j) S[j] = mfma<BF>(qa[kb], u32x4{op[0][j], op[1][j], op[2][j], op[3][j]}, S[j]);
  }

  // Row 16 pass + r of the weights = part (16 pass + r) / GP of head r % GP.
  __device__ __forceinline__ void p_products(int kb, const uint32_t (&op)[4][NC]) {
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
      const u32x4 w = *(const u32x4*)(pw + (16 * pass + n) * kPRow + 64 * kb + 16 * kq);
#pragma unroll
      for (int j = 0; j < NC; ++j) O[j] = mfma<BF>(w, u32x4{op[0][j], op[1][j], op[2][j], op[3][j]}, O[j]);
    }
  }

  // Logits to weights in LDS, nt tokens of the tile valid.  A lane takes its
  // own positions only: with GP 4 and 8 the rows repeat, and the lane groups
  // that hold the same heads share the tokens.
  __device__ __forceinline__ void softmax(const float4v (&S)[NJ], int nt) {
    float x[U][4];
    const int start = GP == 4 ? kq * U : GP == 8 ? (kq >> 1) * U : 0;
    bool over = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float v;
        if constexpr (GP == 4) {
          const float v0 = kq & 1 ? S[U + u][i] : S[u][i], v1 = kq & 1 ? S[3 * U + u][i] : S[2 * U + u][i];
          v = kq & 2 ? v1 : v0;
        } else if constexpr (GP == 8) {
          v = kq & 2 ? S[U + u][i] : S[u][i];
        } else {
          v = S[u][i];
        }
        v *= scale;
        if (nt < TILE) v = NJ * n + start + u < nt ? v : -INFINITY;
        x[u][i] = v;
        over |= v > m_run[i] + kTileSlack;
      }
    }
    if (__ballot(over) != 0ull) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float mx = x[0][i];
#pragma unroll
        for (int u = 1; u < U; ++u) mx = fmaxf(mx, x[u][i]);
#pragma unroll
        for (int off = 1; off < 16; off <<= 1) mx = fmaxf(mx, __shfl_xor(mx, off, 64));
        if (GP == 4) mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
        if (GP <= 8) mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        const float m_new = fmaxf(m_run[i], mx);
        const float alpha = m_new == -INFINITY ? 1.f : __builtin_amdgcn_exp2f((m_run[i] - m_new) * kLog2e);
        l_part[i] *= alpha;
        m_run[i] = m_new;
#pragma unroll
        for (int j = 0; j < NC; ++j) O[j][i] *= alpha;
      }
    }
    // weights (fp16 operands: times 2^7, undone in the record) and their parts
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int head = GP == 4 ? i : GP == 8 ? 4 * (kq & 1) + i : 4 * kq + i;
      float w[U];
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float dlt = x[u][i] - m_run[i];
        w[u] = __builtin_amdgcn_exp2f(BF ? dlt * kLog2e : __builtin_fmaf(dlt, kLog2e, 7.f));
        l_part[i] += w[u];
      }
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        uint32_t part[U > 1 ? U / 2 : 1];
#pragma unroll
        for (int u = 0; u < U; u += 2) {
          const float w0 = w[u], w1 = U > 1 ? w[(u + 1) % U] : 0.f;
          float r0, r1;
          if constexpr (BF) {
            const uint32_t b0 = __builtin_bit_cast(uint32_t, w0), b1 = __builtin_bit_cast(uint32_t, w1);
            part[u / 2] = perm(b1, b0, 0x07060302u);
            r0 = w0 - __builtin_bit_cast(float, b0 & 0xffff0000u);
            r1 = w1 - __builtin_bit_cast(float, b1 & 0xffff0000u);
          } else {
            const auto h = __builtin_amdgcn_cvt_pkrtz(w0, w1);
            part[u / 2] = __builtin_bit_cast(uint32_t, h);
            r0 = w0 - (float)h[0];
            r1 = w1 - (float)h[1];
          }
          w[u] = r0;
          if (U > 1) w[(u + 1) % U] = r1;
        }
        uint8_t* dst = pw + (k * GP + head) * kPRow + 2 * (NJ * n + start);
        if constexpr (U == 1) *(uint16_t*)dst = (uint16_t)part[0];
        else if constexpr (U == 2) *(uint32_t*)dst = part[0];
        else if constexpr (U == 4) *(uint2*)dst = make_uint2(part[0], part[1]);
        else *(uint4*)dst = make_uint4(part[0], part[1], part[2], part[3]);
      }
    }
  }

  // One tile of dense rows: tokens t0 .. t0 + nt - 1 of k, v ([tokens][D]).
  __device__ __forceinline__ void dense_tile(const uint16_t* k, const uint16_t* v, int t0, int nt) {
    float4v S[NJ];
#pragma unroll
    for (int j = 0; j < NJ; ++j) {
      S[j] = float4v{0.f, 0.f, 0.f, 0.f};
      const uint32_t off = 2 * ((t0 + min(NJ * n + j, nt - 1)) * D + 8 * kq);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) S[j] = mfma<BF>(qa[kb], gload<u32x4>(k, off + 64 * kb), S[j]);
    }
    softmax(S, nt);
    lds_sync();
#pragma unroll 1
    for (int kb = 0; kb < VB; ++kb) {
      if (32 * kb >= nt) break;  // the weights of later tokens are zero
      uint32_t r[8][NC / 2];
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int tok = 32 * kb + 8 * kq + i;
        typedef uint32_t row_t __attribute__((ext_vector_type(NC / 2)));
        const row_t x = gload<row_t>(v, 2 * ((t0 + min(tok, nt - 1)) * D + NC * n));
#pragma unroll
        for (int c = 0; c < NC / 2; ++c) r[i][c] = tok < nt ? x[c] : 0u;
      }
#pragma unroll
      for (int pass = 0; pass < PASSES; ++pass) {
        const u32x4 w = *(const u32x4*)(pw + (16 * pass + n) * kPRow + 64 * kb + 16 * kq);
#pragma unroll
        for (int j = 0; j < NC; ++j) {
          const uint32_t sel = j % 2 ? 0x07060302u : 0x05040100u;
          O[j] = mfma<BF>(w, u32x4{perm(r[1][j / 2], r[0][j / 2], sel), perm(r[3][j / 2], r[2][j / 2], sel),
                                   perm(r[5][j / 2], r[4][j / 2], sel), perm(r[7][j / 2], r[6][j / 2], sel)}, O[j]);
        }
      }
    }
    lds_sync();
  }
};

// Rest entries s0 .. s1 - 1 (in this kernel's numbering) of one (batch, kv
// head) element by element in fp32, by one wave: lane = channels lane, lane +
// 64.  Only for splits with non-finite sums.
template <int D>
__device__ __forceinline__ void scalar_split(const TileParams& p, int bhi, int split, int s0, int s1, int lane) {
  const DecodeParams& d = p.d;
  const dkv_decode_args& a = d.a;
  const int64_t b = bhi / (int)a.Hkv, kvh = bhi % (int)a.Hkv;
  const int cache_dt = (int)a.cache_dtype, meta = (int)a.meta_dtype;
  constexpr int R = D / 64;
#pragma unroll 1
  for (int h = 0; h < d.group; ++h) {
    const int64_t hq = kvh * d.group + h;
    float q[R], acc[R], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int r = 0; r < R; ++r) {
      q[r] = dev_load(a.query, b * a.q_sb + hq * a.q_sh + lane + 64 * r, (int)a.q_dtype);
      acc[r] = 0.f;
    }
#pragma unroll 1
    for (int i = s0; i < s1; ++i) {
      const int j = i - p.n_packed;
      const dkv_segment seg = general_segment(d, i < p.n_packed ? p.packed_first + i : j < p.packed_first ? j : j + p.n_packed);
      int slot[R];
#pragma unroll
      for (int r = 0; r < R; ++r) {
        slot[r] = -1;
        if (seg.key_kind != DKV_KEY_MIXED) continue;
        for (int k = 0; k < seg.promoted; ++k)
          if (((const int32_t*)seg.key[2])[bhi * seg.key_bh[2] + k] == lane + 64 * r) slot[r] = k;
      }
#pragma unroll 1
      for (int t = 0; t < seg.tokens; ++t) {
        float x = 0.f;
#pragma unroll
        for (int r = 0; r < R; ++r)
          x = fmaf(q[r], key_value(seg, bhi, lane + 64 * r, t, D, slot[r], cache_dt, meta), x);
        x = wave_sum(x) * (float)a.scale;
        const float m_new = fmaxf(m, x), old = expf(m - m_new), w = expf(x - m_new);
        l = l * old + w;
        m = m_new;
#pragma unroll
        for (int r = 0; r < R; ++r)
          acc[r] = acc[r] * old + w * value_value(seg, bhi, t, lane + 64 * r, D, cache_dt, meta);
      }
    }
    float* rec = (float*)a.workspace + ((b * a.Hq + hq) * d.split_stride + d.split_offset + split) * (D + 2);
    if (lane == 0) {
      rec[0] = m;
      rec[1] = l;
    }
#pragma unroll
    for (int r = 0; r < R; ++r) rec[2 + lane + 64 * r] = acc[r];
  }
}

// KBITS: key code width; MIXED: Dart pages (KBITS 2); VBITS: value code width.
template <int D, bool BF, int GP, int KBITS, bool MIXED, int VBITS>
__global__ void __launch_bounds__(64 * kTileWaves, 2) decode_tiles(TileParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int TILE = KBITS == 8 || VBITS == 8 ? 64 : 128;
  typedef TileState<D, BF, GP, TILE> St;
  constexpr int NJ = St::NJ, NC = St::NC, KB = St::KB, VB = St::VB, PASSES = St::PASSES;
  constexpr int KK = D / 4, VK = TILE / 4;  // K indices of a lane
  constexpr int KIT = kMaxGroups * D / 64, VIT = kMaxGroups * TILE / 64;  // table items of a lane
  constexpr int KSTEP = D / 64, VSTEP = TILE / 64;                       // items per group
  constexpr int kTabK = D * 8 + 16, kTabV = TILE * 8 + 16;
  typedef Codes<KBITS, NJ> KC;
  typedef Codes<VBITS, NC> VC;
  const DecodeParams& d = p.d;
  const dkv_decode_args& a = d.a;
  const int lane = threadIdx.x & 63;
  const int wave = uni(threadIdx.x >> 6);
  const int n = lane & 15, kq = lane >> 4;
  const int worker = (int)blockIdx.x * kTileWaves + wave;
  const int Hkv = (int)a.Hkv, G = d.group;
  if (worker >= (int)a.B * Hkv * p.splits) return;
  const int split = uni(worker % p.splits), bhi = uni(worker / p.splits);
  const int b = uni(bhi / Hkv), kvh = uni(bhi % Hkv);
  const int64_t bh = bhi;
  uint8_t* lds = smem + wave * p.wave_bytes;
  const int s0 = uni((int)(((int64_t)split * d.n_total) / p.splits));
  const int s1 = uni((int)(((int64_t)(split + 1) * d.n_total) / p.splits));
  const uint32_t m3 = in_sgpr(0x03030303u), sel2 = in_vgpr(0x04000400u);
  const int kgroup = p.key_group, vgroup = p.value_group, promoted = p.promoted;
  const int Gv = groups_of(D, vgroup), vrow = Gv * vgroup * VBITS / 8;

  // ---- the query: A operands of row n (head n % GP, zero past G), and its
  // rows in LDS for the promoted channels ----
  St st;
  st.n = n;
  st.kq = kq;
  st.pw = lds + p.pw;
  st.scale = (float)a.scale;
  {
    const int head = n % GP;
    const uint16_t* q = (const uint16_t*)a.query + (int64_t)b * a.q_sb + (int64_t)(kvh * G + (head < G ? head : 0)) * a.q_sh;
#pragma unroll
    for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
      for (int w = 0; w < 4; ++w) {
        const int c = 32 * kb + 8 * kq + 2 * w;
        const uint32_t v = (uint32_t)gload<uint16_t>(q, 2 * c) | ((uint32_t)gload<uint16_t>(q, 2 * c + 2) << 16);
        st.qa[kb][w] = head < G ? v : 0u;
      }
      if (MIXED && n < GP) *(u32x4*)(lds + p.q + 2 * (n * D + 32 * kb + 8 * kq)) = st.qa[kb];
    }
  }
  // the weight rows past the three parts stay zero
  for (int i = lane; i < (16 * PASSES - 3 * GP) * St::kPRow / 4; i += 64)
    *(uint32_t*)(st.pw + 3 * GP * St::kPRow + 4 * i) = 0u;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    st.m_run[i] = -INFINITY;
    st.l_part[i] = 0.f;
  }
#pragma unroll
  for (int j = 0; j < NC; ++j) st.O[j] = float4v{0.f, 0.f, 0.f, 0.f};

  // ---- packed tiles ----
  {
    uint32_t kc[KK / 2 * KC::kPairRegs], vc[VK / 2 * VC::kPairRegs];  // the codes of the tile to come
    uint32_t ksz[KIT], vsz[VIT];  // its scales and zero points
    int kidx[8];                  // its promoted channels of this lane, first block (slots 8 kq ..)
    auto load_keys = [&](const Packed& t, int t0) {
      const int Gp = groups_of(t.tokens, kgroup), padded = Gp * kgroup;
      const int row = padded * KBITS / 8;  // bytes of a channel
      const int first = min(t0 + NJ * n, padded - NJ);  // a lane past the page repeats its last tokens
      const uint32_t off = (uint32_t)(first * KBITS / 8 + 8 * kq * row);
      load_codes<KBITS, NJ, KK>(
          kc, [&](int k) { return t.k + (32 * (k >> 3) + (k & 7)) * row; }, [&](int) { return off; });
      const int g0 = t0 / kgroup, ng = min(Gp - g0, max(1, TILE / kgroup));
#pragma unroll
      for (int m = 0; m < KIT; ++m)
        if (m / KSTEP < ng) ksz[m] = load_sz(t.ks, t.kz, lane * Gp, 64 * (m % KSTEP) * Gp + g0 + m / KSTEP);
      if constexpr (MIXED) {
#pragma unroll
        for (int i = 0; i < 8; ++i) kidx[i] = gload<int>(t.ki, 4 * min(8 * kq + i, promoted - 1));
      }
    };
    auto load_values = [&](const Packed& t, int t0) {
      const int last = t.tokens - 1;
      const uint32_t col = (uint32_t)(NC * n * VBITS / 8);
      if (t0 + TILE <= t.tokens) {  // a whole tile's addresses step by the row
        const uint32_t off = col + (uint32_t)(8 * kq * vrow);
        load_codes<VBITS, NC, VK>(
            vc, [&](int k) { return t.v + (t0 + 32 * (k >> 3) + (k & 7)) * vrow; }, [&](int) { return off; });
#pragma unroll
        for (int m = 0; m < VIT; ++m)
          if (m / VSTEP < Gv) vsz[m] = load_sz(t.vs, t.vz, lane * Gv, (t0 + 64 * (m % VSTEP)) * Gv + m / VSTEP);
      } else {  // a partial one repeats its last token
        load_codes<VBITS, NC, VK>(
            vc, [&](int) { return t.v; },
            [&](int k) { return col + (uint32_t)(min(t0 + 32 * (k >> 3) + 8 * kq + (k & 7), last) * vrow); });
#pragma unroll
        for (int m = 0; m < VIT; ++m)
          if (m / VSTEP < Gv) vsz[m] = load_sz(t.vs, t.vz, min(t0 + lane + 64 * (m % VSTEP), last) * Gv, m / VSTEP);
      }
    };
    const uint8_t* vtab = lds + p.vt + (NC * n / vgroup) * kTabV;

    int si = s0, t0 = 0;
    const int stop = min(s1, p.n_packed);
    bool live = si < stop;
    Packed nxt;
    if (live) {
      nxt = packed_segment(rest_entry(d, p.packed_first + si), bh);
      load_keys(nxt, 0);
      load_values(nxt, 0);
    }
#pragma unroll 1
    while (live) {
      const Packed cur = nxt;
      const int cur0 = t0, nt = min(TILE, cur.tokens - t0);
      t0 += TILE;
      if (t0 >= cur.tokens) {
        ++si;
        t0 = 0;
        live = si < stop;
        if (live) nxt = packed_segment(rest_entry(d, p.packed_first + si), bh);
      }

      // ---- key tables ----
      const int Gp = groups_of(cur.tokens, kgroup), g0 = cur0 / kgroup;
      const int ng = min(Gp - g0, max(1, TILE / kgroup));
      const int lane_group = min((cur0 + NJ * n) / kgroup - g0, ng - 1);
      const int row = Gp * kgroup * KBITS / 8;
      const uint32_t tok_off = (uint32_t)(min(cur0 + NJ * n, Gp * kgroup - NJ) * KBITS / 8);
      uint32_t pl[4], ph[4];  // promoted channels' codes of the lane
      auto load_promoted = [&](int block, const int (&idx)[8]) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          uint32_t lo[2], hi[2];
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const int slot = min(32 * block + 8 * kq + 2 * w + e, promoted - 1);
            const uint32_t la = (uint32_t)((idx[2 * w + e] & (D - 1)) * row) + tok_off, ha = (uint32_t)(slot * row) + tok_off;
            lo[e] = NJ == 8 ? (uint32_t)gload<uint16_t>(cur.k, la) : (uint32_t)gload<uint8_t>(cur.k, la);
            hi[e] = NJ == 8 ? (uint32_t)gload<uint16_t>(cur.kh, ha) : (uint32_t)gload<uint8_t>(cur.kh, ha);
          }
          pl[w] = lo[0] | (lo[1] << 16);
          ph[w] = hi[0] | (hi[1] << 16);
        }
      };
      if constexpr (MIXED) load_promoted(0, kidx);
#pragma unroll
      for (int m = 0; m < KIT; ++m) {
        if (m / KSTEP < ng) {
          const int c = lane + 64 * (m % KSTEP), g = m / KSTEP;
          put_table<BF>(lds + p.kt + g * kTabK, c, ksz[m], KBITS == 2);
          if (MIXED) *(uint32_t*)(lds + p.sz + 4 * (g * D + c)) = ksz[m];
        }
      }
      if constexpr (MIXED) {
        lds_sync();
        for (int i = lane; i < promoted * ng; i += 64) {
          const int g = i / promoted, c = gload<int>(cur.ki, 4 * (i % promoted)) & (D - 1);
          *(uint2*)(lds + p.kt + g * kTabK + 8 * c) = make_uint2(0u, 0u);
        }
      }
      lds_sync();

      // ---- S = Q K ----
      float4v S[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) S[j] = float4v{0.f, 0.f, 0.f, 0.f};
      const uint8_t* ktab = lds + p.kt + lane_group * kTabK;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        uint32_t op[4][NJ];
        const uint4* tab = (const uint4*)(ktab + (KBITS == 2 ? 8 : 4) * (32 * kb + 8 * kq));
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if constexpr (KBITS == 2) {
            const uint4 tt = tab[w];
            lookup_pair<NJ>(kc[4 * kb + w], tt.x, tt.y, tt.z, tt.w, m3, sel2, op[w]);
          } else {
            const uint4 tt = tab[w / 2];
            chain_pair<BF, KBITS, NJ>(&kc[KC::kPairRegs * (4 * kb + w)], w % 2 ? tt.z : tt.x, w % 2 ? tt.w : tt.y, op[w]);
          }
        }
        st.q_products(kb, op, S);
      }
      // promoted channels: 4-bit codes of 32 slots per block
      if constexpr (MIXED) {
#pragma unroll 1
        for (int block = 0; 32 * block < promoted; ++block) {
          if (block) {
#pragma unroll
            for (int i = 0; i < 8; ++i) kidx[i] = gload<int>(cur.ki, 4 * min(32 * block + 8 * kq + i, promoted - 1));
            load_promoted(block, kidx);
          }
          u32x4 qp;
          uint32_t op[4][NJ];
          const uint16_t* q = (const uint16_t*)(lds + p.q) + (n % GP) * D;
          const uint32_t* sz = (const uint32_t*)(lds + p.sz) + lane_group * D;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const int slot = 32 * block + 8 * kq + 2 * w;
            const int c0 = kidx[2 * w] & (D - 1), c1 = kidx[2 * w + 1] & (D - 1);
            // slots past the last one: zero query, zero scale and zero point
            uint32_t q0 = q[c0], q1 = q[c1], sz0 = sz[c0], sz1 = sz[c1];
            q0 = slot < promoted ? q0 : 0u;
            q1 = slot + 1 < promoted ? q1 : 0u;
            sz0 = slot < promoted ? sz0 : 0u;
            sz1 = slot + 1 < promoted ? sz1 : 0u;
            qp[w] = q0 | (q1 << 16);
            const half2v s = __builtin_bit_cast(half2v, perm(sz1, sz0, 0x05040100u));
            const half2v z = __builtin_bit_cast(half2v, perm(sz1, sz0, 0x07060302u));
            const uint32_t yl = NJ == 8 ? perm(0u, pl[w], 0x03010200u) : perm(pl[w] >> 4, pl[w], 0x06040200u);
            const uint32_t yh = NJ == 8 ? perm(0u, ph[w], 0x03010200u) : perm(ph[w] >> 4, ph[w], 0x06040200u);
#pragma unroll
            for (int j = 0; j < NJ / 2; ++j) {
              const uint32_t e = ((yl >> (2 * j)) & m3) | (((yh >> (2 * j)) & m3) << 2);
              const half2v x = codes16<false>(e) * s, y = codes16<true>(e) * s;
              op[w][j] = to_operand<BF>(x + z);
              op[w][j + NJ / 2] = to_operand<BF>(y + z);
            }
          }
#pragma unroll
          for (int j = 0; j < NJ; ++j) S[j] = mfma<BF>(qp, u32x4{op[0][j], op[1][j], op[2][j], op[3][j]}, S[j]);
        }
      }
      if (live) load_keys(nxt, t0);

      st.softmax(S, nt);

      // ---- value tables (tokens past the tile's end: zero) ----
#pragma unroll
      for (int m = 0; m < VIT; ++m) {
        if (m / VSTEP < Gv) {
          const int tok = lane + 64 * (m % VSTEP);
          put_table<BF>(lds + p.vt + (m / VSTEP) * kTabV, tok, tok < nt ? vsz[m] : 0u, VBITS == 2);
        }
      }
      lds_sync();

      // ---- O += P V ----
#pragma unroll
      for (int kb = 0; kb < VB; ++kb) {
        uint32_t op[4][NC];
        const uint4* tab = (const uint4*)(vtab + (VBITS == 2 ? 8 : 4) * (32 * kb + 8 * kq));
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if constexpr (VBITS == 2) {
            const uint4 tt = tab[w];
            lookup_pair<NC>(vc[4 * kb + w], tt.x, tt.y, tt.z, tt.w, m3, sel2, op[w]);
          } else {
            const uint4 tt = tab[w / 2];
            chain_pair<BF, VBITS, NC>(&vc[VC::kPairRegs * (4 * kb + w)], w % 2 ? tt.z : tt.x, w % 2 ? tt.w : tt.y, op[w]);
          }
        }
        st.p_products(kb, op);
      }
      if (live) load_values(nxt, t0);
      lds_sync();
    }
  }

  // ---- dense segments ----
  const int n_rest = (int)a.n_segments - d.skip_count;
#pragma unroll 1
  for (int i = max(s0, p.n_packed); i < s1; ++i) {
    const int j = i - p.n_packed, e = uni(j < p.packed_first ? j : j + p.n_packed);
    int tokens;
    uint64_t k, v;
    if (e < n_rest) {
      const_segment& s = rest_entry(d, e);
      tokens = s.tokens;
      k = s.key[0] + (uint64_t)(2 * bh * s.key_bh[0]);
      v = s.value[0] + (uint64_t)(2 * bh * s.value_bh[0]);
    } else {
      tokens = a.tail.tokens;
      if (a.tail_tokens_dev != nullptr) {
        const int64_t live_tokens = *a.tail_tokens_dev;
        tokens = (int)(live_tokens < 0 ? 0 : (live_tokens < tokens ? live_tokens : tokens));
      }
      k = a.tail.key[0] + (uint64_t)(2 * bh * a.tail.key_bh[0]);
      v = a.tail.value[0] + (uint64_t)(2 * bh * a.tail.value_bh[0]);
    }
    tokens = uni(tokens);
#pragma unroll 1
    for (int at = 0; at < tokens; at += TILE)
      st.dense_tile((const uint16_t*)uniform_u64(k), (const uint16_t*)uniform_u64(v), at, min(TILE, tokens - at));
  }

  // ---- partial state ----
  constexpr float unscale = BF ? 1.f : 0.0078125f;
  float* ws = (float*)a.workspace;
  bool finite = true;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    float l = st.l_part[i];
#pragma unroll
    for (int off = 1; off < 16; off <<= 1) l += __shfl_xor(l, off, 64);
    if (GP == 4) l += __shfl_xor(l, 16, 64);
    if (GP <= 8) l += __shfl_xor(l, 32, 64);
    const int head = GP == 4 ? i : GP == 8 ? 4 * (kq & 1) + i : 4 * kq + i;
    float* rec = ws + (((int64_t)b * a.Hq + kvh * G + head) * d.split_stride + d.split_offset + split) * (D + 2);
    // the lane group that writes this head's record
    const bool writes = head < G && (GP == 4 ? kq == 0 : GP == 8 ? kq < 2 : true);
    if (writes && n == 0) {
      rec[0] = st.m_run[i];
      rec[1] = l * unscale;
    }
    float sum = l;
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      float o = st.O[j][i];
      if (GP == 4) o += __shfl_xor(o, 16, 64);
      if (GP <= 8) o += __shfl_xor(o, 32, 64);
      if (writes) rec[2 + NC * n + j] = o * unscale;
      sum += fabsf(o);
    }
    finite = finite && (!writes || __builtin_isfinite(sum));
  }
  // An infinite value times a weight part that is zero is NaN where the weight
  // itself is not: a split whose sums are not finite is done again one element
  // at a time.
  if (__ballot(!finite) != 0ull) scalar_split<D>(p, bhi, split, s0, s1, lane);
}

bool dense_ok(const dkv_segment& g) {
  return g.tokens < (1 << 20) && g.value_kind == DKV_VALUE_DENSE && g.key[0] % 16 == 0 && (2 * g.key_bh[0]) % 16 == 0 &&
         g.value[0] % 16 == 0 && (2 * g.value_bh[0]) % 16 == 0;
}

// Whether the tile kernel reads this packed segment (host).
bool packed_ok(const dkv_segment& g, int D) {
  if (g.tokens < 1 || g.tokens > (1 << 16) || g.value_kind != DKV_VALUE_UNIFORM) return false;
  if (g.key_kind != DKV_KEY_MIXED && g.key_kind != DKV_KEY_UNIFORM) return false;
  const bool mixed = g.key_kind == DKV_KEY_MIXED;
  const int bits = mixed ? 2 : g.key_bits;
  if ((bits != 2 && bits != 4 && bits != 8) || g.value_bits != bits) return false;
  if (g.key_group != 32 && g.key_group != 64 && (g.key_group < 128 || g.key_group % 128 != 0)) return false;
  if (g.key[0] % 4 != 0 || g.key_bh[0] % 4 != 0 || g.key[3] % 2 != 0 || g.key[4] % 2 != 0) return false;
  if (mixed && (g.promoted < 1 || g.promoted > D || g.key[1] % 4 != 0 || g.key_bh[1] % 4 != 0 || g.key[2] % 4 != 0))
    return false;
  const int groups = (D + g.value_group - 1) / g.value_group;
  const int align = std::max(1, D / 16 * bits / 8);
  return g.value_group >= 8 && g.value_group % 8 == 0 && groups <= kMaxGroups && g.value[0] % align == 0 &&
         g.value_bh[0] % align == 0 && g.value[1] % 2 == 0 && g.value[2] % 2 == 0;
}

bool same_layout(const dkv_segment& a, const dkv_segment& b) {
  return a.key_kind == b.key_kind && a.key_bits == b.key_bits && a.key_group == b.key_group &&
         a.promoted == b.promoted && a.value_bits == b.value_bits && a.value_group == b.value_group;
}

template <int D, bool BF, int GP, int KBITS, bool MIXED>
int launch_tiles(TileParams& p, hipStream_t s) {
  constexpr int TILE = KBITS == 8 ? 64 : 128;
  typedef TileState<D, BF, GP, TILE> St;
  const int kgroups = p.key_group >= TILE ? 1 : TILE / p.key_group;
  const int vgroups = (D + p.value_group - 1) / p.value_group;
  int o = 0;
  p.kt = o; o += kgroups * (D * 8 + 16);
  p.vt = o; o += vgroups * (TILE * 8 + 16);
  p.pw = o; o += 16 * St::PASSES * St::kPRow;
  p.sz = o; o += MIXED ? kgroups * D * 4 : 0;
  p.q = o; o += MIXED ? GP * D * 2 : 0;
  p.wave_bytes = o;
  const int64_t workers = p.d.a.B * p.d.a.Hkv * p.splits;
  const dim3 grid((unsigned)((workers + kTileWaves - 1) / kTileWaves));
  hipLaunchKernelGGL((decode_tiles<D, BF, GP, KBITS, MIXED, KBITS>), grid, dim3(64 * kTileWaves),
                     (size_t)kTileWaves * o, s, p);
  return dkv_check_launch("dkv_decode_attention(tiles)");
}

template <int D, bool BF, int GP>
int launch_tiles_kind(TileParams& p, int bits, bool mixed, hipStream_t s) {
  if (mixed) return launch_tiles<D, BF, GP, 2, true>(p, s);
  if (bits == 2) return launch_tiles<D, BF, GP, 2, false>(p, s);
  if (bits == 4) return launch_tiles<D, BF, GP, 4, false>(p, s);
  return launch_tiles<D, BF, GP, 8, false>(p, s);
}

template <int D, bool BF>
int launch_tiles_heads(TileParams& p, int bits, bool mixed, hipStream_t s) {
  if (p.d.group <= 4) return launch_tiles_kind<D, BF, 4>(p, bits, mixed, s);
  if (p.d.group <= 8) return launch_tiles_kind<D, BF, 8>(p, bits, mixed, s);
  return launch_tiles_kind<D, BF, 16>(p, bits, mixed, s);
}

}  // namespace

namespace dkv {

int launch_tile_decode(const DecodeParams& d, hipStream_t stream, bool* taken) {
  *taken = false;
  const dkv_decode_args& a = d.a;
  if ((a.cache_dtype != kBF16 && a.cache_dtype != kF16) || a.q_dtype != a.cache_dtype || a.meta_dtype != kF16)
    return DKV_OK;
  if ((a.D != 64 && a.D != 128) || d.group > 16 || (a.n_segments > 0 && a.segments_host == nullptr)) return DKV_OK;
  if (a.B * a.Hkv * d.splits >= (int64_t)1 << 31) return DKV_OK;
  const int n_rest = (int)a.n_segments - d.skip_count;
  auto entry = [&](int i) -> const dkv_segment& {
    return i >= n_rest ? a.tail : a.segments_host[i < d.skip_first ? i : i + d.skip_count];
  };
  // one run of packed segments of one layout, everything else dense
  int first = 0, count = 0;
  for (int i = 0; i < d.n_total; ++i) {
    const dkv_segment& g = entry(i);
    if (g.key_kind == DKV_KEY_DENSE) {
      if (!dense_ok(g)) return DKV_OK;
      continue;
    }
    if (i >= n_rest || !packed_ok(g, (int)a.D)) return DKV_OK;
    if (count == 0) first = i;
    else if (i != first + count || !same_layout(entry(first), g)) return DKV_OK;
    ++count;
  }
  TileParams p;
  p.d = d;
  p.splits = d.splits;
  p.packed_first = first;
  p.n_packed = count;
  // (without packed segments the layout is not used)
  const dkv_segment* g = count ? &entry(first) : nullptr;
  p.key_group = g ? g->key_group : 128;
  p.value_group = g ? g->value_group : 64;
  const bool mixed = g && g->key_kind == DKV_KEY_MIXED;
  p.promoted = mixed ? g->promoted : 0;
  const int bits = g ? g->value_bits : 2;
  *taken = true;
  const bool bf = a.cache_dtype == kBF16;
  if (a.D == 64)
    return bf ? launch_tiles_heads<64, true>(p, bits, mixed, stream)
              : launch_tiles_heads<64, false>(p, bits, mixed, stream);
  return bf ? launch_tiles_heads<128, true>(p, bits, mixed, stream)
            : launch_tiles_heads<128, false>(p, bits, mixed, stream);
}

}  // namespace dkv
