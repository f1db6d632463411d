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
// One wave owns one split, a contiguous range of work items (packed segments,
// pieces of dense ones) of one (batch, kv head), and walks it in tiles of TILE tokens (128, or 64 with 8-bit codes,
// whose registers a larger tile would not leave room for).
//
// Bound by VALU issue and by the latency between a tile's steps at two waves
// per SIMD (three in a few forms; 151 to 256 VGPRs, no private memory: the build
// checks it), not by memory.  Against decode_split_general, which spent about
// 100 VALU per element on scalar index arithmetic (one layer, MI355X): 8
// sequences x 4,096 tokens, 2-bit pages in groups of 64, fp16: 572 -> 19.8 µs; 8
// x 8,011 tokens of Dart pages, six heads per KV head: 1,456 -> 32.9 µs; 16 x
// 4,000 tokens of head_dim 64: 841 -> 24.5 µs.
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
// rounding chain), the query is exact in the operand type, and a softmax weight
// is the sum of three 16-bit parts: exact for bf16 (8 + 8 + 8 bits); for fp16
// (11 + 11 + 2 bits, whose smallest step is fixed) within three steps of 2^-37
// of the running maximum's weight, 2e-7 of the result over 8,192 tokens of one
// split in the worst case, under the rounding of fp32 sums.  The parts of 4
// heads take 12 of the 16 rows of one MFMA (those of 8 heads two MFMAs, of 16
// heads three), and their products meet in the fp32 accumulators when the split
// ends.
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
constexpr int kPiece = 128;         // tokens of a dense work item
constexpr int kMaxGroups = 4;       // key groups per tile, value groups per token
// Natural-log headroom of a weight before the running maximum moves, and the
// power of two weights are scaled by.  fp16's range sets how small a part can
// be: e^2.07 x 2^13 = 64,900 of 65,504.  (With 5.5 and 2^7, steps of 2^-31, the
// error reached 1.7e-5 over 8,192 tokens of one split; with 0.68 and 2^15 the
// maximum moved in most tiles: 1 to 2 % more time.)
template <bool BF> constexpr float kTileSlack = BF ? 5.5f : 2.07f;
template <bool BF> constexpr int kWeightExp = BF ? 0 : 13;

struct TileParams {
  // This kernel's work items (d.n_total of them, dealt to the splits in order)
  // are the packed segments, item i < n_packed being rest entry packed_first + i,
  // then the dense entries' pieces of kPiece tokens: the first piece of each
  // entry, then the second ones (rest entries: the descriptors outside the page
  // kernels' run, then the tail).  A piece is the work of a page, so a long
  // dense window spreads over the splits: with 4,096 tokens beside 64 uniform
  // 4-bit pages of one sequence, eight rows, a call takes 19 µs (as one item
  // 142; the page kernel with its 32-token chunks 54).
  DecodeParams d;
  int packed_first, n_packed, n_dense, splits;
  // what every packed segment shares
  int key_group, value_group, promoted;
  // LDS of one wave (bytes): the key tables, and after Q K the value tables in
  // their place; the weights, before them the scale/zero pairs of a Dart page's
  // channels; the query rows
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
template <class T, int ALIGN = alignof(T)>
__device__ __forceinline__ T gload(const void* base, uint32_t off) {
  typedef T aligned_t __attribute__((aligned(ALIGN)));
  typedef __attribute__((address_space(1))) const uint8_t gbyte;
  typedef __attribute__((address_space(1))) const aligned_t gtype;
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

// A product below 2^32 of factors below 2^24, in one full-rate instruction (a
// 32-bit product takes four).
__device__ __forceinline__ uint32_t mul24(uint32_t a, uint32_t b) { return __umul24(a, b); }

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
// value row) of one K index are NP * BITS / 8 bytes ----
//
// Where that is one or two bytes, neighbouring lanes share their loads: of the
// pair of K indices (k0, k1) the even lane loads k0's and the odd lane k1's
// codes of both lanes' positions, and they exchange halves when the codes are
// used.  (A load each, packed into one register, waits for its data where it is
// issued: the packing cannot leave the load's block.)
template <int BITS, int NP>
struct Codes {
  static constexpr int kBytes = NP * BITS / 8;                    // 1, 2, 4 or 8
  static constexpr bool kShared = kBytes <= 2;
  static constexpr int kPairRegs = kShared ? 1 : kBytes / 2;      // registers of two K indices
  static constexpr int kSpan = kShared ? 2 * NP : NP;             // positions of one load
};

// No value: a register that only one branch of a loop body loads would otherwise
// hold its old contents through the whole body (at sixteen rows the kernel
// spilled up to eight registers).
template <class T>
__device__ __forceinline__ void forget(T& x) { asm volatile("" : "=v"(x)); }
template <class T, int N>
__device__ __forceinline__ void forget(T (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; ++i) forget(x[i]);
}

// Codes of K indices 0 .. NK - 1 of the lane into regs: index k's are at
// base(k) (wave-uniform) + off(k) bytes; a shared load asks for the pair's
// first index, and off adds the odd lane's step.
template <int BITS, int NP, int NK, int N, class Base, class Off>
__device__ __forceinline__ void load_codes(uint32_t (&regs)[N], Base base, Off off) {
  typedef Codes<BITS, NP> C;
  static_assert(N == NK / 2 * C::kPairRegs, "one tile's codes");
#pragma unroll
  for (int p = 0; p < NK / 2; ++p) {
    const uint8_t* a = base(2 * p);
    const uint32_t oa = off(2 * p);
    // (a shared load is aligned to one lane's codes only: value rows of an odd number of them)
    if constexpr (C::kBytes == 1) {
      regs[p] = gload<uint16_t, 1>(a, oa);
    } else if constexpr (C::kBytes == 2) {
      regs[p] = gload<uint32_t, 2>(a, oa);
    } else if constexpr (C::kBytes == 4) {
      regs[2 * p] = gload<uint32_t>(a, oa);
      regs[2 * p + 1] = gload<uint32_t>(base(2 * p + 1), off(2 * p + 1));
    } else {
      const u32x2 x = gload<u32x2>(a, oa), y = gload<u32x2>(base(2 * p + 1), off(2 * p + 1));
      regs[4 * p] = x.x; regs[4 * p + 1] = x.y;
      regs[4 * p + 2] = y.x; regs[4 * p + 3] = y.y;
    }
  }
}

// The other lane's register of a lane pair.
__device__ __forceinline__ uint32_t swap_pair(uint32_t x) {
  return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)x, 0xb1, 0xf, 0xf, true);  // quad_perm 1, 0, 3, 2
}

// Maximum over the 16 lanes of a row.
template <int CTRL>
__device__ __forceinline__ float dpp_max(float x) {
  const int y = __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, x), CTRL, 0xf, 0xf, true);
  return fmaxf(x, __builtin_bit_cast(float, y));
}
__device__ __forceinline__ float max16(float x) {
  x = dpp_max<0xb1>(x);   // lanes 1, 0, 3, 2 of each four
  x = dpp_max<0x4e>(x);   // lanes 2, 3, 0, 1
  x = dpp_max<0x141>(x);  // the other four of eight (row_half_mirror)
  return dpp_max<0x140>(x);  // the other eight (row_mirror)
}

// Selector of unshare() for this lane: its own positions of (k0, k1) as bytes
// (k0, k1, k0, k1), or (k0, k1, 0, 0) where a lane has one byte of each.
template <int BYTES>
__device__ __forceinline__ uint32_t unshare_sel(int lane) {
  if (BYTES == 2) return lane & 1 ? 0x03070206u : 0x05010400u;
  return lane & 1 ? 0x0c0c0105u : 0x0c0c0400u;
}
__device__ __forceinline__ uint32_t unshare(uint32_t x, uint32_t sel) { return perm(swap_pair(x), x, sel); }

// Bytes (k0, k1, k0, k1) at positions j and j + NP / 2 of unshared 2-bit codes.
template <int NP>
__device__ __forceinline__ uint32_t two_bit_bytes(uint32_t y) { return NP == 8 ? y : perm(y >> 4, y, 0x05040100u); }

// Operand dword w (a pair of K indices) at every position j, from 2-bit codes.
// (The dwords of an operand are one vector from the start: gathered from an
// array per pair, they went through private memory at head_dim 64 with up to
// four heads per KV head; 16 x 16,384 tokens, 2-bit pages in groups of 64: 66.0
// -> 44.0 µs.)
template <int NP>
__device__ __forceinline__ void lookup_pair(uint32_t y, uint32_t lo0, uint32_t hi0, uint32_t lo1, uint32_t hi1,
                                            uint32_t m3, uint32_t sel2, u32x4 (&op)[NP], int w) {
#pragma unroll
  for (int j = 0; j < NP / 2; ++j) {
    const uint32_t e = ((y >> (2 * j)) & m3) | sel2;
    const uint32_t l = perm(lo1, lo0, e), h = perm(hi1, hi0, e);
    op[j][w] = perm(h, l, 0x05010400u);
    op[j + NP / 2][w] = perm(h, l, 0x07030602u);
  }
}

// (m & a) | (~m & b), one v_bfi_b32
__device__ __forceinline__ uint32_t bit_select(uint32_t m, uint32_t a, uint32_t b) { return (m & a) | (~m & b); }

// Two code bytes (values below 16) of word half W as an fp16 pair.
template <bool HI>
__device__ __forceinline__ half2v codes16(uint32_t e) {
  return __builtin_bit_cast(half2v, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(e, 512.f, HI));
}

// The same from 4- or 8-bit codes by the arithmetic chain; s, z hold the two
// indices' scales and zero points, sel is the unshare selector.
template <bool BF, int BITS, int NP>
__device__ __forceinline__ void chain_pair(const uint32_t* codes, uint32_t s, uint32_t z, uint32_t sel,
                                           u32x4 (&op)[NP], int w) {
  const half2v sv = __builtin_bit_cast(half2v, s), zv = __builtin_bit_cast(half2v, z);
  auto value = [&](half2v c) {
    const half2v prod = c * sv;  // -ffp-contract=off: one rounding each
    return to_operand<BF>(prod + zv);
  };
  if constexpr (BITS == 4) {
#pragma unroll
    for (int q = 0; q < NP / 4; ++q) {  // four positions: bytes (k0, k1, k0, k1), two positions per byte
      const uint32_t y = NP == 8 ? perm(codes[1], codes[0], q ? 0x07030602u : 0x05010400u) : unshare(codes[0], sel);
      const uint32_t even = y & 0x0f0f0f0fu, odd = (y >> 4) & 0x0f0f0f0fu;
      op[4 * q][w] = value(codes16<false>(even));
      op[4 * q + 1][w] = value(codes16<false>(odd));
      op[4 * q + 2][w] = value(codes16<true>(even));
      op[4 * q + 3][w] = value(codes16<true>(odd));
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
        op[4 * q + j][w] = value(c);
      }
    }
  }
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

// The leading 16-bit parts of two values (rounded toward zero) as operands,
// and what is left of them, exactly: three parts hold an fp32 value (8 + 8 + 8
// bits in bf16, 11 + 11 + 2 in fp16 within its range).
template <bool BF>
__device__ __forceinline__ uint32_t take_part(float x0, float x1, float& r0, float& r1) {
  if constexpr (BF) {
    const uint32_t b0 = __builtin_bit_cast(uint32_t, x0), b1 = __builtin_bit_cast(uint32_t, x1);
    r0 = x0 - __builtin_bit_cast(float, b0 & 0xffff0000u);
    r1 = x1 - __builtin_bit_cast(float, b1 & 0xffff0000u);
    return perm(b1, b0, 0x07060302u);
  } else {
    const auto h = __builtin_amdgcn_cvt_pkrtz(x0, x1);
    r0 = x0 - (float)h[0];
    r1 = x1 - (float)h[1];
    return __builtin_bit_cast(uint32_t, h);
  }
}

// A pair of weight parts, none of them zero: an infinite value times a zero
// part would be NaN where the weight itself is not zero (a zero weight keeps its
// zero first part).  The smallest step, 2^-126 (bf16) or 2^-24 of weights
// scaled by 2^13 (fp16), is below what the sums resolve.
template <bool BF>
constexpr __device__ uint32_t tiny_part() { return BF ? 0x0080u : 0x0001u; }
__device__ __forceinline__ uint32_t at_least(uint32_t x, uint32_t least) {
  typedef uint16_t u16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(u16x2, x), __builtin_bit_cast(u16x2, least)));
}
template <bool BF>
__device__ __forceinline__ uint32_t at_least_tiny(uint32_t x) { return at_least(x, tiny_part<BF>() * 0x10001u); }

// The softmax state and accumulators of a wave, and the steps both kinds of
// tile share.  GP: query rows per KV head rounded up to 4, 8 or 16.  S[j] row 4
// kq + i = head (4 kq + i) % GP, column n = token NJ n + j; O[j] row 4 kq + i =
// weight part and head of that row (head % GP), column n = channel NC n + j.
// PARTS: the query comes in three parts.
template <int D, bool BF, int GP, int TILE, bool PARTS>
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

  const uint8_t* q;  // query rows in LDS: part p of head h at row p GP + h (Dart pages, or more than one part)

  // The lane's A operand of query part `part`, channel block kb.
  __device__ __forceinline__ u32x4 q_part(int part, int kb) const {
    return *(const u32x4*)((const uint16_t*)q + (part * GP + n % GP) * D + 32 * kb + 8 * kq);
  }

  __device__ __forceinline__ void q_products(int kb, const u32x4 (&op)[NJ], float4v (&S)[NJ]) const {
#pragma unroll
    for (int j = 0; j < NJ; ++j) S[j] = mfma<BF>(qa[kb], op[j], S[j]);
    if constexpr (PARTS) {
#pragma unroll
      for (int part = 1; part < 3; ++part) {
        const u32x4 a = q_part(part, kb);
#pragma unroll
        for (int j = 0; j < NJ; ++j) S[j] = mfma<BF>(a, op[j], S[j]);
      }
    }
  }

  // Row 16 pass + r of the weights = part (16 pass + r) / GP of head r % GP.
  // A tile's products meet in T, which the logits no longer need, and are added
  // to O once: straight into an O that a few tokens dominate, the small parts of
  // the others' weights were rounded away (one dominant token, 8,191 of 2^-20 to
  // 2^-29 of its weight in one split: error against 64 bits 2.8e-5).
  __device__ __forceinline__ void p_products(int kb, const u32x4 (&op)[NC], float4v (&T)[NC]) {
#pragma unroll
    for (int pass = 0; pass < PASSES; ++pass) {
      const u32x4 w = *(const u32x4*)(pw + (16 * pass + n) * kPRow + 64 * kb + 16 * kq);
#pragma unroll
      for (int j = 0; j < NC; ++j) T[j] = mfma<BF>(w, op[j], T[j]);
    }
  }
  __device__ __forceinline__ static void clear(float4v (&T)[NC]) {
#pragma unroll
    for (int j = 0; j < NC; ++j) T[j] = float4v{0.f, 0.f, 0.f, 0.f};
  }
  __device__ __forceinline__ void add_tile(const float4v (&T)[NC]) {
#pragma unroll
    for (int j = 0; j < NC; ++j) O[j] += T[j];
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
        over |= v > m_run[i] + kTileSlack<BF>;
      }
    }
    if (__ballot(over) != 0ull) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        float mx = x[0][i];
#pragma unroll
        for (int u = 1; u < U; ++u) mx = fmaxf(mx, x[u][i]);
        mx = max16(mx);
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
    // weights (fp16 operands: times 2^13, undone in the record) and their parts;
    // with 8 heads the last part takes two rows, half of it each
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int head = GP == 4 ? i : GP == 8 ? 4 * (kq & 1) + i : 4 * kq + i;
      float w[U], sum = 0.f;  // (added to l once per tile, as O is)
      const float m_safe = m_run[i] == -INFINITY ? 0.f : m_run[i];  // (no token with a logit above it yet)
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const float dlt = x[u][i] - m_safe;
        w[u] = __builtin_amdgcn_exp2f(BF ? dlt * kLog2e : __builtin_fmaf(dlt, kLog2e, (float)kWeightExp<BF>));
        sum += w[u];
        // a weight below fp16's smallest step, but not zero, gets one (at_least_tiny)
        if (!BF) w[u] = w[u] > 0.f ? fmaxf(w[u], 0x1p-24f) : w[u];
      }
      l_part[i] += sum;
#pragma unroll
      for (int k = 0; k < 3; ++k) {
        uint32_t part[U > 1 ? U / 2 : 1];
#pragma unroll
        for (int u = 0; u < U; u += 2) {
          float w0 = w[u], w1 = U > 1 ? w[(u + 1) % U] : 0.f;
          if (GP == 8 && k == 2) w0 *= 0.5f, w1 *= 0.5f;
          float r0, r1;
          part[u / 2] = take_part<BF>(w0, w1, r0, r1);
          w[u] = r0;
          if (U > 1) w[(u + 1) % U] = r1;
          if (k > 0) part[u / 2] = at_least_tiny<BF>(part[u / 2]);
        }
        auto put = [&](int row) {
          uint8_t* dst = pw + row * kPRow + 2 * (NJ * n + start);
          if constexpr (U == 1) *(uint16_t*)dst = (uint16_t)part[0];
          else if constexpr (U == 2) *(uint32_t*)dst = part[0];
          else if constexpr (U == 4) *(uint2*)dst = make_uint2(part[0], part[1]);
          else *(uint4*)dst = make_uint4(part[0], part[1], part[2], part[3]);
        };
        put(k * GP + head);
        if (GP == 8 && k == 2) put(3 * GP + head);
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
      for (int kb = 0; kb < KB; ++kb) {
        const u32x4 row = gload<u32x4>(k, off + 64 * kb);
        S[j] = mfma<BF>(qa[kb], row, S[j]);
        if constexpr (PARTS) {
          S[j] = mfma<BF>(q_part(1, kb), row, S[j]);
          S[j] = mfma<BF>(q_part(2, kb), row, S[j]);
        }
      }
    }
    softmax(S, nt);
    lds_order();
    float4v T[NC];
    clear(T);
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
          T[j] = mfma<BF>(w, u32x4{perm(r[1][j / 2], r[0][j / 2], sel), perm(r[3][j / 2], r[2][j / 2], sel),
                                   perm(r[5][j / 2], r[4][j / 2], sel), perm(r[7][j / 2], r[6][j / 2], sel)}, T[j]);
        }
      }
    }
    add_tile(T);
    lds_order();
  }
};

// KBITS: key code width; MIXED: Dart pages (KBITS 2); VBITS: value code width;
// PARTS: the query is of another type than the cache.
template <int D, bool BF, int GP, int KBITS, bool MIXED, int VBITS, bool PARTS>
__global__ void __launch_bounds__(64 * kTileWaves, 2) decode_tiles(TileParams p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  constexpr int TILE = KBITS == 8 || VBITS == 8 ? 64 : 128;
  typedef TileState<D, BF, GP, TILE, PARTS> St;
  constexpr int NJ = St::NJ, NC = St::NC, KB = St::KB, VB = St::VB, PASSES = St::PASSES;
  constexpr int KK = D / 4, VK = TILE / 4;  // K indices of a lane
  constexpr int KSTEP = D / 64, VSTEP = TILE / 64;       // table items of a lane per group
  constexpr int KIT = 2 * KSTEP, VIT = 2 * VSTEP;        // ... that wait in registers: two groups' (the others
                                                         // are loaded when their tables are made)
  // Forms whose registers are full form the lane's coordinates anew for each
  // tile: the addresses made from them would otherwise be kept from tile to tile
  // and spilled (elsewhere this costs 2 %).
  constexpr bool kRederive = D == 128 && GP >= 8 && (MIXED || (GP == 16 && KBITS == 4));
  constexpr int kTabK = D * 8 + 16, kTabV = TILE * 8 + 16;
  typedef Codes<KBITS, NJ> KC;
  typedef Codes<VBITS, NC> VC;
  const DecodeParams& d = p.d;
  const dkv_decode_args& a = d.a;
  int lane = threadIdx.x & 63;
  const int wave = uni(threadIdx.x >> 6);
  int n = lane & 15, kq = lane >> 4;
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
  const uint32_t ksel = unshare_sel<KC::kBytes>(lane), vsel = unshare_sel<VC::kBytes>(lane);
  int odd = lane & 1;
  const int kgroup = p.key_group, vgroup = p.value_group, promoted = p.promoted;
  const int Gv = groups_of(D, vgroup), vrow = Gv * vgroup * VBITS / 8;

  // ---- the query: A operands of row n (head n % GP, zero past G), and its
  // rows in LDS for the promoted channels and for further parts ----
  St st;
  st.n = n;
  st.kq = kq;
  st.pw = lds + p.pw;
  st.q = lds + p.q;
  st.scale = (float)a.scale;
  {
    const int head = n % GP;
    const int64_t at = (int64_t)b * a.q_sb + (int64_t)(kvh * G + (head < G ? head : 0)) * a.q_sh;
    if constexpr (!PARTS) {
      const uint16_t* q = (const uint16_t*)a.query + at;
      // Aligned heads take one load per 32 channels in place of eight: a wave has
      // few tiles, so what it does once counts (with the records below stored
      // 16 bytes at a time, six heads per KV head: 34.6 -> 32.3 µs; one tile per
      // wave 21.0 -> 19.8).
      if ((((uint64_t)(uintptr_t)a.query | 2 * (uint64_t)(a.q_sb | a.q_sh)) & 15) == 0) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) st.qa[kb] = gload<u32x4>(q, 2 * (32 * kb + 8 * kq));
      } else {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const int c = 32 * kb + 8 * kq + 2 * w;
            st.qa[kb][w] = (uint32_t)gload<uint16_t>(q, 2 * c) | ((uint32_t)gload<uint16_t>(q, 2 * c + 2) << 16);
          }
        }
      }
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
#pragma unroll
        for (int w = 0; w < 4; ++w) st.qa[kb][w] = head < G ? st.qa[kb][w] : 0u;
        if (MIXED && n < GP) *(u32x4*)(lds + p.q + 2 * (n * D + 32 * kb + 8 * kq)) = st.qa[kb];
      }
    } else {
      // a query of another type as the exact sum of three parts; for fp16
      // operands it is scaled by a power of two that the logit scale takes back
      float x[8 * KB];
#pragma unroll
      for (int i = 0; i < 8 * KB; ++i) {
        x[i] = dev_load(a.query, at + 32 * (i >> 3) + 8 * kq + (i & 7), (int)a.q_dtype);
        x[i] = head < G ? x[i] : 0.f;
      }
      const int e = BF ? 0 : query_exponent(x);
      st.scale = ldexpf(st.scale, e);
#pragma unroll
      for (int i = 0; i < 8 * KB; ++i) x[i] = ldexpf(x[i], -e);
      // a part that is zero where the element is not gets the smallest step and
      // the element's sign: an infinite key times a zero part would be NaN
      uint32_t sign[4 * KB], least[4 * KB];
#pragma unroll
      for (int i = 0; i < 4 * KB; ++i) {
        const uint32_t b0 = __builtin_bit_cast(uint32_t, x[2 * i]), b1 = __builtin_bit_cast(uint32_t, x[2 * i + 1]);
        sign[i] = perm(b1, b0, 0x07060302u) & 0x80008000u;
        least[i] = (x[2 * i] != 0.f ? tiny_part<BF>() : 0u) | (x[2 * i + 1] != 0.f ? tiny_part<BF>() << 16 : 0u);
      }
#pragma unroll
      for (int part = 0; part < 3; ++part) {
#pragma unroll
        for (int kb = 0; kb < KB; ++kb) {
          u32x4 row;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            float &x0 = x[8 * kb + 2 * w], &x1 = x[8 * kb + 2 * w + 1];
            float r0, r1;
            row[w] = take_part<BF>(x0, x1, r0, r1);
            x0 = r0;
            x1 = r1;
            row[w] = sign[4 * kb + w] | at_least(row[w] & 0x7fff7fffu, least[4 * kb + w]);
          }
          if (part == 0) st.qa[kb] = row;
          if (n < GP) *(u32x4*)(lds + p.q + 2 * ((part * GP + n) * D + 32 * kb + 8 * kq)) = row;
        }
      }
    }
  }
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
    uint16_t ks[KIT], kz[KIT], vs[VIT], vz[VIT];  // its scales and zero points
    int kidx[4];  // its promoted channels: slots 8 kq + 2 w + odd of the first block
    int zidx;     // ... and slot `lane`
    auto load_keys = [&](const Packed& t, int t0) {
      const int Gp = groups_of(t.tokens, kgroup), padded = Gp * kgroup;
      const int row = padded * KBITS / 8;  // bytes of a channel
      constexpr int span = KC::kSpan;
      const int at = KC::kShared ? n >> 1 : n;
      const int first = min(t0 + span * at, padded - span);  // a lane past the page repeats its last tokens
      const uint32_t off = (uint32_t)(first * KBITS / 8) + mul24(8 * kq + (KC::kShared ? odd : 0), row);
      load_codes<KBITS, NJ, KK>(
          kc, [&](int k) { return t.k + (32 * (k >> 3) + (k & 7)) * row; }, [&](int) { return off; });
      const int g0 = t0 / kgroup, ng = min(Gp - g0, max(1, TILE / kgroup));
#pragma unroll
      for (int m = 0; m < KIT; ++m) {
        forget(ks[m]);
        forget(kz[m]);
        if (m / KSTEP < ng) {
          const int step = 64 * (m % KSTEP) * Gp + g0 + m / KSTEP;
          ks[m] = gload<uint16_t>(t.ks + step, mul24(2 * lane, Gp));
          kz[m] = gload<uint16_t>(t.kz + step, mul24(2 * lane, Gp));
        }
      }
      if constexpr (MIXED) {
#pragma unroll
        for (int w = 0; w < 4; ++w) kidx[w] = gload<int>(t.ki, 4 * min(8 * kq + 2 * w + odd, promoted - 1));
        zidx = gload<int>(t.ki, 4 * min(lane, promoted - 1));
      }
    };
    auto load_values = [&](const Packed& t, int t0) {
      const int last = t.tokens - 1;
      const uint32_t col = (uint32_t)(VC::kSpan * (VC::kShared ? n >> 1 : n) * VBITS / 8);
      const int step = VC::kShared ? odd : 0;
      if (t0 + TILE <= t.tokens) {  // a whole tile's addresses step by the row
        const uint32_t off = col + mul24(8 * kq + step, vrow);
        load_codes<VBITS, NC, VK>(
            vc, [&](int k) { return t.v + (t0 + 32 * (k >> 3) + (k & 7)) * vrow; }, [&](int) { return off; });
#pragma unroll
        for (int m = 0; m < VIT; ++m) {
          forget(vs[m]);
          forget(vz[m]);
          if (m / VSTEP < Gv) {
            const int item = (t0 + 64 * (m % VSTEP)) * Gv + m / VSTEP;
            vs[m] = gload<uint16_t>(t.vs + item, mul24(2 * lane, Gv));
            vz[m] = gload<uint16_t>(t.vz + item, mul24(2 * lane, Gv));
          }
        }
      } else {  // a partial one repeats its last token
        load_codes<VBITS, NC, VK>(
            vc, [&](int) { return t.v; },
            [&](int k) { return col + mul24(min(t0 + 32 * (k >> 3) + 8 * kq + (k & 7) + step, last), vrow); });
#pragma unroll
        for (int m = 0; m < VIT; ++m) {
          forget(vs[m]);
          forget(vz[m]);
          if (m / VSTEP < Gv) {
            const uint32_t item = 2 * (mul24(min(t0 + lane + 64 * (m % VSTEP), last), Gv) + m / VSTEP);
            vs[m] = gload<uint16_t>(t.vs, item);
            vz[m] = gload<uint16_t>(t.vz, item);
          }
        }
      }
    };
    auto no_keys = [&] {
      forget(kc);
      forget(ks);
      forget(kz);
      forget(kidx);
      forget(zidx);
    };
    auto no_values = [&] {
      forget(vc);
      forget(vs);
      forget(vz);
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
      if constexpr (kRederive) {
        asm volatile("" : "+v"(lane));
        n = st.n = lane & 15;
        kq = st.kq = lane >> 4;
        odd = lane & 1;
      }
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
      // codes of the promoted slots 32 block + 8 kq + 2 w + odd, shared as the others are
      const uint32_t tok_off = (uint32_t)(min(cur0 + 2 * NJ * (n >> 1), Gp * kgroup - 2 * NJ) / 4);
      uint32_t pl[4], ph[4];
      auto load_promoted = [&](int block, const int (&idx)[4]) {
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const int slot = min(32 * block + 8 * kq + 2 * w + odd, promoted - 1);
          const uint32_t la = mul24(idx[w] & (D - 1), row) + tok_off, ha = mul24(slot, row) + tok_off;
          pl[w] = NJ == 8 ? gload<uint32_t>(cur.k, la) : (uint32_t)gload<uint16_t>(cur.k, la);
          ph[w] = NJ == 8 ? gload<uint32_t>(cur.kh, ha) : (uint32_t)gload<uint16_t>(cur.kh, ha);
        }
      };
      if constexpr (MIXED) load_promoted(0, kidx);
      auto key_item = [&](int m, uint32_t sz) {
        const int c = lane + 64 * (m % KSTEP), g = m / KSTEP;
        put_table<BF>(lds + p.kt + g * kTabK, c, sz, KBITS == 2);
        if (MIXED) *(uint32_t*)(lds + p.sz + 4 * (g * D + c)) = sz;
      };
#pragma unroll
      for (int m = 0; m < KIT; ++m)
        if (m / KSTEP < ng) key_item(m, ks[m] | ((uint32_t)kz[m] << 16));
#pragma unroll 1
      for (int m = KIT; m < ng * KSTEP; ++m) {
        const uint32_t at = 2 * ((lane + 64 * (m % KSTEP)) * Gp + g0 + m / KSTEP);
        key_item(m, gload<uint16_t>(cur.ks, at) | ((uint32_t)gload<uint16_t>(cur.kz, at) << 16));
      }
      if constexpr (MIXED) {  // promoted channels take the 4-bit pass: their 2-bit tables become zero
        lds_order();
#pragma unroll 1
        for (int j = lane; j < promoted; j += 64) {
          const int c = (j == lane ? zidx : gload<int>(cur.ki, 4 * j)) & (D - 1);
#pragma unroll 1
          for (int g = 0; g < ng; ++g) *(uint2*)(lds + p.kt + g * kTabK + 8 * c) = make_uint2(0u, 0u);
        }
      }
      lds_order();

      // ---- S = Q K ----
      float4v S[NJ];
#pragma unroll
      for (int j = 0; j < NJ; ++j) S[j] = float4v{0.f, 0.f, 0.f, 0.f};
      const uint8_t* ktab = lds + p.kt + lane_group * kTabK;
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        u32x4 op[NJ];
        const uint4* tab = (const uint4*)(ktab + (KBITS == 2 ? 8 : 4) * (32 * kb + 8 * kq));
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if constexpr (KBITS == 2) {
            const uint4 tt = tab[w];
            lookup_pair<NJ>(two_bit_bytes<NJ>(unshare(kc[4 * kb + w], ksel)), tt.x, tt.y, tt.z, tt.w, m3, sel2, op, w);
          } else {
            const uint4 tt = tab[w / 2];
            chain_pair<BF, KBITS, NJ>(&kc[KC::kPairRegs * (4 * kb + w)], w % 2 ? tt.z : tt.x, w % 2 ? tt.w : tt.y, ksel,
                                      op, w);
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
            for (int w = 0; w < 4; ++w) kidx[w] = gload<int>(cur.ki, 4 * min(32 * block + 8 * kq + 2 * w + odd, promoted - 1));
            load_promoted(block, kidx);
          }
          // slots past the last one: zero query, zero scale and zero point
          const bool whole = 32 * block + 32 <= promoted;
          u32x4 op[NJ];
          u32x4 qp[PARTS ? 3 : 1];
          const uint32_t* sz = (const uint32_t*)(lds + p.sz) + lane_group * D;
#pragma unroll
          for (int w = 0; w < 4; ++w) {
            const int own = kidx[w] & (D - 1), next = (int)swap_pair((uint32_t)own);
            const int c0 = odd ? next : own, c1 = odd ? own : next, slot = 32 * block + 8 * kq + 2 * w;
#pragma unroll
            for (int part = 0; part < (PARTS ? 3 : 1); ++part) {
              const uint16_t* q = (const uint16_t*)(lds + p.q) + (part * GP + n % GP) * D;
              uint32_t v = q[c0] | ((uint32_t)q[c1] << 16);
              if (!whole) v &= (slot < promoted ? 0xffffu : 0u) | (slot + 1 < promoted ? 0xffff0000u : 0u);
              qp[part][w] = v;
            }
            uint32_t mine = sz[own];
            if (!whole) mine = slot + odd < promoted ? mine : 0u;
            const uint32_t other = swap_pair(mine);
            // (s0, s1) and (z0, z1): the even lane's first
            const half2v s = __builtin_bit_cast(half2v, perm(other, mine, odd ? 0x01000504u : 0x05040100u));
            const half2v z = __builtin_bit_cast(half2v, perm(other, mine, odd ? 0x03020706u : 0x07060302u));
            const uint32_t yl = two_bit_bytes<NJ>(unshare(pl[w], ksel)), yh = two_bit_bytes<NJ>(unshare(ph[w], ksel));
            // nibbles of positions j and j + 2 (even) and j + 1 and j + 3 (odd) per byte, from both planes
            const uint32_t even = bit_select(0x33333333u, yl, yh << 2), oddn = bit_select(0x33333333u, yl >> 2, yh);
#pragma unroll
            for (int j = 0; j < NJ / 2; ++j) {
              const uint32_t e = ((j & 1 ? oddn : even) >> (4 * (j >> 1))) & 0x0f0f0f0fu;
              const half2v x = codes16<false>(e) * s, y = codes16<true>(e) * s;
              op[j][w] = to_operand<BF>(x + z);
              op[j + NJ / 2][w] = to_operand<BF>(y + z);
            }
          }
#pragma unroll
          for (int part = 0; part < (PARTS ? 3 : 1); ++part) {
#pragma unroll
            for (int j = 0; j < NJ; ++j) S[j] = mfma<BF>(qp[part], op[j], S[j]);
          }
        }
      }
      no_keys();
      if (live) load_keys(nxt, t0);
      lds_order();
      st.softmax(S, nt);

      // ---- value tables (tokens past the tile's end: zero) ----
      auto value_item = [&](int m, uint32_t sz) {
        const int tok = lane + 64 * (m % VSTEP);
        put_table<BF>(lds + p.vt + (m / VSTEP) * kTabV, tok, tok < nt ? sz : 0u, VBITS == 2);
      };
#pragma unroll
      for (int m = 0; m < VIT; ++m)
        if (m / VSTEP < Gv) value_item(m, vs[m] | ((uint32_t)vz[m] << 16));
#pragma unroll 1
      for (int m = VIT; m < Gv * VSTEP; ++m) {
        const uint32_t at = 2 * ((cur0 + min(lane + 64 * (m % VSTEP), nt - 1)) * Gv + m / VSTEP);
        value_item(m, gload<uint16_t>(cur.vs, at) | ((uint32_t)gload<uint16_t>(cur.vz, at) << 16));
      }
      lds_order();

      // ---- O += P V ----
      float4v T[NC];
      St::clear(T);
#pragma unroll
      for (int kb = 0; kb < VB; ++kb) {
        u32x4 op[NC];
        const uint4* tab = (const uint4*)(vtab + (VBITS == 2 ? 8 : 4) * (32 * kb + 8 * kq));
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          if constexpr (VBITS == 2) {
            const uint4 tt = tab[w];
            lookup_pair<NC>(two_bit_bytes<NC>(unshare(vc[4 * kb + w], vsel)), tt.x, tt.y, tt.z, tt.w, m3, sel2, op, w);
          } else {
            const uint4 tt = tab[w / 2];
            chain_pair<BF, VBITS, NC>(&vc[VC::kPairRegs * (4 * kb + w)], w % 2 ? tt.z : tt.x, w % 2 ? tt.w : tt.y, vsel,
                                      op, w);
          }
        }
        st.p_products(kb, op, T);
      }
      st.add_tile(T);
      no_values();
      if (live) load_values(nxt, t0);
      lds_order();
    }
  }

  // ---- dense pieces ----
  bool seen = s0 < min(s1, p.n_packed);  // the split has tokens
  const int n_rest = (int)a.n_segments - d.skip_count;
#pragma unroll 1
  for (int i = max(s0, p.n_packed); i < s1; ++i) {
    const int j = i - p.n_packed, piece = uni(j / p.n_dense), entry = uni(j % p.n_dense);
    const int e = entry < p.packed_first ? entry : entry + p.n_packed;
    int tokens;
    uint64_t k, v;
    bool dense = true;
    if (e < n_rest) {
      const_segment& s = rest_entry(d, e);
      tokens = s.tokens;
      dense = s.key_kind == DKV_KEY_DENSE && s.value_kind == DKV_VALUE_DENSE;
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
    const int first = piece * kPiece;
    tokens = uni(min(tokens - first, kPiece));
    k += (uint64_t)first * (2 * D);
    v += (uint64_t)first * (2 * D);
    seen |= tokens > 0;
    if (!dense) {  // (a caller that passed no host copy of the descriptors to check): a NaN record
      st.m_run[0] = st.m_run[1] = st.m_run[2] = st.m_run[3] = NAN;
      tokens = 0;
    }
#pragma unroll 1
    for (int at = 0; at < tokens; at += TILE)
      st.dense_tile((const uint16_t*)uniform_u64(k), (const uint16_t*)uniform_u64(v), at, min(TILE, tokens - at));
  }

  // ---- partial state ----
  constexpr float unscale = 1.f / (1 << kWeightExp<BF>);
  float* ws = (float*)a.workspace;
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
      rec[1] = seen && st.m_run[i] == -INFINITY ? kNoWeight : l * unscale;
    }
    float o[NC];
#pragma unroll
    for (int j = 0; j < NC; ++j) {
      o[j] = GP == 4 && kq == 3 ? 0.f : st.O[j][i];  // (the fourth part's rows hold nothing)
      if (GP == 4) o[j] += __shfl_xor(o[j], 16, 64);
      if (GP <= 8) o[j] += __shfl_xor(o[j], 32, 64);
    }
    if (writes) {  // one test for all channels: they are stored together
#pragma unroll
      for (int j = 0; j < NC; ++j) rec[2 + NC * n + j] = o[j] * unscale;
    }
  }
}

bool dense_ok(const dkv_segment& g) {
  return g.tokens < (1 << 20) && g.value_kind == DKV_VALUE_DENSE && g.key[0] % 16 == 0 && (2 * g.key_bh[0]) % 16 == 0 &&
         g.value[0] % 16 == 0 && (2 * g.value_bh[0]) % 16 == 0;
}

// Whether the tile kernel reads this packed segment (host).  The bounds on its
// tokens and groups (a page of any size in use has far smaller ones) keep the
// kernel's 32-bit offsets in range: a key row is at most 2^17 bytes, a segment's
// values at most 2^28.
bool packed_ok(const dkv_segment& g, int D) {
  if (g.tokens < 1 || g.tokens > (1 << 16) || g.key_group > (1 << 16) || g.value_group > (1 << 12)) return false;
  if (g.value_kind != DKV_VALUE_UNIFORM) return false;
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

template <int D, bool BF, int GP, int KBITS, bool MIXED, bool PARTS = false>
int launch_tiles(TileParams& p, hipStream_t s) {
  constexpr int TILE = KBITS == 8 ? 64 : 128;
  typedef TileState<D, BF, GP, TILE, PARTS> St;
  const int kgroups = p.key_group >= TILE ? 1 : TILE / p.key_group;
  const int vgroups = (D + p.value_group - 1) / p.value_group;
  int o = 0;
  p.kt = p.vt = o; o += std::max(kgroups * (D * 8 + 16), vgroups * (TILE * 8 + 16));
  p.pw = p.sz = o; o += std::max(16 * St::PASSES * St::kPRow, MIXED ? kgroups * D * 4 : 0);
  p.q = o; o += MIXED || PARTS ? (PARTS ? 3 : 1) * GP * D * 2 : 0;
  p.wave_bytes = o;
  const int64_t workers = p.d.a.B * p.d.a.Hkv * p.splits;
  const dim3 grid((unsigned)((workers + kTileWaves - 1) / kTileWaves));
  hipLaunchKernelGGL((decode_tiles<D, BF, GP, KBITS, MIXED, KBITS, PARTS>), grid, dim3(64 * kTileWaves),
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

// Both sides measured, one layer with its merge (tile | page kernel, MI355X):
// * Dart pages, sixteen rows (the page kernel has no such form any more): 8 x 8
//   heads x 64 pages 37 | 71 µs.  Up to four rows the page kernel, whose staged
//   pages serve every row, is the faster everywhere: four rows, 64 x 8 x 255
//   pages 524 | 424, 16 x 8 x 64 51 | 40, one sequence x 8 pages 15.1 | 12.2; one
//   row 521 | 393, 50 | 36, 14.8 | 12.9.  Eight rows are even (582 | 532, 55 | 53,
//   15.1 | 16.6) and stay with it.
// * Uniform pages of one code width, eight rows: 16 x 8 heads x 128 pages 104 |
//   127 µs at 4 bits, 69 | 122 at 2 bits, 151 | 191 at 8 bits; one sequence x 8
//   pages at 2 bits 14.1 | 17.5, at 8 bits 19.1 | 17.9.
// * Fewer rows, where the launch fills the device.  The page kernel's work grows
//   with the rows, the tile kernel's hardly does; its bf16 rounding chain is the
//   dearer one, and a launch pays for its prologue.  2 bits: one row, 64 x 8 x
//   255 pages 400 | 637, 16 x 8 x 64 40 | 48, but 16 pages (every wave has one, and
//   the dense pieces start a second round of waves) 23 | 21.  4 bits in value
//   groups of 32 channels: 676 | 1,036, 26 | 30; else fp16 with one row 494 | 624,
//   50 | 52, but 32 pages 31 | 30; bf16 with four rows 608 | 675, 16 x 8 x 128
//   pages 95 | 98, but 64 pages 55 | 54, with one row 590 | 651, but 16 x 8 x 128
//   93 | 90.  8 bits: bf16 with two rows 938 | 1,075, 84 | 87, with one 934 |
//   1,041, but 64 pages 83 | 82; fp16 with four rows 913 | 871, but 24 pages 36 | 40.
bool tiles_take_run(const dkv_decode_args& a, int group) {
  if (a.fast_promoted > 0) return group == 16;
  if (a.q_dtype != a.cache_dtype || a.fast_key_bits != a.fast_value_bits || 128 / a.fast_value_group > kMaxGroups)
    return false;
  const int64_t pages = a.B * a.Hkv * a.fast_count, bits = a.fast_key_bits;
  constexpr int64_t kFull = 2048;  // waves the device holds
  if (group >= 8) return bits < 8 || pages >= kFull;
  if (pages < kFull) return false;
  const bool bf = a.cache_dtype == kBF16, more = pages > kFull;
  if (bits == 2) return group == 4 || more;
  if (bits == 4 && a.fast_value_group == 32) return true;
  if (bits == 4 && bf) return pages >= (group == 4 ? 8 : 32) * kFull;
  if (bits == 4) return group == 4 || (group == 2 && more) || pages >= 4 * kFull;
  if (bf) return group >= 2 || pages >= 16 * kFull;
  return group >= 2 && pages <= kFull * 3 / 2;
}

int tile_items(int count, int n_dense, int64_t dense_tokens) {
  return (int)std::min<int64_t>(INT32_MAX, count + n_dense * ((dense_tokens + kPiece - 1) / kPiece));
}

int launch_tile_run(const DecodeParams& d, int first, int count, int n_dense, int splits, const TileLayout& g,
                    hipStream_t s) {
  const dkv_decode_args& a = d.a;
  DKV_CHECK(a.B * a.Hkv * splits < (int64_t)1 << 31, DKV_ERR_UNSUPPORTED, "too many splits for one launch");
  TileParams p;
  p.d = d;
  p.splits = splits;
  p.packed_first = first;
  p.n_packed = count;
  p.n_dense = n_dense;
  p.key_group = g.key_group;
  p.value_group = g.value_group;
  p.promoted = g.promoted;
  const bool mixed = g.promoted > 0, bf = a.cache_dtype == kBF16;
  if (a.q_dtype != a.cache_dtype)  // (16 heads on Dart pages: tiles_take_run)
    return bf ? launch_tiles<128, true, 16, 2, true, true>(p, s) : launch_tiles<128, false, 16, 2, true, true>(p, s);
  if (a.D == 64)
    return bf ? launch_tiles_heads<64, true>(p, g.bits, mixed, s) : launch_tiles_heads<64, false>(p, g.bits, mixed, s);
  return bf ? launch_tiles_heads<128, true>(p, g.bits, mixed, s) : launch_tiles_heads<128, false>(p, g.bits, mixed, s);
}

bool tiles_take_rest(const DecodeParams& d, TileRest* rest) {
  const dkv_decode_args& a = d.a;
  if ((a.cache_dtype != kBF16 && a.cache_dtype != kF16) || a.q_dtype != a.cache_dtype || a.meta_dtype != kF16)
    return false;
  if ((a.D != 64 && a.D != 128) || d.group > 16 || (a.n_segments > 0 && a.segments_host == nullptr)) return false;
  if (a.B * a.Hkv * d.splits >= (int64_t)1 << 31) return false;
  const int n_rest = (int)a.n_segments - d.skip_count;
  auto entry = [&](int i) -> const dkv_segment& {
    return i >= n_rest ? a.tail : a.segments_host[i < d.skip_first ? i : i + d.skip_count];
  };
  // one run of packed segments of one layout, everything else dense
  int most = 0;  // tokens of a dense entry
  *rest = TileRest{0, 0, 0, 0, TileLayout{2, 128, 64, 0}};  // (without packed segments the layout is not used)
  for (int i = 0; i < d.n_total; ++i) {
    const dkv_segment& g = entry(i);
    if (g.key_kind == DKV_KEY_DENSE) {
      if (!dense_ok(g)) return false;
      most = std::max(most, g.tokens);
      continue;
    }
    if (i >= n_rest || !packed_ok(g, (int)a.D)) return false;
    if (rest->count == 0) {
      rest->first = i;
      rest->layout =
          TileLayout{g.value_bits, g.key_group, g.value_group, g.key_kind == DKV_KEY_MIXED ? g.promoted : 0};
    } else if (i != rest->first + rest->count || !same_layout(entry(rest->first), g)) {
      return false;
    }
    ++rest->count;
  }
  rest->n_dense = d.n_total - rest->count;
  rest->items = tile_items(rest->count, rest->n_dense, most);
  return true;
}

}  // namespace dkv
