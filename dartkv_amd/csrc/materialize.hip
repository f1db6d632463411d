// A cache's contents as dense K and V in one launch (gfx950): every segment of
// every (batch, kv head) dequantized, or copied, straight to its tokens of the
// two [B][H][tokens][D] outputs (reference src/dart/cache.py:192-204: each
// segment dequantized, src/dart/quantization.py:96-109 and
// src/dart/mixed.py:72-94, then concatenated).
//
// Bound by the outputs' stores: about 4 bytes written per byte read at 2 bits.
// One workgroup per (128-token chunk, batch, kv head) and side, which gives
// 4,096 workgroups at 8 x 8 heads x 4,096 tokens.  A lane owns 8 channels x 8
// tokens of a key chunk (codes are packed along the tokens: one load of 2, 4 or
// 8 bytes per channel, the metadata of the eight channels in one load each where
// a page is one group) and 8 channels of a value row, so every store is 16
// bytes and 16 lanes write one 256-byte row; the values are transposed in
// registers.  One launch per segment, a copy of each transposed result and the
// concatenation took 1,810 µs there; this kernel takes 39 µs (4.1 TB/s of packed
// bytes read and dense bytes written; a fill of the outputs takes 20) and the
// call 55.  With a load of its own for each channel's scale and zero point it
// took 51.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "dkv_capi_util.h"
#include "dkv_dense.h"
#include "dkv_device.h"

using namespace dkv;

namespace {

constexpr int kThreads = 256;
constexpr int kChunk = 128;

typedef _Float16 half2v __attribute__((ext_vector_type(2)));

// Eight fp16 values (the rounding chain's sums, as pairs) to out[at ..].
template <int OUT>
__device__ __forceinline__ void store8(void* out, int64_t at, const half2v (&v)[4]) {
  if constexpr (OUT == kF32) {
    float4* o = (float4*)((float*)out + at);
    o[0] = make_float4((float)v[0][0], (float)v[0][1], (float)v[1][0], (float)v[1][1]);
    o[1] = make_float4((float)v[2][0], (float)v[2][1], (float)v[3][0], (float)v[3][1]);
  } else if constexpr (OUT == kF16) {
    *(uint4*)((_Float16*)out + at) =
        make_uint4(__builtin_bit_cast(uint32_t, v[0]), __builtin_bit_cast(uint32_t, v[1]),
                   __builtin_bit_cast(uint32_t, v[2]), __builtin_bit_cast(uint32_t, v[3]));
  } else {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    uint32_t w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k)
      w[k] = __builtin_bit_cast(uint32_t, __builtin_convertvector((f32x2){(float)v[k][0], (float)v[k][1]}, bf16x2));
    *(uint4*)((uint16_t*)out + at) = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

__device__ __forceinline__ half2v half_pair(uint32_t a, uint32_t b) {
  return half2v{(_Float16)(uint16_t)a, (_Float16)(uint16_t)b};
}
__device__ __forceinline__ _Float16 as_half(uint16_t x) { return __builtin_bit_cast(_Float16, x); }

// Eight consecutive codes at p (2, 4 or 8 bytes).
template <int BITS>
__device__ __forceinline__ uint64_t codes8(const uint8_t* p) {
  if constexpr (BITS == 2) return *(const uint16_t*)p;
  else if constexpr (BITS == 4) return *(const uint32_t*)p;
  else return *(const uint64_t*)p;
}
template <int BITS>
__device__ __forceinline__ uint32_t code_at(uint64_t w, int j) {
  if constexpr (BITS == 8) return (uint32_t)(w >> (8 * j)) & 255u;
  else return ((uint32_t)w >> (BITS * j)) & ((1u << BITS) - 1u);
}

// Keys of tokens t0 .. t0 + nt - 1 of a packed segment to out (row 0 = token
// t0).  inv: slot of each channel among the promoted ones, -1 for none.
template <int BITS, bool MIXED, int OUT>
__device__ __forceinline__ void key_chunk(const dkv_segment& s, int64_t bh, int D, int t0, int nt, const int16_t* inv,
                                          void* out, int64_t out0) {
  const int kg = s.key_group, G = (s.tokens + kg - 1) / kg, row = G * kg * BITS / 8, d8 = D / 8;
  const uint8_t* low = (const uint8_t*)s.key[0] + bh * s.key_bh[0];
  const uint8_t* high = (const uint8_t*)s.key[1] + bh * s.key_bh[1];
  const uint16_t* scale = (const uint16_t*)s.key[3] + bh * s.key_bh[3];
  const uint16_t* zero = (const uint16_t*)s.key[4] + bh * s.key_bh[4];
  // one group per page and aligned rows: eight channels' metadata in one load
  const bool meta8 = G == 1 && ((s.key[3] | s.key[4] | 2 * (uint64_t)(s.key_bh[3] | s.key_bh[4])) & 15) == 0;
  for (int i = threadIdx.x; i < d8 * ((nt + 7) / 8); i += kThreads) {
    const int c0 = 8 * (i % d8), at = 8 * (i / d8), t = t0 + at, g = t / kg;
    uint64_t w[8], h[8];
    half2v sv[4], zv[4];
    if (meta8) {
      const uint4 sw = *(const uint4*)(scale + c0), zw = *(const uint4*)(zero + c0);
      sv[0] = __builtin_bit_cast(half2v, sw.x); sv[1] = __builtin_bit_cast(half2v, sw.y);
      sv[2] = __builtin_bit_cast(half2v, sw.z); sv[3] = __builtin_bit_cast(half2v, sw.w);
      zv[0] = __builtin_bit_cast(half2v, zw.x); zv[1] = __builtin_bit_cast(half2v, zw.y);
      zv[2] = __builtin_bit_cast(half2v, zw.z); zv[3] = __builtin_bit_cast(half2v, zw.w);
    }
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      const int c = c0 + k;
      w[k] = codes8<BITS>(low + (int64_t)c * row + t * BITS / 8);
      h[k] = 0;
      if constexpr (MIXED) {
        const int slot = inv[c];
        if (slot >= 0) h[k] = codes8<2>(high + (int64_t)slot * row + t / 4);
      }
      if (!meta8) {
        sv[k / 2][k % 2] = as_half(scale[c * G + g]);
        zv[k / 2][k % 2] = as_half(zero[c * G + g]);
      }
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      half2v v[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        uint32_t a = code_at<BITS>(w[2 * k], j), b = code_at<BITS>(w[2 * k + 1], j);
        if constexpr (MIXED) {
          a |= code_at<2>(h[2 * k], j) << 2;
          b |= code_at<2>(h[2 * k + 1], j) << 2;
        }
        const half2v prod = half_pair(a, b) * sv[k];  // -ffp-contract=off: one rounding each
        v[k] = prod + zv[k];
      }
      if (at + j < nt) store8<OUT>(out, (out0 + at + j) * D + c0, v);
    }
  }
}

template <int BITS, int OUT>
__device__ __forceinline__ void value_chunk(const dkv_segment& s, int64_t bh, int D, int t0, int nt, void* out,
                                            int64_t out0) {
  const int vg = s.value_group, G = (D + vg - 1) / vg, row = G * vg * BITS / 8, d8 = D / 8;
  const uint8_t* codes = (const uint8_t*)s.value[0] + bh * s.value_bh[0];
  const uint16_t* scale = (const uint16_t*)s.value[1] + bh * s.value_bh[1];
  const uint16_t* zero = (const uint16_t*)s.value[2] + bh * s.value_bh[2];
#pragma unroll 4
  for (int i = threadIdx.x; i < d8 * nt; i += kThreads) {
    const int c0 = 8 * (i % d8), at = i / d8, t = t0 + at;
    const uint64_t w = codes8<BITS>(codes + (int64_t)t * row + c0 * BITS / 8);
    const _Float16 s1 = as_half(scale[t * G + c0 / vg]), z1 = as_half(zero[t * G + c0 / vg]);
    half2v v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const half2v prod = half_pair(code_at<BITS>(w, 2 * k), code_at<BITS>(w, 2 * k + 1)) * half2v{s1, s1};
      v[k] = prod + half2v{z1, z1};
    }
    store8<OUT>(out, (out0 + at) * D + c0, v);
  }
}

// Any layout and type, one element at a time.
__device__ __forceinline__ void any_chunk(const dkv_segment& s, bool key, int64_t bh, int D, int t0, int nt,
                                          const int16_t* inv, int meta, int dt, void* out, int64_t out0) {
  for (int i = threadIdx.x; i < D * nt; i += kThreads) {
    const int c = i % D, t = t0 + i / D;
    const PackedElem e = key ? key_code(s, bh, c, t, D, s.key_kind == DKV_KEY_MIXED ? inv[c] : -1)
                             : value_code(s, bh, t, c, D);
    const int64_t sb = key ? s.key_bh[3] : s.value_bh[1], zb = key ? s.key_bh[4] : s.value_bh[2];
    dev_dequant_store(out, (out0 + i / D) * D + c, e.code, dev_load_meta(e.scale, bh * sb + e.at, meta),
                      dev_load_meta(e.zero, bh * zb + e.at, meta), meta, dt);
  }
}

template <int OUT>
__global__ void __launch_bounds__(kThreads) materialize(dkv_materialize_args a) {
  extern __shared__ int16_t inv[];  // [D]
  const int64_t bhs = a.B * a.H;
  const bool key = (blockIdx.x & 1) == 0;
  const int64_t item = blockIdx.x >> 1, bh = item % bhs;
  const int chunk = (int)(item / bhs);
  const int D = (int)a.D, meta = (int)a.meta_dtype, dt = (int)a.dtype;
  dkv_segment s;
  int t0;
  int64_t at;
  if (chunk < a.n_chunks) {
    const int32_t* c = a.chunks + 3 * chunk;
    s = a.segments[c[0]];
    t0 = c[1];
    at = c[2];
  } else {
    s = a.tail;
    t0 = (chunk - (int)a.n_chunks) * kChunk;
    at = a.tail_start + t0;
  }
  const int nt = min(kChunk, s.tokens - t0);
  const int64_t out0 = bh * a.tokens + at;
  void* out = key ? a.keys : a.values;
  if (key ? s.key_kind == DKV_KEY_DENSE : s.value_kind == DKV_VALUE_DENSE) {
    const int esize = dt == kF64 ? 8 : dt == kF32 ? 4 : 2, row = D * esize;
    const uint8_t* src = (const uint8_t*)(key ? s.key[0] : s.value[0]) +
                         ((key ? s.key_bh[0] : s.value_bh[0]) * bh + (int64_t)t0 * D) * esize;
    uint8_t* dst = (uint8_t*)out + out0 * row;
    if ((((uintptr_t)src | (uintptr_t)dst | (uintptr_t)row) & 15) == 0) {
      for (int i = threadIdx.x; i < nt * row / 16; i += kThreads) ((uint4*)dst)[i] = ((const uint4*)src)[i];
    } else {
      for (int i = threadIdx.x; i < nt * row / 2; i += kThreads) ((uint16_t*)dst)[i] = ((const uint16_t*)src)[i];
    }
    return;
  }
  const bool mixed = key && s.key_kind == DKV_KEY_MIXED;
  if (mixed) {
    for (int c = threadIdx.x; c < D; c += kThreads) inv[c] = -1;
    __syncthreads();
    const int32_t* idx = (const int32_t*)s.key[2] + bh * s.key_bh[2];
    for (int j = threadIdx.x; j < s.promoted; j += kThreads) {
      const int32_t c = idx[j];
      if (c >= 0 && c < D) inv[c] = (int16_t)j;
    }
    __syncthreads();
  }
  // 8 codes of one group per load: whole octets in a group, aligned rows
  const int bits = mixed ? 2 : key ? s.key_bits : s.value_bits, group = key ? s.key_group : s.value_group;
  const uint64_t base = key ? s.key[0] | (uint64_t)s.key_bh[0] : s.value[0] | (uint64_t)s.value_bh[0];
  const uint64_t hbase = mixed ? s.key[1] | (uint64_t)s.key_bh[1] : 0;
  const bool octets = meta == kF16 && D % 8 == 0 && group % 8 == 0 && base % bits == 0 && hbase % 2 == 0;
  if constexpr (OUT == kF64) {
    any_chunk(s, key, bh, D, t0, nt, inv, meta, dt, out, out0);
  } else if (!octets) {
    any_chunk(s, key, bh, D, t0, nt, inv, meta, dt, out, out0);
  } else if (key) {
    if (mixed) key_chunk<2, true, OUT>(s, bh, D, t0, nt, inv, out, out0);
    else if (bits == 2) key_chunk<2, false, OUT>(s, bh, D, t0, nt, inv, out, out0);
    else if (bits == 4) key_chunk<4, false, OUT>(s, bh, D, t0, nt, inv, out, out0);
    else key_chunk<8, false, OUT>(s, bh, D, t0, nt, inv, out, out0);
  } else {
    if (bits == 2) value_chunk<2, OUT>(s, bh, D, t0, nt, out, out0);
    else if (bits == 4) value_chunk<4, OUT>(s, bh, D, t0, nt, out, out0);
    else value_chunk<8, OUT>(s, bh, D, t0, nt, out, out0);
  }
}

}  // namespace

extern "C" int dkv_materialize(const dkv_materialize_args* args, void* stream) {
  DKV_CHECK(args != nullptr, DKV_ERR_INVALID, "args is NULL");
  const dkv_materialize_args& a = *args;
  auto is_float = [](int64_t dt) { return dt == kF32 || dt == kF16 || dt == kBF16 || dt == kF64; };
  DKV_CHECK(a.B > 0 && a.H > 0 && a.D > 0 && a.tokens > 0, DKV_ERR_INVALID, "bad materialize shape");
  DKV_CHECK(is_float(a.dtype) && is_float(a.meta_dtype), DKV_ERR_DTYPE,
            "cache and metadata dtypes must be f64, f32, f16 or bf16");
  DKV_CHECK(a.n_chunks >= 0 && (a.n_chunks == 0 || (a.segments != nullptr && a.chunks != nullptr)), DKV_ERR_INVALID,
            "segments or chunks missing");
  DKV_CHECK(a.tail.tokens >= 0 && (a.tail.tokens == 0 || a.tail_start + a.tail.tokens <= a.tokens), DKV_ERR_INVALID,
            "the tail lies outside the outputs");
  DKV_CHECK(a.D <= 16384, DKV_ERR_UNSUPPORTED, "head_dim %lld is too large", (long long)a.D);
  DKV_CHECK(a.keys != nullptr && a.values != nullptr, DKV_ERR_INVALID, "outputs missing");
  const int64_t chunks = a.n_chunks + (a.tail.tokens + kChunk - 1) / kChunk;
  const int64_t blocks = 2 * chunks * a.B * a.H;
  DKV_CHECK(blocks < (int64_t)1 << 31, DKV_ERR_UNSUPPORTED, "too many chunks for one launch");
  if (blocks == 0) return DKV_OK;
  const dim3 grid((unsigned)blocks);
  const size_t lds = (size_t)a.D * sizeof(int16_t);
  hipStream_t s = (hipStream_t)stream;
  if (a.dtype == kBF16) hipLaunchKernelGGL(materialize<kBF16>, grid, dim3(kThreads), lds, s, a);
  else if (a.dtype == kF16) hipLaunchKernelGGL(materialize<kF16>, grid, dim3(kThreads), lds, s, a);
  else if (a.dtype == kF32) hipLaunchKernelGGL(materialize<kF32>, grid, dim3(kThreads), lds, s, a);
  else hipLaunchKernelGGL(materialize<kF64>, grid, dim3(kThreads), lds, s, a);
  return dkv_check_launch("dkv_materialize");
}
