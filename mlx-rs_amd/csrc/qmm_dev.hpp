// Device code that the products on raw codes (qmm_codes.hip, qmm_rows.hip) and over weights packed along N (qmm_cols.hip) share.
#pragma once
#include "common.hpp"

namespace mi_moe {

typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4_t;
typedef __attribute__((__vector_size__(2 * sizeof(uint32_t)))) uint32_t u32x2_t;
typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
typedef __attribute__((__vector_size__(8 * sizeof(_Float16)))) _Float16 f16x8_t;

template <int DT> struct ElemOf;  // mi_moe_dtype
template <> struct ElemOf<0> { typedef uint16_t type; };
template <> struct ElemOf<1> { typedef _Float16 type; };
template <> struct ElemOf<2> { typedef float type; };

template <class T> __device__ __forceinline__ T rounded(float v) { return (T)v; }
template <> __device__ __forceinline__ uint16_t rounded<uint16_t>(float v) { return (uint16_t)(cvt_pk_bf16(v, 0.f) & 0xffffu); }

__device__ __forceinline__ __amdgpu_buffer_rsrc_t rsrc_of(const void *base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
}

// Eight values a lane of bf16 (DT 0; pieces of f32 as well) or f16: 32 x 32 results over 16 K values, 16 x 16 over 32.
template <int DT>
__device__ __forceinline__ f32x16_t mfma(u32x4_t a, u32x4_t b, f32x16_t c) {
  if constexpr (DT == 1)
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}
template <int DT>
__device__ __forceinline__ f32x4_t mfma(u32x4_t a, u32x4_t b, f32x4_t c) {
  if constexpr (DT == 1)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8_t, a), __builtin_bit_cast(f16x8_t, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, a), __builtin_bit_cast(bf16x8_t, b), c, 0, 0, 0);
}

// The products on raw codes multiply centred codes q - 8 and q - 128: s q + b = s (q - c) + (b + c s).  Without the centre the code
// and bias terms of a group are several times their sum, and what they lose to each other's rounding is too.
constexpr float centre_of(int bits) { return (float)(1 << (bits - 1)); }
// Centred codes of one word as f32: two 4-bit codes a byte, times 16 (their byte's upper half), or 8-bit ones.  The signed byte
// comes out of the conversion itself.
__device__ __forceinline__ void centred_codes(uint32_t w, float (&v)[8]) {  // 4-bit: 16 (q_i - 8)
  const uint32_t even = ((w << 4) ^ 0x88888888u) & 0xf0f0f0f0u, odd = (w ^ 0x88888888u) & 0xf0f0f0f0u;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    v[2 * i] = (float)(int8_t)(even >> (8 * i));
    v[2 * i + 1] = (float)(int8_t)(odd >> (8 * i));
  }
}
__device__ __forceinline__ void centred_codes(uint32_t w, float (&v)[4]) {  // 8-bit: q_i - 128
#pragma unroll
  for (int i = 0; i < 4; ++i) v[i] = (float)(int8_t)((w ^ 0x80808080u) >> (8 * i));
}
__device__ __forceinline__ uint32_t upper_halves(float lo, float hi) {  // two bf16 of values that are bf16 already
  return __builtin_amdgcn_perm(__float_as_uint(hi), __float_as_uint(lo), 0x07060302u);
}

template <int BITS>
__device__ __forceinline__ uint32_t f16_centred(uint32_t v) {  // two halves 1024 + q -> q - centre: exact
  constexpr _Float16 off = (_Float16)(1024.0f + centre_of(BITS));
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(half2_t, v) - half2_t{off, off});
}

// ROWS rows of x against one row of weights packed along K, an fma per k on the dequantised weight, in the order of k.  The products
// on raw codes take it where their own sum is not finite: an infinity against codes and biases apart cancels to no number where
// the dequantised weight keeps its sign, and sums of unscaled codes overflow earlier.  order: of the 8-blocks of
// x.  open: the rows that are wanted.  K and the group are multiples of 32, x and w are aligned for 16 bytes.
// It is one lane's chain over K and the latency of its loads, so 32 values of each row are fetched at a time.
// us of a product 4096 x 4096 with finite rows / one infinity in one row / one in each: bf16 4-bit 1 row 12 / 79, 16 rows 17 / 89 / 284, 200 rows 36 /
// 200 / 1460, 1000 rows 66 / 274 / 1840; f16 8-bit 777 rows 58 / 222 / 1830 (one row and word at a time 12 / 108, 17 / 118 / 480, 38 / 174 / 5530, 73 /
// 268 / 11800, 61 / 290 / 24000; a wave per output element 3160 for the last).  Rows of NaNs cost next to nothing.
template <int BITS, int ROWS, class T>
__device__ __forceinline__ void plain_rows(const T *const (&x)[ROWS], RowOrder order, const uint32_t *w, const T *s, const T *b, int K, int group,
                                           uint32_t open, float (&sum)[ROWS]) {
  static_assert(sizeof(T) == 2, "eight values are 16 bytes");
  constexpr int PER = 32 / BITS;  // codes of a word
#pragma unroll
  for (int r = 0; r < ROWS; ++r) sum[r] = 0.f;
#pragma unroll 1
  for (int k = 0; k < K && open; k += 32) {
    uint4 xv[ROWS][4];
    uint32_t words[BITS];
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
#pragma unroll
      for (int i = 0; i < 4; ++i) xv[r][i] = reinterpret_cast<const uint4 *>(x[r] + k)[i];
    __builtin_memcpy(words, __builtin_assume_aligned(w + k / PER, 16), sizeof words);
    const float sc = as_f32(s[k / group]), bi = as_f32(b[k / group]);
#pragma unroll
    for (int i = 0; i < 32; ++i) {
      const int at = i & 7, from = place_of_value(order, at);
      const float wf = __builtin_fmaf(sc, (float)((words[i / PER] >> (i % PER * BITS)) & ((1u << BITS) - 1u)), bi);
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        T v[8];
        __builtin_memcpy(v, &xv[r][i / 8], sizeof v);
        sum[r] = __builtin_fmaf(as_f32(v[from]), wf, sum[r]);
      }
    }
#pragma unroll
    for (int r = 0; r < ROWS; ++r)
      if (sum[r] != sum[r]) open &= ~(1u << r);  // (no number stays none)
  }
}

}  // namespace mi_moe
