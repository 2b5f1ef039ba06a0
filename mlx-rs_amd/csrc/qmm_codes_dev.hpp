// What the two tiled products on raw codes (qmm_tiles.hip, qmm_codes.hip) share: the layout of the prepared rows.
#pragma once
#include <atomic>

#include "qmm_dev.hpp"

namespace mi_moe {

constexpr int kSlots = 8;  // K slots of a group in the bias product
// Codes multiplied without a centre leave the bias as it is, one bf16: three slots hold the products with it, and the fourth nothing.
constexpr int sum_slots(bool plain_codes) { return plain_codes ? 4 : kSlots; }

// v = h + m + l exactly, each a bf16 (8 significant bits; by truncation, so nothing overflows).  A value that is not
// finite gives a NaN.
struct Pieces { uint32_t h, m, l; };  // bf16 bits in the low halves
__device__ __forceinline__ Pieces split3(float v) {
  const uint32_t u = __float_as_uint(v);
  const uint32_t hu = u & 0xffff0000u;
  const float r = v - __uint_as_float(hu);
  const uint32_t mu = __float_as_uint(r) & 0xffff0000u;
  const float q = r - __uint_as_float(mu);
  return Pieces{hu >> 16, mu >> 16, __float_as_uint(q) >> 16};
}

// A group sum of a row as the bias product's operand: the pieces against those of the biases (six products), or against one.
__device__ __forceinline__ void put_sums(uint16_t *to, int slots, float sum) {
  const Pieces p = split3(sum);
  if (slots == kSlots) *reinterpret_cast<uint4 *>(to) = make_uint4(p.h | p.m << 16, p.l | p.h << 16, p.m | p.h << 16, 0u);
  else *reinterpret_cast<uint2 *>(to) = make_uint2(p.h | p.m << 16, p.l);
}

constexpr RowOrder row_order(int bits) { return bits == 4 ? RowOrder::kPaired : RowOrder::kPlain; }
constexpr int padded_groups(int G) { return (G + 15) / 16 * 16; }  // whole windows of the bias product; the groups past the row's end are zeros

// One thread's part of preparing rows: eight values of x (octet i of all rows).  Whole groups go through lanes of one wave.  ORDER of the copy (kPaired or kQuads),
// SLOTS of a group sum.
// What bounds it is latency: as a launch of its own 4.6 us for 61 rows of 2176 and 5.2 for 611 of 1152 (bf16, with a profiler's overhead).  One lane writes all the
// zeros behind a row's sums, so it writes 16 bytes at a time: with 8, and the two forms told apart at run time, products whose groups fill no multiple of sixteen
// took 0.2 to 0.7 us more (61 x 2320 x 2176 4-bit 14.6 us for 14.0, 611 x 2864 x 1152 18.6 for 17.9, 494 x 960 x 2432 8-bit 17.3 for 16.6).
template <int DT, RowOrder ORDER, int SLOTS>
__device__ __forceinline__ void prepare_octet(const PrepareArgs &a, int64_t i) {
  float v[8];
  const uint4 w = reinterpret_cast<const uint4 *>(a.x)[i];
  const uint32_t u[4] = {w.x, w.y, w.z, w.w};
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    if constexpr (DT == 0) {
      v[2 * j] = bf16lo_to_f32(u[j]);
      v[2 * j + 1] = bf16hi_to_f32(u[j]);
    } else {
      const half2_t hh = __builtin_bit_cast(half2_t, u[j]);
      v[2 * j] = (float)hh.x;
      v[2 * j + 1] = (float)hh.y;
    }
  }
  if (a.copy) {
    constexpr bool QUADS = ORDER == RowOrder::kQuads;
    const uint32_t y = QUADS ? w.z : w.y, z = QUADS ? w.y : w.z;  // the words that meet: neighbours (kQuads), or 0 and 2, 1 and 3 (kPaired)
    uint4 p;
    p.x = (w.x & 0xffffu) | (z << 16);
    p.y = (w.x >> 16) | (z & 0xffff0000u);
    p.z = (y & 0xffffu) | (w.w << 16);
    p.w = (y >> 16) | (w.w & 0xffff0000u);
    *reinterpret_cast<uint4 *>(a.copy + 8 * i) = p;
  }
  float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  sum += __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(sum)));
  sum += __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(sum)));
  if (a.lanes_log2 >= 3) sum += __uint_as_float(dpp_u32<kDppHalfMirror>(__float_as_uint(sum)));
  if (a.lanes_log2 == 4) sum += __uint_as_float(dpp_u32<kDppMirror>(__float_as_uint(sum)));
  if ((i & ((1 << a.lanes_log2) - 1)) == 0) {
    const int64_t row = i / a.octets_per_row;
    const int g = (int)(i % a.octets_per_row) >> a.lanes_log2, G = a.octets_per_row >> a.lanes_log2;
    uint16_t *const to = a.sums + row * a.sums_row;
    put_sums(to + g * SLOTS, SLOTS, sum);
    if (g == G - 1)  // (an even number of groups where a group has four slots)
      for (int k = G * SLOTS; k < a.sums_row; k += 8) *reinterpret_cast<uint4 *>(to + k) = make_uint4(0, 0, 0, 0);
  }
}

// The eight codes of a word as bf16, in the order kQuads.  A byte of 0 to 15 is that many 2^-9 as an 8-bit float (four exponent bits, three of mantissa): the
// conversion takes two at a time.
__device__ __forceinline__ void quads_of(uint32_t even, uint32_t odd, u32x4_t &o) {
  o[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 512.0f, false));
  o[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 512.0f, false));
  o[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(even, 512.0f, true));
  o[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(odd, 512.0f, true));
}
__device__ __forceinline__ void plain_codes(uint32_t w, u32x4_t &o) { quads_of(w & 0x0f0f0f0fu, (w >> 4) & 0x0f0f0f0fu, o); }
// The same less 8: sizes of 0 to 8 in all eight nibbles at once (a code under the centre is its complement and one more), the sign in front of them in a byte.  Five instructions
// more than without a centre, for a word.
__device__ __forceinline__ void signed_codes(uint32_t w, u32x4_t &o) {
  uint32_t under = ~w & 0x88888888u;
  asm("" : "+v"(under));  // (bits that are known to be zero would be taken out of the selections below, an instruction each)
  const uint32_t one = under >> 3, size = (w ^ (0x88888888u - one)) + one;
  quads_of((size & 0x0f0f0f0fu) | (under << 4 & 0xf0f0f0f0u), (size >> 4 & 0x0f0f0f0fu) | (under & 0xf0f0f0f0u), o);
}

// silu(g) u, fp32.  The quotient is as the division gives it.  1 + exp(-g) reaches 2^128, so the reciprocal is taken of a quarter of it (beyond 2^126 that of a
// normal number is none, and v_rcp_f32 gives zero) and one correction follows; where the sum is infinite the quotient is zero, and no correction (an infinite g
// comes out as no number, and is looked at again with all that are not finite).
__device__ __forceinline__ float gated(float g, float u) {
  const float d = 1.0f + __expf(-g), r = __builtin_amdgcn_rcpf(0.25f * d) * 0.25f, q = g * r;
  return (d < INFINITY ? __builtin_fmaf(__builtin_fmaf(-d, q, g), r, q) : q) * u;
}

// A kernel's leave to use more than 64 KB of LDS, asked for once a GPU (half a microsecond a launch otherwise).  done: a bit per GPU.
inline hipError_t allow_lds(const void *kernel, int bytes, std::atomic<uint64_t> &done) {
  int dev = 0;
  if (hipError_t e = hipGetDevice(&dev); e != hipSuccess) return e;
  const uint64_t bit = dev < 64 ? uint64_t{1} << dev : 0;
  if (bit && (done.load(std::memory_order_relaxed) & bit)) return hipSuccess;
  const hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess) done.fetch_or(bit, std::memory_order_relaxed);
  return e;
}

// The dense products that qmm_codes.hip takes (see dense_rule.hpp); share: K is shared by two groups of waves.  small: bf16, 8-bit
// codes in groups of 32.
hipError_t launch_qmm_codes_middle(const CodesArgs &a, bool share, int group, int bits, int dt, hipStream_t st);
hipError_t launch_qmm_codes_small(const CodesArgs &a, hipStream_t st);

}  // namespace mi_moe
