// Tiled quantized product on raw codes: activations in bfloat16 or float16, groups of 32, 64 or 128, any number of
// output columns; dense, or (4-bit codes in groups of 64) the pieces of a mixture-of-experts block's segments.
//
// Contract: mlx_quantized_matmul / mlx_gather_qmm with transpose = true (mlx-rs/src/ops/quantization.rs:91-122,160-230).
//
// Arithmetic: sum_c x_c (s q_c + b) = s sum_c x_c (q_c - c) + (b + c s) sum_c x_c per quantisation group, with a centre c of
// the codes.  q - c is exact in bf16 and in f16, so the matrix cores multiply the activations with it and nothing is
// rounded on the way in:
//   bf16  x as it is; codes through v_cvt_f32_i32 of signed bytes (4-bit codes times 16), c = 8 or 128
//   f16   x as it is, codes in f16 (v_mfma_f32_32x32x16_f16), the same c
//   blocks with 4-bit codes in groups of 64: c = 0, codes through v_cvt_scalef32_pk_bf16_fp8 (a byte of 0 .. 15 is that many 2^-9 as an
//         8-bit float, exactly), 8 instructions a multiply for 15
// Share of results that are not the float64 product's nearest value (bf16, 4-bit, 64 to 777 rows): plain float32 sums 0.9e-4 .. 1.5e-4, c = 8
// 1.1e-4 .. 1.7e-4, c = 0 3.3e-4, 128 + q (what the streaming kernel multiplies with) 4.7e-3, weights rounded to bf16 (the 256-column
// tiles) no comparison.  Groups of 32 and 128 and the dense products keep c = 8.
// float32 does not come here: without the centre its error was 3.3e-7 to 5.7e-7 (a wave per output element 1.0e-7 to 1.5e-7).
// The fp32 sums of a group are scaled once, when the group ends.  The bias term sum_g b_g (sum_c x_c) is a product of
// its own over the groups: the group sums of x (fp32, split into three bf16 pieces) against the biases (three pieces
// as well), eight K slots a group (xh bh, xm bh, xl bh, xh bm, xm bm, xh bl: every product down to 2^-24): K / group * 8 / K = 12 % more
// matrix work with groups of 64.  It runs a window of 8 or 16 groups ahead of the window's codes, so that the sums never drift far.
//
// A kernel of its own (prepare_rows) walks x once and writes the group sums in that form and, for 4-bit codes with bf16
// and f16, the copy with paired 8-blocks that their unpacking wants.
#include <type_traits>

#include "dense_rule.hpp"
#include "lds_copies.hpp"
#include "qmm_codes_dev.hpp"

namespace mi_moe {

// One thread per eight values of x.
template <int DT, RowOrder ORDER>
__global__ __launch_bounds__(256) void prepare_rows_kernel(PrepareArgs a) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i < a.octets) prepare_octet<DT, ORDER, kSlots>(a, i);  // (whole groups leave together)
}

// What a launch of the kernel below is made of, for its two sides.
template <int BITS, int MS, int NT, int WN, int S>
struct Ring {
  static constexpr int KS = BITS == 4 ? 128 : 64;  // K values of a stage: 64 bytes of codes per weight row
  static constexpr int XROW = KS * 2;              // bytes of a token row
  static constexpr int X = 32 * MS * XROW;         // token rows of a stage
  static constexpr int W = NT * 2048;              // one wave's codes
  static constexpr int STAGE = X + WN * W;
  static constexpr int XI = (X + 1024 * WN - 1) / (1024 * WN);  // copies a wave makes of a stage's token rows
  static constexpr int COPIES = XI + 2 * NT;                    // and in all
  static constexpr int WINDOW = NT * 1024;                      // 32 bytes of scales per weight row of a wave
  static constexpr int BYTES = S * STAGE + WN * WINDOW;
};

// LDS of a block: where two blocks share a CU, each takes its half.
constexpr int kHalfLds = 80 * 1024;
constexpr int lds_of(int kw, int bytes) { return kw == 1 && bytes > kHalfLds / 2 && bytes <= kHalfLds ? kHalfLds : kw * bytes; }
// Waves a SIMD holds: those of one block, of two where two share the CU. A bound above that only takes registers: 32 x 64 tiles of
// 4-bit codes, held to 128 of the 134 registers they want, ran in 18.0 us at 77 x 1680 x 2432 in groups of 32 (bf16) instead of 17.1.
constexpr int waves_of(int waves, int lds) {
  const int blocks = lds <= kHalfLds ? 2 : 1;
  return blocks * waves > 8 ? blocks * waves / 4 : 2;
}

// LIST: pieces of a block with 4-bit codes in groups of 64 (bf16); else dense.
template <int DT, int BITS, bool G32, bool LIST, int MS, int NT, int WN, int S>
struct Tile {
  static_assert(!LIST || (DT == 0 && BITS == 4 && !G32), "other blocks' pieces: qmm_short.hip, qmm_bytes.hip");
  typedef typename ElemOf<DT>::type T;
  typedef Ring<BITS, MS, NT, WN, S> R;
  static constexpr bool SPLIT = BITS == 8 || G32;  // which K values a multiply takes: see unpack
  static constexpr bool kPlainCodes = LIST;
  static constexpr float kCentre = kPlainCodes ? 0.0f : centre_of(BITS);                       // the codes are multiplied as
  static constexpr float kUnit = BITS == 4 && DT == 0 && !kPlainCodes ? 0.0625f : 1.0f;  // (q - kCentre) / kUnit
  static constexpr int JS = R::KS / 64;  // steps of a stage
  static constexpr int NQ = BITS == 4 ? 1 : 2;
  static constexpr int NS = G32 ? 2 : 1;
  static constexpr int GB = R::KS / 8;   // groups of a stage of the bias product

  // 4-bit codes in groups of 32: the words dealt so that a multiply stays inside one group
  static __device__ __forceinline__ void deal(u32x4_t (&q)[NQ]) {
    if constexpr (BITS == 4 && G32) {
#pragma unroll
      for (int w = 0; w < 2; ++w) {
        const auto r = __builtin_amdgcn_permlane32_swap(q[0][w], q[0][w + 2], false, false);
        q[0][w] = r[0];
        q[0][w + 2] = r[1];
      }
    }
  }
  // the eight codes of multiply h
  static __device__ __forceinline__ void unpack(const u32x4_t (&q)[NQ], int h, u32x4_t &o) {
      if constexpr (kPlainCodes) {
        plain_codes(q[0][h], o);
      } else if constexpr (BITS == 4 && DT == 0) {
        float v[8];
        centred_codes(q[0][h], v);
#pragma unroll
        for (int i = 0; i < 4; ++i) o[i] = upper_halves(v[i], v[i + 4]);
      } else if constexpr (BITS == 4) {
        const uint32_t w = q[0][h];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (i % 2 == 0) {
            o[i] = f16_centred<4>(__builtin_amdgcn_bitop3_b32(w >> (4 * i), 0x000f000fu, 0x64006400u, 0xEA));  // (a & b) | c
          } else {  // 1024 + 16 q -> q - 8, exact as well: one shift serves two nibbles
            const half2_t v = __builtin_bit_cast(half2_t, __builtin_amdgcn_bitop3_b32(w >> (4 * (i - 1)), 0x00f000f0u, 0x64006400u, 0xEA));
            o[i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, half2_t{(_Float16)0.0625f, (_Float16)0.0625f}, half2_t{(_Float16)-72.0f, (_Float16)-72.0f}));
          }
        }
      } else if constexpr (DT == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i)  // bytes 2 i, 2 i + 1 under the exponent of 1024
          o[i] = f16_centred<8>(__builtin_amdgcn_perm(0x64646464u, q[h >> 1][2 * (h & 1) + (i >> 1)], (i & 1) ? 0x07030702u : 0x07010700u));
      } else {
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          float v[4];
          centred_codes(q[h >> 1][2 * (h & 1) + (i >> 1)], v);
          o[i] = upper_halves(v[0], v[1]);
          o[i + 1] = upper_halves(v[2], v[3]);
        }
      }
  }
};


// The bias product of a window of sixteen groups where the codes have no centre: the group sums' three pieces against the bias, a bf16 as it is.  A lane
// has two groups of a token row in 16 bytes (`place` of its row in LDS), and their two biases in a word.  Groups from `real` on are not this product's.
template <int MS, int NT, class Place>
__device__ __forceinline__ void add_plain_biases(float (&tot)[MS][NT][16], const unsigned char *rows_at, int row_bytes, Place place, const unsigned char *biases, int real, int ln, int kb) {
  u32x4_t o[NT][4];
#pragma unroll
  for (int t = 0; t < NT; ++t)
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int g = 4 * i + 2 * kb;
      const uint32_t b = g < real ? *reinterpret_cast<const uint32_t *>(biases + t * 1024 + g * 2) : 0u;  // (an even number of groups)
      o[t][i] = u32x4_t{__builtin_amdgcn_perm(b, b, 0x01000100u), b & 0xffffu, __builtin_amdgcn_perm(b, b, 0x03020302u), b >> 16};
    }
#pragma unroll
  for (int m = 0; m < MS; ++m) {
    u32x4_t F[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) F[i] = *reinterpret_cast<const u32x4_t *>(rows_at + (32 * m + ln) * row_bytes + place(2 * i + kb));
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      f32x16_t sum = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int i = 0; i < 4; ++i) sum = mfma<0>(F[i], o[t][i], sum);
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[m][t][v] += sum[v];
    }
  }
}

// The results of a dense tile (see multiply_tile) go out.
template <int DT, int BITS, int MS, int NT, int WN, class WeightRow>
__device__ __forceinline__ void write_tile(const CodesArgs &a, const float (&tot)[MS][NT][16], int wave, int lane, int col0, int64_t row0, int rows,
                                           int glog, WeightRow weight_row, unsigned char *lds_raw) {
  // ---- epilogue: a wave turns its 32 x 32 sub-tiles round in a private piece of LDS and stores 16 bytes a lane
  typedef typename ElemOf<DT>::type T;
  const int N = a.N, K = a.K, G = K >> glog, row_bytes = K * BITS / 8;
  const int ln = lane & 31, kb = lane >> 5;
  constexpr int ROWB = 32 * (int)sizeof(T) + 16;
  constexpr int PV = 16 / (int)sizeof(T);             // values per 16-byte piece
  constexpr int CPR = 32 / PV;                        // pieces per row
  constexpr int RPI = 64 / CPR;                       // rows one store instruction covers
  unsigned char *const mine = lds_raw + wave * (32 * ROWB);
  const int my_piece = lane % CPR, my_row = lane / CPR;
  const bool vec = N % PV == 0;
#pragma unroll
  for (int u = 0; u < MS * NT; ++u) {
    const int m = u / NT, t = u % NT, col = col0 + 32 * t;
    const float lb = a.bias ? as_f32(static_cast<const T *>(a.bias)[col + ln < N ? col + ln : N - 1]) : 0.f;
    auto put = [&](int r, float v) __attribute__((always_inline)) {
      T o = rounded<T>(v);
      if (a.bias) o = rounded<T>(as_f32(o) + lb);
      reinterpret_cast<T *>(mine + (8 * (r >> 2) + 4 * kb + (r & 3)) * ROWB)[ln] = o;
    };
    uint32_t again = 0;  // (bits: which of the sixteen sums are not finite)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      put(r, tot[m][t][r]);
      again |= (not_finite(tot[m][t][r]) ? 1u : 0u) << r;
    }
#pragma unroll 1
    for (int quad = 0; __builtin_expect(again != 0, 0); ++quad, again >>= 4) {  // rows 8 quad + 4 kb + 0 .. 3
      uint32_t open = again & 15u;
      const T *xs[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        int tr = 32 * m + 8 * quad + 4 * kb + i;
        if (tr >= rows) {  // (never stored)
          open &= ~(1u << i);
          tr = rows - 1;
        }
        xs[i] = static_cast<const T *>(a.x) + (row0 + tr) * K;
      }
      if (!open) continue;
      float v[4];
      const int64_t wrow = weight_row(t, ln);
      plain_rows<BITS, 4, T>(xs, row_order(BITS), a.w0 + wrow * (row_bytes / 4), static_cast<const T *>(a.s0) + wrow * G, static_cast<const T *>(a.b0) + wrow * G, K, K / G,
                             open, v);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (open >> i & 1u) put(4 * quad + i, v[i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int my_col = col + PV * my_piece;
#pragma unroll
    for (int i = 0; i < 32 / RPI; ++i) {
      const int row = RPI * i + my_row;
      const int tr = 32 * m + row;
      if (tr < rows && my_col < N) {
        T *const to = static_cast<T *>(a.y) + (row0 + tr) * N + my_col;
        const T *const from = reinterpret_cast<const T *>(mine + row * ROWB) + PV * my_piece;
        if (vec) {
          *reinterpret_cast<u32x4_t *>(to) = *reinterpret_cast<const u32x4_t *>(from);
        } else {
          for (int c = 0; c < PV && my_col + c < N; ++c) to[c] = from[c];
        }
      }
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  }
}

// Where rows l and 64 + l of a piece go, in lane l.
__device__ __forceinline__ void output_rows(const CodesArgs &a, int64_t row0, int rows, int lane, uint32_t (&dst)[2]) {
#pragma unroll
  for (int h = 0; h < 2; ++h) {
    const int64_t r = row0 + (64 * h + lane < rows ? 64 * h + lane : rows - 1);
    dst[h] = a.dst_rows ? a.dst_rows[r] : (uint32_t)r;
  }
}
// The results of a piece of up to 32 MS rows x 256 weight rows (of a block; four waves, 64 weight rows each) go out: N is a multiple of
// 128, there is no bias of the layer's.  Two rows of a column become one register, neighbouring lanes swap halves, and the rows are turned round in LDS:
// GLU: by the whole block, whose 256 bytes a row are two quantisation groups of h, of which the lanes that store them also write the group sums;
// else by each wave, 128 bytes a row.  (Rows found and stored 16 at a time behind a load of their places each: 12 us of the 37 of a block of 128 rows, K = 768.)
template <bool GLU, int MS, class WeightRow>
__device__ __forceinline__ void write_piece(const CodesArgs &a, const float (&tot)[MS][2][16], int wave, int lane, int n0, int64_t row0, int rows, int64_t ebase,
                                            WeightRow weight_row, const uint32_t (&dst)[2], unsigned char *lds_raw) {
  constexpr int ROWB = GLU ? 272 : 144;  // (16 bytes keep rows off each other's banks)
  constexpr int SLOTS = sum_slots(true);
  const int N = a.N, K = a.K, G = K >> 6, row_bytes = K / 2, ln = lane & 31, kb = lane >> 5;
  unsigned char *const mine = GLU ? lds_raw + wave * 64 : lds_raw + wave * (32 * ROWB);
  auto value = [&](int m, int t, int r) __attribute__((always_inline)) { return GLU ? gated(tot[m][0][r], tot[m][1][r]) : tot[m][t][r]; };
  float odd = 0.f;  // no number once a result was not finite
  auto turn = [&](int m, int at) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < (GLU ? 1 : 2); ++t)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float v0 = value(m, t, r), v1 = value(m, t, r + 1);
        odd = __builtin_fmaf(v1, 0.f, __builtin_fmaf(v0, 0.f, odd));
        const uint32_t own = cvt_pk_bf16(v0, v1), theirs = dpp_u32<kDppXor1>(own);
        // even lane: row r of columns c, c + 1; odd lane: row r + 1
        const uint32_t both = __builtin_amdgcn_perm(theirs, own, (ln & 1) ? 0x03020706u : 0x05040100u);
        *reinterpret_cast<uint32_t *>(mine + (at + 8 * (r >> 2) + 4 * kb + (r & 3) + (ln & 1)) * ROWB + (32 * t + (ln & ~1)) * 2) = both;
      }
  };
  // sums that are not finite, again on the dequantised weights (see plain_rows)
  auto repair = [&](int m_first, int m_end, int at) __attribute__((always_inline)) {
    uint64_t again = 0, again_1 = 0;  // (which of a column's rows, of the wave's first and second 32 columns: not an array, which would lie in scratch memory)
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < (GLU ? 1 : 2); ++t) {
        uint32_t bits = 0;
#pragma unroll
        for (int r = 0; r < 16; ++r) bits |= (not_finite(tot[m][t][r]) || (GLU && not_finite(tot[m][1][r])) ? 1u : 0u) << r;
        (t ? again_1 : again) |= (uint64_t)bits << (16 * m);
      }
#pragma unroll 1
    for (int i = m_first * 4 * (GLU ? 1 : 2); i < m_end * 4 * (GLU ? 1 : 2); ++i) {  // four rows of a column at a time
      const int t = GLU ? 0 : i & 1, quad = GLU ? i : i >> 1;  // rows 8 quad + 4 kb + 0 .. 3
      uint32_t open = (uint32_t)((t ? again_1 : again) >> (4 * quad)) & 15u;
      const uint16_t *xs[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        int tr = 8 * quad + 4 * kb + j;
        if (tr >= rows) {  // (never stored)
          open &= ~(1u << j);
          tr = rows - 1;
        }
        xs[j] = static_cast<const uint16_t *>(a.x) + (int64_t)(a.src_rows ? a.src_rows[row0 + tr] : (uint32_t)(row0 + tr)) * K;
      }
      if (!open) continue;
      float v[GLU ? 2 : 1][4];
#pragma unroll
      for (int j = 0; j < (GLU ? 2 : 1); ++j) {
        const int64_t wrow = ebase + weight_row(GLU ? j : t, ln);
        plain_rows<4, 4, uint16_t>(xs, RowOrder::kQuads, (j ? a.w1 : a.w0) + wrow * (row_bytes / 4), static_cast<const uint16_t *>(j ? a.s1 : a.s0) + wrow * G,
                                   static_cast<const uint16_t *>(j ? a.b1 : a.b0) + wrow * G, K, 64, open, v[j]);
      }
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (open >> j & 1u) {
          const float o = GLU ? v[0][j] / (1.0f + __expf(-v[0][j])) * v[GLU ? 1 : 0][j] : v[0][j];
          reinterpret_cast<uint16_t *>(mine + (8 * quad + 4 * kb + j - at) * ROWB)[32 * t + ln] = rounded<uint16_t>(o);
        }
    }
  };
  if constexpr (GLU) {
#pragma unroll
    for (int m = 0; m < MS; ++m) turn(m, 32 * m);
    if (__builtin_expect(odd != odd, 0)) repair(0, MS, 0);
    __syncthreads();
    const int groups = N >> 6, padded = padded_groups(groups);
#pragma unroll
    for (int i = 0; i < 2 * MS; ++i) {
      const int row = 16 * i + (int)(threadIdx.x >> 4), piece = threadIdx.x & 15;
      const u32x4_t w = *reinterpret_cast<const u32x4_t *>(lds_raw + row * ROWB + piece * 16);
      float sum = ((bf16lo_to_f32(w[0]) + bf16hi_to_f32(w[0])) + (bf16lo_to_f32(w[1]) + bf16hi_to_f32(w[1]))) +
                  ((bf16lo_to_f32(w[2]) + bf16hi_to_f32(w[2])) + (bf16lo_to_f32(w[3]) + bf16hi_to_f32(w[3])));
      sum += __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(sum)));
      sum += __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(sum)));
      sum += __uint_as_float(dpp_u32<kDppHalfMirror>(__float_as_uint(sum)));
      if (row < rows) {
        *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(a.y) + (row0 + row) * N + n0 + 8 * piece) = w;
        if ((piece & 7) == 0) put_sums(a.y_sums + ((row0 + row) * padded + (n0 >> 6) + (piece >> 3)) * SLOTS, SLOTS, sum);
      }
    }
    if (n0 + 128 >= N && groups < padded)  // the last block of a row writes the zeros behind its sums
      for (int i = threadIdx.x; i < rows * (padded - groups); i += 256)
        put_sums(a.y_sums + ((row0 + i / (padded - groups)) * padded + groups + i % (padded - groups)) * SLOTS, SLOTS, 0.f);
  } else {
    const bool inside = n0 + 64 * wave < N;  // (else the wave's columns repeat the last one)
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      turn(m, 0);
      if (__builtin_expect(odd != odd, 0)) repair(m, m + 1, 32 * m);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int row = 8 * i + (lane >> 3), tr = 32 * m + row;
        const u32x4_t w = *reinterpret_cast<const u32x4_t *>(mine + row * ROWB + (lane & 7) * 16);
        const uint32_t to = (uint32_t)__shfl((int)dst[m / 2], tr & 63, 64);
        if (tr < rows && inside) *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(a.y) + (int64_t)to * N + n0 + 64 * wave + 8 * (lane & 7)) = w;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
}

// One tile: 32 MS token rows from sorted row `row0` (`rows` of them real) x 32 WN NT weight rows from n0 of matrix e (GLU: of two matrices).
// A wave owns 32 NT weight rows for all the tile's token rows.  K runs in stages of 64 bytes of codes a weight row; token rows and codes are
// copied straight into a ring of S stages in LDS, the rows for all waves (one barrier a stage), the codes for the wave that
// unpacks them.  A lane (weight row l % 32, half l / 32) reads 16 bytes of codes at a time; which K values its eight codes of a multiply
// stand for is free as long as the token operand agrees:
//   4-bit, groups >= 64: 16 bytes are 32 codes, half h holds K values 32 h ..: multiply t takes word t of both halves;
//   4-bit, groups of 32: two v_permlane32_swap deal the words so that a multiply stays inside one group;
//   8-bit: 16 bytes are 16 codes, two reads a step of 64, groups of 32 stay apart by themselves.
// KW > 1: the block's waves form KW groups that share K among them, each with a ring of its own; their sums meet in
// LDS at the end, added in group order.
// What bounds it: the vector instructions (unpacking 8 to 15 a multiply and 32 weight rows, the scaled addition of a group 16 a
// sub-tile) issue beside the matrix instructions at 4 cycles each, about 1250 cycles a stage of 64 x 64 x 128 in c = 0 where its multiplies are
// 1024; two waves a SIMD reach 0.55 of that, as reads, copies and the barrier of a stage add their latencies.  4096 x 4096, 777 rows, bf16 4-bit:
// 58.7 us for the call = 444 TFLOP/s (tiles of 64 x 128 with the codes loaded into registers 63.4).
// Blocks (128 experts, hidden 2048, 4-bit, groups of 64), us of a forward at 128 / 320 / 1024 tokens, even routing: 110 / 121 / 174; with streamed
// segments, 256-column tiles and a copy of x on four streams, which they took at first, 151 / 216 / 266.
template <int DT, int BITS, bool G32, bool LIST, bool GLU, int MS, int NT, int WN, int KW, int S>
__device__ __forceinline__ void multiply_tile(const CodesArgs &a, int e, int64_t row0, int rows, int n0, int scale_shift, unsigned char *lds_raw) {
  typedef Tile<DT, BITS, G32, LIST, MS, NT, WN, S> P;
  typedef typename P::R R;
  typedef typename P::T T;
  constexpr int GB = P::GB;
  constexpr int NM = GLU ? 2 : 1;  // matrices
  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave_all % WN, kg = wave_all / WN;  // column tile, K group
  const int N = a.N, K = a.K;
  const int ln = lane & 31, kb = lane >> 5;
  const int glog = G32 ? 5 : 6 + scale_shift, G = K >> glog;
  const int row_bytes = K * BITS / 8;
  unsigned char *const ring = lds_raw + kg * R::BYTES;
  const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds_raw + (uint32_t)kg * R::BYTES;

  // ---- operands.  Offsets are 32 bits: the host takes this kernel for operands below 4 GiB only.
  const int64_t ebase = (int64_t)e * N;
  const int ext = padded_groups(G) * sum_slots(P::kPlainCodes);
  const i32x4_t xr = words_of(a.x, (uint32_t)(a.x_rows * K * sizeof(T))), xsr = words_of(a.sums, (uint32_t)(a.x_rows * ext * 2));
  const T *s_of[NM], *b_of[NM];
  i32x4_t wr[NM], sr[NM], br[NM];
#pragma unroll
  for (int t = 0; t < NM; ++t) {
    s_of[t] = static_cast<const T *>(t ? a.s1 : a.s0) + ebase * G, b_of[t] = static_cast<const T *>(t ? a.b1 : a.b0) + ebase * G;
    wr[t] = words_of((t ? a.w1 : a.w0) + ebase * (row_bytes / 4), (uint32_t)N * row_bytes);
    sr[t] = words_of(s_of[t], (uint32_t)N * G * sizeof(T)), br[t] = words_of(b_of[t], (uint32_t)N * G * sizeof(T));  // (read in words: the host takes an even number of them)
  }
  // weight row of place `at` (0 .. 31) of the wave's tile t.  Columns past the end repeat the last one (never stored).  Order of h
  // (CodesArgs::y_order): the place p of an 8-block takes the row whose result belongs there.
  const int col0 = n0 + 32 * (GLU ? 1 : NT) * wave;
  auto weight_row = [&](int t, int at) __attribute__((always_inline)) {
    const int p = GLU ? (at & ~7) | value_at_place(a.y_order, at & 7) : at, row = col0 + (GLU ? 0 : 32 * t) + p;
    return row < N ? row : N - 1;
  };
  // ---- what a lane copies, and where it lies in LDS.  LDS gives 256 bytes a cycle, sixteen lanes' pieces, if they lie in different
  // banks: place p of a row holds piece p ^ (a number of the row), so that sixteen rows' pieces of one number do.  (Turned by
  // eight rows only: 7.3 cycles a read of a wave for 4.)
  constexpr int XP = R::XROW / 16;  // pieces of a token row
  constexpr int XALL = R::X / 1024;  // copies of a stage's token rows (fewer than waves: the first XALL of them make one each)
  auto turned = [](int row) __attribute__((always_inline)) { return XP == 16 ? row & 15 : (row >> 1) & 7; };
  uint32_t x_row[R::XI], x_piece[R::XI];
#pragma unroll
  for (int i = 0; i < R::XI; ++i) {
    const int r = (wave * R::XI + i) % XALL * (64 / XP) + lane / XP;
    const int tr = r < rows ? r : rows - 1;  // rows past the end repeat the last one (never stored)
    x_row[i] = a.src_rows ? a.src_rows[row0 + tr] : (uint32_t)(row0 + tr);
    x_piece[i] = ((lane % XP) ^ turned(r)) << 4;
  }
  uint32_t w_off[2 * NT], first_scale[NT], window_row[NT];
#pragma unroll
  for (int i = 0; i < 2 * NT; ++i) {
    const int at = 16 * (i & 1) + (lane >> 2);
    w_off[i] = (uint32_t)weight_row(i / 2, at) * row_bytes + (((lane & 3) ^ ((at >> 2) & 3)) << 4);
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) first_scale[t] = (uint32_t)weight_row(t, ln) * G, window_row[t] = (uint32_t)weight_row(t, lane >> 1) * G;

  // ---- the stages.  K is dealt to the K groups in even shares; a share runs in windows of GB quantisation groups, each a stage of the
  // bias product (which brings the window's scales) and then its stages of codes.
  // Shares are whole 128s (in 256s the longest of four shares of K = 2432 was 768 values for 640: 77 x 1680 x 2432, 4-bit in groups of 32, bf16,
  // 16.7 us for 15.6).  With groups of 128 a lane's first scale can then lie between two words, as it does where rows hold an odd number of
  // them: its window is fetched from the word before, one place late, which leaves fifteen groups in a window of sixteen.  Longer shares are
  // made even, and rows of an odd number of scales are then read where they are (`in_place`: two bytes a group and row; all odd rows
  // in place, 19 x 1856 x 3712 in bf16 17.7 us for 16.3).
  const int per_window = 1 << (glog - 3);  // stages of codes: GB groups
  const bool beyond = BITS == 4 && glog == 7 && share_of_k(K, KW, false) > 15 * 128, in_place = beyond && (G & 1);
  const int share = share_of_k(K, KW, beyond);
  const int k_first = kg * share, k_end = k_first + share < K ? k_first + share : K;
  int scales_at[NT];  // of a lane's row in a window
#pragma unroll
  for (int t = 0; t < NT; ++t) scales_at[t] = t * 1024 + ln * 32 + (in_place ? 0 : ((first_scale[t] + (k_first >> glog)) & 1) * 2);
  const int stages_all = (share < K ? share : K) / R::KS, total = stages_all + (stages_all + per_window - 1) / per_window;  // of every K group
  struct Next {  // a stage to be copied
    int k, pos;  // first K value, place in the window (0: the bias product)
  } next_w = {k_first, 0}, next_x = {k_first, 0};
  auto advance = [&](Next &n) __attribute__((always_inline)) {
    if (n.pos) n.k += R::KS;
    n.pos = n.pos == per_window ? 0 : n.pos + 1;
  };
  // A stage's token rows are copied S - 1 stages ahead, its weights S: a wave's place in the ring is its own, and free as soon as it has read
  // the codes out of it.  (Stages past the end copy the last one again: the number of copies in flight is always the same.)
  auto copy_w = [&](int slot, int i) __attribute__((always_inline)) {  // copy i of 2 NT: the codes or a window's scales and biases
    const int k = next_w.k < K ? next_w.k : K - R::KS;
    const bool bias = next_w.pos == 0;
    i32x4_t from;
    const int of = GLU ? i / 2 : 0, t = i % NT, of_bias = GLU ? t : 0;  // (codes: two copies a tile; bias product: the tiles' scales, then their biases)
#pragma unroll
    for (int w = 0; w < 4; ++w) from[w] = bias ? (i < NT ? sr : br)[of_bias][w] : wr[of][w];
    const uint32_t off = ((window_row[t] + (k >> glog)) * (uint32_t)sizeof(T) & ~3u) + ((lane & 1) << 4);
    copy_to_lds(from, bias ? off : w_off[i], bias ? 0 : k * BITS / 8, ring_at + slot * R::STAGE + R::X + wave * R::W + i * 1024);
  };
  auto copy_x = [&](int slot, int c) __attribute__((always_inline)) {  // copy c of XI: the token rows or their group sums
    const int k = next_x.k < K ? next_x.k : K - R::KS;
    const bool bias = next_x.pos == 0;
    i32x4_t from;
#pragma unroll
    for (int w = 0; w < 4; ++w) from[w] = bias ? xsr[w] : xr[w];
    copy_to_lds(from, x_row[c] * (uint32_t)(bias ? ext * 2 : K * (int)sizeof(T)) + x_piece[c], bias ? (k >> glog) * (2 * sum_slots(P::kPlainCodes)) : k * (int)sizeof(T),
                ring_at + slot * R::STAGE + (wave * R::XI + c) % XALL * 1024);
  };
  auto copy_weights = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 2 * NT; ++i) copy_w(slot, i);
  };
  auto copy_rows = [&](int slot) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < R::XI; ++c) copy_x(slot, c);
  };

  float tot[MS][NT][16];  // (not vectors: the multiplies never touch them, and each may lie in a register of its own)
  const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[m][t][v] = 0.f;

  // the bias product of the window that begins at k: group sums of x against b + centre s, accumulated into the result
  unsigned char *const scales = ring + S * R::STAGE + wave * R::WINDOW;  // [tile][weight row][16 scales]
  auto bias_product = [&](const unsigned char *at, int real, auto scale_and_bias) __attribute__((always_inline)) {
    f32x16_t sum[MS][NT];
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) sum[m][t] = zero;
#pragma unroll 1
    for (int i = 0; i < GB / 2 && !P::kPlainCodes; ++i) {
      const int g = 2 * i + kb;
      u32x4_t F[MS];
#pragma unroll
      for (int m = 0; m < MS; ++m) F[m] = *reinterpret_cast<const u32x4_t *>(at + (32 * m + ln) * R::XROW + ((g ^ turned(ln)) << 4));
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        float sv, bv;
        scale_and_bias(t, g, sv, bv);
        const Pieces p = split3(g < real ? __builtin_fmaf(P::kCentre, sv, bv) : 0.f);
        const u32x4_t o = {p.h | p.h << 16, p.h | p.m << 16, p.m | p.l << 16, 0u};
#pragma unroll
        for (int m = 0; m < MS; ++m) sum[m][t] = mfma<0>(F[m], o, sum[m][t]);
      }
    }
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 16; ++v) tot[m][t][v] += sum[m][t][v];
  };
  auto bias_stage = [&](int k, const unsigned char *at) __attribute__((always_inline)) {
    const int g0 = k >> glog, real = (k_end >> glog) - g0;  // (groups past the share's end are another share's)
    if constexpr (P::kPlainCodes) {
      const unsigned char *const mine = at + R::X + wave * R::W;
#pragma unroll
      for (int t = 0; t < NT; ++t) *reinterpret_cast<u32x4_t *>(scales + t * 1024 + lane * 16) = *reinterpret_cast<const u32x4_t *>(mine + t * 1024 + lane * 16);
      add_plain_biases<MS, NT>(tot, at, R::XROW, [&](int piece) __attribute__((always_inline)) { return (piece ^ turned(ln)) << 4; },
                               mine + NT * 1024 + ln * 32, real, ln, kb);
    } else if (in_place) {
      bias_product(at, real, [&](int t, int g, float &sv, float &bv) __attribute__((always_inline)) {
        const uint32_t from = first_scale[t] + g0 + (g < real ? g : 0);
        const T s1 = s_of[GLU ? t : 0][from];
        sv = as_f32(s1);
        bv = as_f32(b_of[GLU ? t : 0][from]);
        *reinterpret_cast<T *>(scales + scales_at[t] + g * 2) = s1;
      });
    } else {
      const unsigned char *const mine = at + R::X + wave * R::W;
#pragma unroll
      for (int t = 0; t < NT; ++t) *reinterpret_cast<u32x4_t *>(scales + t * 1024 + lane * 16) = *reinterpret_cast<const u32x4_t *>(mine + t * 1024 + lane * 16);
      bias_product(at, real, [&](int t, int g, float &sv, float &bv) __attribute__((always_inline)) {
        sv = as_f32(*reinterpret_cast<const T *>(mine + scales_at[t] + g * 2));
        bv = as_f32(*reinterpret_cast<const T *>(mine + NT * 1024 + scales_at[t] + g * 2));
      });
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };

  uint32_t xa[4], wa[2];  // this lane's pieces of a step
#pragma unroll
  for (int h = 0; h < 4; ++h) {
    const int piece = P::SPLIT ? 4 * (h >> 1) + 2 * kb + (h & 1) : 4 * kb + h;
    xa[h] = ln * R::XROW + ((piece ^ turned(ln)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) wa[i] = R::X + wave * R::W + ln * 64 + (((2 * i + kb) ^ ((ln >> 2) & 3)) << 4);
  // A stage of codes that begins k values into its window.  Program order is kept as it stands: behind every multiply a few of the
  // scaled additions of the sub-tile before it, the reads and the unpacking that the operands it was the last to use make room
  // for, and now and then one of the next stage's copies.
  constexpr int SUBS = P::JS * MS * P::NS;  // sub-tiles' groups of a stage
  auto code_stage = [&](int k, const unsigned char *at, int slot, int to) __attribute__((always_inline)) {
    f32x16_t acc[2][NT];  // the group sums being multiplied, and those before them, which are still to be scaled
    float pending_s[NT];
    const unsigned char *const sc = scales + (k >> glog) * 2;
    u32x4_t F[4], q[NT][P::NQ], op[NT][4];
    float s[NT][P::NS];
    auto fetch = [&](int j, int m, int h) __attribute__((always_inline)) {
      F[h] = *reinterpret_cast<const u32x4_t *>(at + (xa[h] ^ (j * 128)) + m * (32 * R::XROW));  // (the turn reaches over both steps of a row)
    };
    auto fetch_codes = [&](int j) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < P::NQ; ++i) q[t][i] = *reinterpret_cast<const u32x4_t *>(at + wa[BITS == 4 ? j : i] + t * 2048);
    };
    auto fetch_scales = [&](int j, float (&to)[NT][P::NS]) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < P::NS; ++i) to[t][i] = P::kUnit * as_f32(*reinterpret_cast<const T *>(sc + scales_at[t] + (G32 ? 2 * j + i : j >> scale_shift) * 2));
    };
    fetch_codes(0);
#pragma unroll
    for (int h = 0; h < 4; ++h) fetch(0, 0, h);
    fetch_scales(0, s);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      P::deal(q[t]);
#pragma unroll
      for (int h = 0; h < 4; ++h) P::unpack(q[t], h, op[t][h]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < P::JS; ++j) {
      float s_next[NT][P::NS];
      if (j + 1 < P::JS) {
        fetch_codes(j + 1);
        fetch_scales(j + 1, s_next);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int m = 0; m < MS; ++m) {
        const bool more = m + 1 < MS || j + 1 < P::JS;
        const int nj = m + 1 < MS ? j : j + 1, nm = m + 1 < MS ? m + 1 : 0;
#pragma unroll
        for (int i = 0; i < P::NS; ++i) {
          const int sub = (j * MS + m) * P::NS + i, cur = sub & 1;
          const int pm = i > 0 ? m : (m > 0 ? m - 1 : MS - 1);  // the pending sub-tile
          constexpr int SLOTS = 4 / P::NS * NT, EACH = 16 * NT / SLOTS, PLACES = SUBS * SLOTS;
          constexpr int W_FROM = P::JS == 1 ? PLACES / 2 : PLACES / P::JS * (P::JS - 1);  // (the last step's codes have been read)
          if (m == MS - 1 && i == 0 && j + 1 < P::JS) {
#pragma unroll
            for (int t = 0; t < NT; ++t) P::deal(q[t]);
          }
#pragma unroll
          for (int n = 0; n < SLOTS; ++n) {
            const int h = 4 / P::NS * i + n / NT, t = n % NT, place = sub * SLOTS + n;
            acc[cur][t] = mfma<DT>(F[h], op[t][h], n < NT ? zero : acc[cur][t]);
#pragma unroll
            for (int v = n * EACH; v < (n + 1) * EACH && sub > 0; ++v)
              tot[pm][v / 16][v % 16] = __builtin_fmaf(pending_s[v / 16], acc[cur ^ 1][v / 16][v % 16], tot[pm][v / 16][v % 16]);
            if (t == NT - 1 && more) fetch(nj, nm, h);
            if (m == MS - 1 && j + 1 < P::JS) P::unpack(q[t], h, op[t][h]);
#pragma unroll
            for (int c = R::XI * place / W_FROM; c < R::XI * (place + 1) / W_FROM && place < W_FROM; ++c) copy_x(to, c);
#pragma unroll
            for (int c = 2 * NT * (place - W_FROM) / (PLACES - W_FROM); c < 2 * NT * (place - W_FROM + 1) / (PLACES - W_FROM) && place >= W_FROM; ++c)
              copy_w(slot, c);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int t = 0; t < NT; ++t) pending_s[t] = s[t][i];
        }
      }
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < P::NS; ++i) s[t][i] = j + 1 < P::JS ? s_next[t][i] : 0.f;
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[MS - 1][t][v] = __builtin_fmaf(pending_s[t], acc[(SUBS - 1) & 1][t][v], tot[MS - 1][t][v]);
  };

  copy_weights(0);
  advance(next_w);
#pragma unroll
  for (int p = 0; p < S - 1; ++p) {
    copy_rows(p);
    advance(next_x);
    copy_weights(p + 1);
    advance(next_w);
  }
  int slot = 0, to = S - 1, left = total;
  auto begin = [&]() __attribute__((always_inline)) {  // this stage's copies have arrived, in every wave, and its predecessor's rows are read
    wait_copies<2 * NT + (S - 2) * R::COPIES>();
    block_barrier();
  };
  auto end = [&]() __attribute__((always_inline)) {
    advance(next_x);
    advance(next_w);
    slot = slot + 1 == S ? 0 : slot + 1;
    to = to + 1 == S ? 0 : to + 1;
    --left;
  };
  for (int k = k_first; k < k_end;) {
    const int k_window = k, k_last = k + per_window * R::KS < k_end ? k + per_window * R::KS : k_end;
    begin();
    copy_rows(to);
    bias_stage(k, ring + slot * R::STAGE);
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    copy_weights(slot);
    end();
#pragma unroll 1
    for (; k < k_last; k += R::KS) {
      begin();
      code_stage(k - k_window, ring + slot * R::STAGE, slot, to);
      end();
    }
  }
  for (; KW > 1 && left > 0; --left) {  // (the last share may be a shorter one)
    wait_copies<0>();
    block_barrier();
  }
  uint32_t dst[2] = {};
  if constexpr (LIST && !GLU) output_rows(a, row0, rows, lane, dst);
  wait_copies<0>();
  block_barrier();

  if constexpr (KW > 1) {  // the K groups' sums meet in LDS, added in group order
    constexpr int kPiece = 64 * WN * 4;
    float *const parts = reinterpret_cast<float *>(lds_raw) + (wave * 64 + lane) * 4;  // 16-byte pieces, lane by lane
#pragma unroll
    for (int g = 1; g < KW; ++g) {
#pragma unroll
      for (int m = 0; m < MS; ++m)
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
          for (int r = 0; r < 4; ++r)
            if (kg == g)
              *reinterpret_cast<float4 *>(parts + ((m * NT + t) * 4 + r) * kPiece) =
                  make_float4(tot[m][t][4 * r], tot[m][t][4 * r + 1], tot[m][t][4 * r + 2], tot[m][t][4 * r + 3]);
      __syncthreads();
      if (kg == 0) {
#pragma unroll
        for (int m = 0; m < MS; ++m)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
              const float4 v = *reinterpret_cast<const float4 *>(parts + ((m * NT + t) * 4 + r) * kPiece);
              tot[m][t][4 * r] += v.x;
              tot[m][t][4 * r + 1] += v.y;
              tot[m][t][4 * r + 2] += v.z;
              tot[m][t][4 * r + 3] += v.w;
            }
      }
      __syncthreads();
    }
    if (kg != 0) return;
  }

  if constexpr (LIST) write_piece<GLU, MS>(a, tot, wave, lane, n0, row0, rows, ebase, weight_row, dst, lds_raw);
  else write_tile<DT, BITS, MS, NT, WN>(a, tot, wave, lane, col0, row0, rows, glog, weight_row, lds_raw);
}


// A tile of 65 to 128 token rows of a block with 4-bit codes in groups of 64: 32 MS rows x 256 weight rows by four waves, each of which owns 64 weight rows
// (GLU: 32 gate and 32 up rows) for all the token rows.  What multiply_tile does, with the pipeline that so many sums a wave leave room for:
//   token rows  two places of 64 K values, one barrier each; copied while the other place is multiplied;
//   codes       two places of 128 K values, the wave's own; unpacked while the last token rows of the 64 values before are multiplied.
// Two blocks share a CU and fill each other's waits.
// What bounds it: 2048 cycles of matrix work a wave and 128 K values beside 1640 of vector instructions (256 scaled additions, 112 of unpacking), the reads of
// LDS, and the clock, 1.8 to 1.9 GHz under all of them on a warm card: a copy of the loop alone, fed from LDS, reached 1390 TFLOP/s.  65536 rows of 128 experts, K = 2048,
// 1536 columns 504 us = 818 TFLOP/s; K = 4096, 3072 columns 948 (tiles of 256 x 256 with their weights dequantised once a block 764 and 900, all classes).  A block
// takes 77 us a slot at K = 2048, some 12 of them its ends.  Counters, 32 620 rows, gate/up: matrix units 0.47 busy, 9.1 vector instructions a multiply with all that is
// outside the loop.  GLU keeps 18 registers a lane in scratch memory around the loop over windows (else 12): 27 of the 81 MB that gate/up writes, 23 of down's 157.
struct LongRing {
  static constexpr int XROW = 128, W = 4096, WALL = 4 * W, WINDOWS = 4 * 2048;
  static constexpr int bytes(int ms) { return 2 * (32 * ms * XROW) + 2 * WALL + WINDOWS + ms * 1024; }
};
template <bool GLU, int MS>
__device__ __forceinline__ void multiply_long_tile(const CodesArgs &a, int e, int64_t row0, int rows, int n0, unsigned char *lds_raw) {
  typedef Tile<0, 4, false, true, MS, 2, 4, 2> P;
  typedef LongRing R;
  constexpr int NM = GLU ? 2 : 1, X = 32 * MS * R::XROW, XI = MS;  // copies a wave makes of a place of token rows
  const int lane = threadIdx.x & 63, ln = lane & 31, kb = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = a.N, K = a.K, G = K >> 6, row_bytes = K / 2, ext = padded_groups(G) * sum_slots(true);
  const int64_t ebase = (int64_t)e * N;
  const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds_raw;
  unsigned char *const codes_at = lds_raw + 2 * X + wave * R::W, *const scales = lds_raw + 2 * X + 2 * R::WALL + wave * 2048;
  const i32x4_t xr = words_of(a.x, (uint32_t)(a.x_rows * K * 2)), xsr = words_of(a.sums, (uint32_t)(a.x_rows * ext * 2));
  i32x4_t wr[NM], sr[NM], br[NM];
#pragma unroll
  for (int t = 0; t < NM; ++t) {
    wr[t] = words_of((t ? a.w1 : a.w0) + ebase * (row_bytes / 4), (uint32_t)N * row_bytes);
    sr[t] = words_of(static_cast<const uint16_t *>(t ? a.s1 : a.s0) + ebase * G, (uint32_t)N * G * 2);
    br[t] = words_of(static_cast<const uint16_t *>(t ? a.b1 : a.b0) + ebase * G, (uint32_t)N * G * 2);
  }
  const int col0 = n0 + (GLU ? 32 : 64) * wave;
  auto weight_row = [&](int t, int at) __attribute__((always_inline)) {
    const int p = GLU ? (at & ~7) | value_at_place(a.y_order, at & 7) : at, row = col0 + (GLU ? 0 : 32 * t) + p;
    return row < N ? row : N - 1;
  };
  auto turned = [](int row) __attribute__((always_inline)) { return (row >> 1) & 7; };
  uint32_t x_off[XI], w_off[4], window_row[2];
  uint32_t *const sums_off = reinterpret_cast<uint32_t *>(lds_raw + 2 * X + 2 * R::WALL + R::WINDOWS) + wave * (64 * XI) + lane;  // (read once a window)
#pragma unroll
  for (int i = 0; i < XI; ++i) {
    const int r = (wave * XI + i) * 8 + lane / 8, tr = r < rows ? r : rows - 1;  // rows past the end repeat the last one (never stored)
    const uint32_t row = a.src_rows ? a.src_rows[row0 + tr] : (uint32_t)(row0 + tr), piece = (uint32_t)((lane % 8) ^ turned(r)) << 4;
    x_off[i] = row * (uint32_t)(K * 2) + piece;
    sums_off[64 * i] = row * (uint32_t)(ext * 2) + piece;
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int at = 16 * (i & 1) + (lane >> 2);
    w_off[i] = (uint32_t)weight_row(i / 2, at) * row_bytes + (((lane & 3) ^ ((at >> 2) & 3)) << 4);
  }
#pragma unroll
  for (int t = 0; t < 2; ++t) window_row[t] = (uint32_t)weight_row(t, lane >> 1) * G * 2 + ((lane & 1) << 4);

  // ---- copies.  K runs in windows of 16 groups; place 0 of a window is its bias product (group sums; scales and biases), then come its K values.
  struct Next { int k, pos; } next_x = {0, 0}, next_w = {0, 0};
  int xs = 0, ws = 0;  // the places being read
  auto copy_rows = [&](int slot, auto sums_too) __attribute__((always_inline)) {  // sums_too: a window's group sums may be what comes next
    const int k = next_x.k < K ? next_x.k : K - 64;  // (past the end the last ones again)
    const bool sums = decltype(sums_too)::value && next_x.pos == 0;
    i32x4_t from;
#pragma unroll
    for (int w = 0; w < 4; ++w) from[w] = sums ? xsr[w] : xr[w];
#pragma unroll
    for (int c = 0; c < XI; ++c) {
      uint32_t off = x_off[c];
      if constexpr (decltype(sums_too)::value) {
        const uint32_t other = sums_off[64 * c];
        off = sums ? other : off;
      }
      copy_to_lds(from, off, sums ? (k >> 6) * 8 : k * 2, ring_at + slot * X + (wave * XI + c) * 1024);
    }
    if (!sums) next_x.k += 64;
    next_x.pos = next_x.pos == 16 ? 0 : next_x.pos + 1;
  };
  auto copy_weights = [&](int slot) __attribute__((always_inline)) {
    const int k = next_w.k < K ? next_w.k : K - 128;
    const bool bias = next_w.pos == 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {  // codes: two copies a tile; bias product: the tiles' scales, then their biases
      i32x4_t from;
#pragma unroll
      for (int w = 0; w < 4; ++w) from[w] = bias ? (i < 2 ? sr : br)[GLU ? i % 2 : 0][w] : wr[GLU ? i / 2 : 0][w];
      copy_to_lds(from, bias ? window_row[i % 2] : w_off[i], bias ? (k >> 6) * 2 : k / 2, ring_at + 2 * X + slot * R::WALL + wave * R::W + i * 1024);
    }
    if (!bias) next_w.k += 128;
    next_w.pos = next_w.pos == 8 ? 0 : next_w.pos + 1;
  };

  float tot[MS][2][16];
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[m][t][v] = 0.f;
  const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t acc[2] = {zero, zero};  // the group sums being multiplied, and those before them, which are still to be scaled
  float pending_s = 0.f;
  u32x4_t op[2][4], q[2][1];  // the codes of 64 K values as operands, and as they are
  uint32_t xa[4], wa[2];
#pragma unroll
  for (int h = 0; h < 4; ++h) xa[h] = ln * R::XROW + (((4 * kb + h) ^ turned(ln)) << 4);
#pragma unroll
  for (int i = 0; i < 2; ++i) wa[i] = ln * 64 + (((2 * i + kb) ^ ((ln >> 2) & 3)) << 4);
  auto fetch_codes = [&](int slot, int half) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < 2; ++t) q[t][0] = *reinterpret_cast<const u32x4_t *>(codes_at + slot * R::WALL + wa[half] + t * 2048);
  };

  // 64 K values: the token rows from place xs, the operands in registers; those of the 64 values behind are made on the way, from half next_half of
  // place next_slot.  Program order is kept as it stands.
  auto multiply = [&](int group, int next_slot, int next_half, auto await) __attribute__((always_inline)) {
    const unsigned char *const at = lds_raw + xs * X;
    u32x4_t F[4];
#pragma unroll
    for (int h = 0; h < 4; ++h) F[h] = *reinterpret_cast<const u32x4_t *>(at + xa[h]);
    float s[2];
#pragma unroll
    for (int t = 0; t < 2; ++t) s[t] = as_f32(*reinterpret_cast<const uint16_t *>(scales + t * 1024 + ln * 32 + group * 2));
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      if (m == MS - 1) {
        await();
        fetch_codes(next_slot, next_half);
      }
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int cur = t, pm = t ? m : (m ? m - 1 : MS - 1), pt = t ^ 1;  // the pending sums' place
#pragma unroll
        for (int h = 0; h < 4; ++h) {
          acc[cur] = mfma<0>(F[h], op[t][h], h ? acc[cur] : zero);
#pragma unroll
          for (int v = 4 * h; v < 4 * h + 4; ++v) tot[pm][pt][v] = __builtin_fmaf(pending_s, acc[cur ^ 1][v], tot[pm][pt][v]);
          if (t == 1 && m + 1 < MS) F[h] = *reinterpret_cast<const u32x4_t *>(at + xa[h] + (m + 1) * (32 * R::XROW));
          if (m == MS - 1) P::unpack(q[t], h, op[t][h]);
          __builtin_amdgcn_sched_barrier(0);
        }
        pending_s = s[t];
      }
    }
  };
  auto begin = [&](auto left) __attribute__((always_inline)) {  // what this step reads has arrived, in every wave, and the place copied to next is free
    wait_copies<decltype(left)::value>();
    block_barrier();
  };
  const std::integral_constant<int, 0> all{};
  const std::integral_constant<int, 4> but_codes{};

  const std::true_type yes{};
  const std::false_type no{};
  copy_rows(0, yes);
  copy_weights(0);
  for (int k = 0; k < K;) {
    const int k_window = k, k_last = k + 1024 < K ? k + 1024 : K;
    begin(all);
    copy_rows(xs ^ 1, no);
    copy_weights(ws ^ 1);
    {
      const unsigned char *const mine = codes_at + ws * R::WALL;
#pragma unroll
      for (int t = 0; t < 2; ++t) *reinterpret_cast<u32x4_t *>(scales + t * 1024 + lane * 16) = *reinterpret_cast<const u32x4_t *>(mine + t * 1024 + lane * 16);
      add_plain_biases<MS, 2>(tot, lds_raw + xs * X, R::XROW, [&](int piece) __attribute__((always_inline)) { return (piece ^ turned(ln)) << 4; },
                              mine + 2048 + ln * 32, (K - k) >> 6, ln, kb);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
    xs ^= 1;
    ws ^= 1;
    wait_copies<0>();  // (this wave's codes: unpacked ahead of the barrier)
    fetch_codes(ws, 0);
#pragma unroll
    for (int t = 0; t < 2; ++t)
#pragma unroll
      for (int h = 0; h < 4; ++h) P::unpack(q[t], h, op[t][h]);
#pragma unroll 1
    for (; k < k_last; k += 128) {
      begin(all);
      copy_rows(xs ^ 1, no);
      copy_weights(ws ^ 1);
      multiply((k - k_window) >> 6, ws, 1, [] {});
      xs ^= 1;
      begin(but_codes);
      copy_rows(xs ^ 1, yes);
      multiply(((k - k_window) >> 6) + 1, ws ^ 1, 0, [&]() __attribute__((always_inline)) {  // the next codes were asked for before the rows
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(XI) : "memory");
      });
      xs ^= 1;
      ws ^= 1;
    }
    // (the window's last sums ahead of the next one's bias product: every sum in the order of multiply_tile, wherever its row stands)
#pragma unroll
    for (int v = 0; v < 16; ++v) tot[MS - 1][1][v] = __builtin_fmaf(pending_s, acc[1][v], tot[MS - 1][1][v]);
    pending_s = 0.f;
  }
  uint32_t dst[2] = {};
  if constexpr (!GLU) output_rows(a, row0, rows, lane, dst);
  wait_copies<0>();
  block_barrier();
  write_piece<GLU, MS>(a, tot, wave, lane, n0, row0, rows, ebase, weight_row, dst, lds_raw);
}

// The tiles of a list of pieces of up to 128 rows (ShortTiles::piece), 4-bit codes in groups of 64: by their rows, 32 at a time.
// Ids are dealt round-robin over the 8 XCDs, whole pieces to each (the blocks of one share its gathered rows).  Two or four pieces that follow each other in the
// list on one XCD: fewer bytes (an expert's weights are read once by every XCD that has a piece of it), 0 to 2 % slower.
template <bool GLU>
__global__ __launch_bounds__(256, 2) void qmm_pieces_kernel(CodesArgs a, const uint32_t *__restrict__ list, int n_ntiles) {
  constexpr int NI = GLU ? 128 : 256;
  const uint32_t xcd = blockIdx.x & 7, j = blockIdx.x >> 3, id = j / (uint32_t)n_ntiles * 8u + xcd;
  const int nt = (int)(j % (uint32_t)n_ntiles);
  if (id >= list[0]) return;
  const uint4 rec = reinterpret_cast<const uint4 *>(list)[1 + id];
  const int e = __builtin_amdgcn_readfirstlane((int)rec.x), rows = __builtin_amdgcn_readfirstlane((int)rec.z);
  const int64_t row0 = (int64_t)__builtin_amdgcn_readfirstlane((int)rec.y);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  if (rows > 96) return multiply_long_tile<GLU, 4>(a, e, row0, rows, nt * NI, lds_raw);
  if (rows > 64) return multiply_long_tile<GLU, 3>(a, e, row0, rows, nt * NI, lds_raw);
  if (rows > 32) return multiply_tile<0, 4, false, true, GLU, 2, 2, 4, 1, 2>(a, e, row0, rows, nt * NI, 0, lds_raw);
  typedef Ring<4, 1, 2, 4, 2> Short;
  constexpr int S1 = (kHalfLds - 4 * Short::WINDOW) / Short::STAGE;  // as many stages as fit
  multiply_tile<0, 4, false, true, GLU, 1, 2, 4, 1, S1>(a, e, row0, rows, nt * NI, 0, lds_raw);
}

// A block computes 32 MS token rows x 32 WN weight rows with WN KW waves (see multiply_tile), tiles of up to 32 rows with half the
// token operand.
template <int DT, int BITS, bool G32, int MS, int NT, int WN, int KW, int S>
__global__ __launch_bounds__(64 * WN * KW, waves_of(WN * KW, lds_of(KW, Ring<BITS, MS, NT, WN, S>::BYTES))) void qmm_tiles_kernel(
    CodesArgs a, int n_mtiles, int n_ntiles, int scale_shift) {
  constexpr int BM = 32 * MS, NI = 32 * WN * NT;
  // block -> (M tile, N tile).  Ids are dealt round-robin over the 8 XCDs: an XCD takes every eighth N tile
  // and all M tiles of it, so its L2 holds the weights of a few N tiles and x streams through.
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3, nt = j / n_mtiles * 8 + xcd;
  if (nt >= n_ntiles) return;
  const int64_t row0 = (int64_t)(j % n_mtiles) * BM;
  const int rows = a.M - row0 < BM ? (int)(a.M - row0) : BM;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  if constexpr (MS > 1) {
    if (rows <= 32) {
      typedef Ring<BITS, 1, NT, WN, 2> Short;
      constexpr int S1 = (lds_of(KW, Ring<BITS, MS, NT, WN, S>::BYTES) / KW - WN * Short::WINDOW) / Short::STAGE;  // as many stages as fit
      multiply_tile<DT, BITS, G32, false, false, 1, NT, WN, KW, S1>(a, 0, row0, rows, nt * NI, scale_shift, lds_raw);
      return;
    }
  }
  multiply_tile<DT, BITS, G32, false, false, MS, NT, WN, KW, S>(a, 0, row0, rows, nt * NI, scale_shift, lds_raw);
}

size_t codes_copy_bytes(int bits, int64_t rows, int K) {
  return row_order(bits) != RowOrder::kPlain ? (size_t)rows * K * 2 : 0;
}
size_t codes_sums_bytes(int64_t rows, int K, int group, bool plain) { return (size_t)rows * padded_groups(K / group) * sum_slots(plain) * 2; }

PrepareArgs prepare_args(const void *x, int64_t rows, int K, int group, uint16_t *copy, uint16_t *sums, bool plain) {
  PrepareArgs a;
  a.x = x;
  a.octets = rows * (K / 8);
  a.octets_per_row = K / 8;
  a.lanes_log2 = group == 32 ? 2 : (group == 64 ? 3 : 4);
  a.copy = copy;
  a.sums = sums;
  a.sums_row = padded_groups(K / group) * sum_slots(plain);
  a.slots = sum_slots(plain);
  return a;
}
hipError_t launch_prepare_rows(const void *x, int64_t rows, int K, int group, int dt, bool list, uint16_t *copy,
                               uint16_t *sums, hipStream_t st) {
  const PrepareArgs a = prepare_args(x, rows, K, group, copy, sums, false);
  if (a.octets == 0) return hipSuccess;
  const unsigned grid = (unsigned)((a.octets + 255) / 256);
  if (dt == 0 && list) prepare_rows_kernel<0, RowOrder::kQuads><<<grid, 256, 0, st>>>(a);
  else if (dt == 0) prepare_rows_kernel<0, RowOrder::kPaired><<<grid, 256, 0, st>>>(a);
  else if (dt == 1 && !list) prepare_rows_kernel<1, RowOrder::kPaired><<<grid, 256, 0, st>>>(a);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

template <int DT, int BITS, bool G32, int MS, int NT, int WN, int KW, int S>
static hipError_t start_tiles(const CodesArgs &a, int scale_shift, hipStream_t st) {
  constexpr int NI = 32 * WN * NT, BM = 32 * MS;
  constexpr int bufs = lds_of(KW, Ring<BITS, MS, NT, WN, S>::BYTES), sums = KW > 1 ? BM * 32 * WN * NT * 4 : 0;
  constexpr int lds = bufs > sums ? bufs : sums;
  static_assert(lds <= 160 * 1024, "more LDS than a CU has");
  const int n_ntiles = (a.N + NI - 1) / NI, mtiles = (int)((a.M + BM - 1) / BM);
  const int64_t grid = (int64_t)((n_ntiles + 7) / 8) * 8 * mtiles;
  if (grid <= 0 || grid > INT32_MAX) return hipErrorInvalidValue;
  const auto kernel = &qmm_tiles_kernel<DT, BITS, G32, MS, NT, WN, KW, S>;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> allowed{0};
    if (hipError_t e = allow_lds(reinterpret_cast<const void *>(kernel), (int)lds, allowed); e != hipSuccess) return e;
  }
  launch_or_time(kernel, dim3((unsigned)grid), dim3(64 * WN * KW), lds, st, a, mtiles, n_ntiles, scale_shift);
  return hipGetLastError();
}

// Which tile: long_tile_rows, else dense_tile (dense_rule.hpp).  Before those rules, us of the whole call, bf16 4-bit / f16 8-bit, groups of 64 (M, N, K):
//                                       (96, 4096, 4096) (200, 4096, 4096) (1000, 1024, 4096) (400, 4096, 4096) (640, 2304, 2304) (777, 4096, 4096) (2048, 4096, 4096)
//   32 x 64, K shared by four groups       16.9 / 17.5      29.0 / 24.6       40.1 / 28.8        55.7 / 45.1       43.5 / 33.6       102 / 90          - / 211
//   32 x 128, four groups                  21.5 / 22.3      25.8 / 27.2       31.2 / 31.9        49.7 / 52.8       35.8 / 37.0       94 / 106          - / 214
//   32 x 128, two groups                   22.9 / 25.0      27.7 / 31.0       34.3 / 35.3        42.7 / 40.1       29.6 / 26.5       79 / 81           - / 178
//   64 x 256, two groups, 2 tiles a wave   41 / 46          48.9 / 48.1       55.0 / 52.6        53.7 / 50.9       38.3 / 35.0       58.8 / 57.8       - / 124
//   64 x 128, two groups                   32 / 31          - / 33.1          - / 37.1           - / 36.2          - / 25.4          - / 56.6          - / 123
//   64 x 256, one group, 2 tiles a wave    51 / 59          - / 60.9          - / 62.0           - / 61.7          - / 39.9          - / 69.5          - / 114
//   64 x 128, two groups, codes loaded into registers (qmm_codes.hip)
//                                          - / -            32.4 / 32.9       37.9 / 36.0        37.1 / 34.9       26.9 / 25.4       63.4 / 60.4       - / 124
// (8-bit, 64 x 128 and two groups here against registers, 777 x 4096 x 4096 and 900 x 4096 x 2048, either type, any group: 0.3 to 5 us slower.)
// bf16 takes the larger tiles (2048 rows) in qmm_large.hip.
template <int DT, int BITS, bool G32>
static hipError_t start_dense(const CodesArgs &a, int group, hipStream_t st) {
  const int scale_shift = group == 128, longer = long_tile_rows(a.M, a.N, a.K, BITS);
  if (longer == 96) return start_tiles<DT, BITS, G32, 3, 1, 4, 2, BITS == 4 ? 2 : 3>(a, scale_shift, st);
  if constexpr (BITS == 8)
    if (longer == 128) return start_tiles<DT, BITS, G32, 4, 1, 4, 2, 3>(a, scale_shift, st);
  switch (dense_tile(a.M, a.N, a.K, BITS, group, DT == 0)) {
    case DenseTile::k32x64: return start_tiles<DT, BITS, G32, 1, 1, 2, 4, 2>(a, scale_shift, st);
    case DenseTile::kRegisters32x64: return launch_qmm_codes_small(a, st);
    case DenseTile::k32x128:
      if constexpr (BITS == 4) return start_tiles<DT, BITS, G32, 1, 1, 4, 4, 2>(a, scale_shift, st);
      break;
    case DenseTile::k64x256: return start_tiles<DT, BITS, G32, 2, 2, 4, BITS == 4 ? 2 : 1, 2>(a, scale_shift, st);
    case DenseTile::kRegisters64x128: return launch_qmm_codes_middle(a, false, group, BITS, DT, st);
    case DenseTile::kRegisters64x128Shared: return launch_qmm_codes_middle(a, true, group, BITS, DT, st);
  }
  return hipErrorInvalidValue;
}

// The tiles of a list of pieces in one launch (see qmm_pieces_kernel).
template <bool GLU>
static hipError_t start_pieces(const CodesArgs &a, const uint32_t *list, int cap, hipStream_t st) {
  constexpr int NI = GLU ? 128 : 256, lds = kHalfLds;
  static_assert(LongRing::bytes(4) <= lds && Ring<4, 2, 2, 4, 2>::BYTES <= lds, "two blocks share a CU");
  const int n_ntiles = (a.N + NI - 1) / NI;
  const int64_t grid = ((int64_t)cap + 7) / 8 * 8 * n_ntiles;
  if (grid <= 0 || grid > INT32_MAX) return hipErrorInvalidValue;
  static std::atomic<uint64_t> allowed{0};
  if (hipError_t e = allow_lds(reinterpret_cast<const void *>(&qmm_pieces_kernel<GLU>), lds, allowed); e != hipSuccess) return e;
  launch_or_time(&qmm_pieces_kernel<GLU>, dim3((unsigned)grid), dim3(256), lds, st, a, list, n_ntiles);
  return hipGetLastError();
}
hipError_t launch_qmm_pieces(const CodesArgs &a, const uint32_t *list, int cap, bool glu, hipStream_t st) {
  return glu ? start_pieces<true>(a, list, cap, st) : start_pieces<false>(a, list, cap, st);
}

hipError_t launch_qmm_codes_dense(const CodesArgs &a, int group, int bits, int dt, hipStream_t st) {
  if (a.M == 0) return hipSuccess;
  auto with_group = [&](auto d, auto b) {
    constexpr int DT = decltype(d)::value, BITS = decltype(b)::value;
    return group == 32 ? start_dense<DT, BITS, true>(a, group, st) : start_dense<DT, BITS, false>(a, group, st);
  };
  auto with_bits = [&](auto d) {
    return bits == 4 ? with_group(d, std::integral_constant<int, 4>{}) : with_group(d, std::integral_constant<int, 8>{});
  };
  if (dt == 0) return with_bits(std::integral_constant<int, 0>{});
  if (dt == 1) return with_bits(std::integral_constant<int, 1>{});
  return hipErrorInvalidValue;
}

}  // namespace mi_moe
