// Quantized products of a few rows (a decode batch's linear layer; short expert segments with groups of 32 or 128):
// activations in bfloat16 or float16, groups of 32, 64 or 128.
//
// Contract: mlx_quantized_matmul / mlx_gather_qmm with transpose = true (mlx-rs/src/ops/quantization.rs:91-122,160-230);
// with GLU also nn::silu and multiply (nn/activation.rs:142-144,876-880).
//
// Arithmetic as in the tiled product on raw codes (qmm_codes.hip): sum_c x_c (s q_c + b) = s sum_c x_c q_c + b sum_c x_c
// per group with centred codes, unrounded on the matrix cores, fp32 sums; the same precision as plain sums have (results that
// are not the float64 product's nearest value, plain / codes as they are or 128 + q / centred: bf16 4-bit 1.0e-4 / 1.7e-3 / 1.0e-4, f16
// 1.1e-3 / 1.4e-3 / 8e-4).  Here the bias term is fp32 vector work: a tile is 16
// tokens by 16 weight rows (v_mfma_f32_16x16x32), so it is four fma a lane and group.
#include <type_traits>

#include "qmm_dev.hpp"

namespace mi_moe {

namespace {

constexpr int kTokens = 16;  // token slots of a tile
constexpr int kRing = 4;     // 16-byte code loads in flight per lane and matrix (8: no change at any size)

// Two bytes 0 to 15 as bf16, the lower or the upper ones of v: below 16 an e4m3 number is its byte in units of 2^-9.
template <int UPPER>
__device__ __forceinline__ uint32_t small_codes(uint32_t v) {
  return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 512.0f, UPPER != 0));
}
// LDS of a launch: token rows of sk values (tt of them), 64 zero bytes, the sums of x over each group and
// token slot, the (scale, bias) pairs of the block's weight rows, and the partial sums of a shared K.
struct RowsLds {
  int x_stride, zeros, sums, pairs, pair_row, parts, bytes;
  __host__ __device__ RowsLds(int group, int nm, int kw, int K, int sk, int tt) {
    const int nw = 4 / kw;
    x_stride = 2 * sk + 16;
    zeros = tt * x_stride;
    sums = zeros + 64;
    pairs = sums + sk / group * kTokens * 4;
    pair_row = (K / group) * 4 + 4;  // (an odd number of words: 16 rows read one group each without a conflict)
    parts = pairs + ((nw * nm * 16 * pair_row + 15) & ~15);
    bytes = parts + (kw > 1 ? kw * nw * nm * 64 * 16 : 0);
  }
};

}  // namespace

// One block: 16 * 4 / KW weight rows (GLU: of both matrices) of one expert times up to 16 token rows a pass; KW waves
// share the K of a row tile, chunk by chunk.  A lane (weight row l % 16, quarter l / 16) loads 16 bytes: 32 4-bit codes or
// 16 8-bit codes.  A multiply takes 32 K values, eight a lane, and must stay inside one group:
//   4-bit: the four quarters of a row hold 32 consecutive codes each; four lane swaps transpose words against quarters,
//   so that multiply s takes codes 32 s .. 32 s + 31;
//   8-bit: multiply t takes the t-th half of every quarter (groups >= 64), or after two swaps 32 consecutive codes.
// What bounds it: the bytes of the weights and, for one row of a small matrix, the latency of its few dependent steps.
// Measured, 4096 x 4096, us of the kernel at 2 / 4 / 8 / 16 rows (the plain kernel, a wave per output element: f16 4-bit
// 17.5 / 30.2 / 55.6 from 4 rows on): f16 4-bit 7.2 / 8.5 / 11.7 / 17.2, bf16 groups of 32 7.4 / 8.7 / 11.8 / 17.0.  Every block
// stages all rows: that is what grows.
template <int DT, int BITS, int GROUP, bool GLU, int KW>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3, 8))) void qmm_rows_kernel(RowsArgs a, int tt, int sk) {
  typedef typename ElemOf<DT>::type T;
  constexpr int NM = GLU ? 2 : 1;
  constexpr int NW = 4 / KW;
  constexpr int CH = BITS == 4 ? 128 : 64;     // codes per chunk and row
  constexpr int MUL = CH / 32;                 // multiplies per chunk
  // 4-bit codes in bf16 come out of their conversion as they are; a group's sum starts from -8 times that of x instead, which is
  // what the sums of x in LDS hold then.
  constexpr bool kStart = BITS == 4 && DT == 0;
  constexpr bool PAIRED = BITS == 4;  // token rows as 8-blocks (0,4)(1,5)(2,6)(3,7), bf16 (0,2)(1,3)(4,6)(5,7): the order of the unpacking

  int e = 0, cnt = (int)a.M;
  int64_t r0 = 0;
  bool inline_src = false;
  if (a.work) {
    const uint4 rec = reinterpret_cast<const uint4 *>(a.work)[(size_t)blockIdx.y * 4];
    e = (int)rec.x;
    r0 = rec.y;
    cnt = (int)rec.z;
    inline_src = a.src_in_work && rec.w != 0u;
    if (cnt == 0) return;
  }
  const int lane = lane_id(), tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave % KW, wn = wave / KW;
  const int c = lane & 15, kb = lane >> 4;
  const int N = a.N, K = a.K;
  const int n0 = (blockIdx.x * NW + wn) * 16;
  const int G = K / GROUP, row_bytes = K * BITS / 8, nchunks = K / CH;
  const int64_t ebase = (int64_t)e * N;

  extern __shared__ __align__(16) unsigned char lds[];
  const RowsLds L(GROUP, NM, KW, K, sk, tt);
  float *const sums = reinterpret_cast<float *>(lds + L.sums);

  __amdgpu_buffer_rsrc_t wr[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) wr[m] = rsrc_of((m ? a.w1 : a.w0) + ebase * (row_bytes / 4), (uint32_t)N * row_bytes);
  const uint32_t w_voff = (uint32_t)(n0 + c) * row_bytes + kb * 16;  // rows >= N read zeros

  struct Codes {
    u32x4_t q[NM];
  };
  Codes ring[kRing];
  auto issue = [&](int j, Codes &R) __attribute__((always_inline)) {  // the wave's j-th chunk; unconditional (clamped)
    int ch = wk + KW * j;
    ch = ch < nchunks ? ch : nchunks - 1;
#pragma unroll
    for (int m = 0; m < NM; ++m) R.q[m] = __builtin_amdgcn_raw_buffer_load_b128(wr[m], w_voff, ch * 64, 0);
  };
#pragma unroll
  for (int d = 0; d < kRing; ++d) issue(d, ring[d]);

  // (scale, bias) pairs of the block's rows, one LDS read per group and row later on.  The 16 rows of a tile are 16 G
  // consecutive values of each tensor, 16-byte aligned.
  {
    constexpr int PV = 16 / (int)sizeof(T);
    const int per_tile = 16 * G / PV, total = NW * NM * per_tile;
    for (int p = tid; p < total; p += 256) {
      const int tile = p / per_tile, q = p - tile * per_tile;  // tile = wn * NM + m
      const int m = tile % NM, row0 = (blockIdx.x * NW + tile / NM) * 16;
      const __amdgpu_buffer_rsrc_t sr = rsrc_of(static_cast<const T *>(m ? a.s1 : a.s0) + ebase * G, (uint32_t)N * G * sizeof(T));
      const __amdgpu_buffer_rsrc_t br = rsrc_of(static_cast<const T *>(m ? a.b1 : a.b0) + ebase * G, (uint32_t)N * G * sizeof(T));
      const uint32_t off = ((uint32_t)row0 * G + q * PV) * sizeof(T);
      const u32x4_t sv = __builtin_amdgcn_raw_buffer_load_b128(sr, off, 0, 0), bv = __builtin_amdgcn_raw_buffer_load_b128(br, off, 0, 0);
      int row = q * PV / G, g = q * PV - row * G;
      unsigned char *to = lds + L.pairs + (tile * 16 + row) * L.pair_row + g * 2 * (int)sizeof(T);
#pragma unroll
      for (int i = 0; i < PV; ++i) {
        *reinterpret_cast<uint32_t *>(to) = (i & 1) ? __builtin_amdgcn_perm(bv[i >> 1], sv[i >> 1], 0x07060302u)
                                                    : __builtin_amdgcn_perm(bv[i >> 1], sv[i >> 1], 0x05040100u);
        to += 2 * sizeof(T);
        if (++g == G) {
          g = 0;
          to += 4;
        }
      }
    }
  }
  for (int i = tid; i < 4; i += 256) *reinterpret_cast<uint4 *>(lds + L.zeros + 16 * i) = make_uint4(0, 0, 0, 0);
  const unsigned char *const my_pairs = lds + L.pairs + (wn * NM * 16 + c) * L.pair_row;

  for (int t0 = 0; t0 < cnt; t0 += tt) {
    const int nt = cnt - t0 < tt ? cnt - t0 : tt;
    const bool on = c < nt;
    const unsigned char *const xl = on ? lds + c * L.x_stride : lds + L.zeros;
    const int x_step = on ? 1 : 0;
    f32x4_t tot[NM];
#pragma unroll
    for (int m = 0; m < NM; ++m) tot[m] = f32x4_t{0.f, 0.f, 0.f, 0.f};
    if (t0 > 0)
#pragma unroll
      for (int d = 0; d < kRing; ++d) issue(d, ring[d]);

    for (int s0 = 0; s0 < K; s0 += sk) {
      const int sl = K - s0 < sk ? K - s0 : sk;
      if (t0 > 0 || s0 > 0) __syncthreads();  // every wave is done with the previous slab
      // ---- token rows of the slab, eight values a thread, with the sums of their groups
      const int per_row = sl / 8;
      int row = tid / per_row, piece = tid - row * per_row;
      while (row < nt) {
        const int64_t r = r0 + t0 + row;
        int64_t src = r;
        if (inline_src && t0 + row < 12) src = a.work[(size_t)blockIdx.y * 16 + 4 + t0 + row];
        else if (a.src_rows) src = a.src_rows[r];
        const T *const xr = static_cast<const T *>(a.x) + src * K + s0 + piece * 8;
        unsigned char *const to = lds + row * L.x_stride + piece * 16;
        float v[8];
        {
          const uint4 w = *reinterpret_cast<const uint4 *>(xr);
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
          uint4 p = w;
          if constexpr (kStart) {
            p.x = (w.x & 0xffffu) | (w.y << 16);
            p.y = (w.x >> 16) | (w.y & 0xffff0000u);
            p.z = (w.z & 0xffffu) | (w.w << 16);
            p.w = (w.z >> 16) | (w.w & 0xffff0000u);
          } else if constexpr (PAIRED) {
            p.x = (w.x & 0xffffu) | (w.z << 16);
            p.y = (w.x >> 16) | (w.z & 0xffff0000u);
            p.z = (w.y & 0xffffu) | (w.w << 16);
            p.w = (w.y >> 16) | (w.w & 0xffff0000u);
          }
          *reinterpret_cast<uint4 *>(to) = p;
        }
        float sum = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
        sum += __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(sum)));
        sum += __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(sum)));
        if constexpr (GROUP >= 64) sum += __uint_as_float(dpp_u32<kDppHalfMirror>(__float_as_uint(sum)));
        if constexpr (GROUP == 128) sum += __uint_as_float(dpp_u32<kDppMirror>(__float_as_uint(sum)));
        if (piece % (GROUP / 8) == 0) sums[piece / (GROUP / 8) * kTokens + row] = kStart ? -centre_of(BITS) * sum : sum;
        piece += 256;
        while (piece >= per_row) {
          piece -= per_row;
          ++row;
        }
      }
      __syncthreads();

      // ---- the wave's chunks of the slab.  A slab is a whole number of kRing chunks a wave (or the last one): a chunk
      // keeps its slot of the ring.
      const int j1 = ((s0 + sl) / CH - wk + KW - 1) / KW;
      for (int jb = s0 / (CH * KW); jb < j1; jb += kRing) {
#pragma unroll
        for (int d = 0; d < kRing; ++d) {
          const int j = jb + d;
          if (j < j1) {
            const int ch = wk + KW * j, ch_slab = ch - s0 / CH;
            f32x4_t acc[NM];
            constexpr int NG = GROUP < CH ? CH / GROUP : 1;  // groups of a chunk (8-bit groups of 128: half a one)
            float4 xs[NG];
#pragma unroll
            for (int i = 0; i < NG; ++i) xs[i] = *reinterpret_cast<const float4 *>(sums + (ch * CH / GROUP + i - s0 / GROUP) * kTokens + 4 * kb);
            u32x4_t q[NM];
#pragma unroll
            for (int m = 0; m < NM; ++m) {
              q[m] = ring[d].q[m];
              if constexpr (BITS == 4) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                  const auto r = __builtin_amdgcn_permlane32_swap(q[m][i], q[m][i + 2], false, false);
                  q[m][i] = r[0];
                  q[m][i + 2] = r[1];
                }
#pragma unroll
                for (int i = 0; i < 4; i += 2) {
                  const auto r = __builtin_amdgcn_permlane16_swap(q[m][i], q[m][i + 1], false, false);
                  q[m][i] = r[0];
                  q[m][i + 1] = r[1];
                }
              } else if constexpr (GROUP == 32) {
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                  const auto r = __builtin_amdgcn_permlane32_swap(q[m][i], q[m][i + 2], false, false);
                  q[m][i] = r[0];
                  q[m][i + 2] = r[1];
                }
              }
            }
            issue(j + kRing, ring[d]);
#pragma unroll
            for (int s = 0; s < MUL; ++s) {
              // the eight K values of this lane in multiply s
              const int k = BITS == 4 ? 32 * s + 8 * kb : (GROUP == 32 ? 32 * s + 16 * (kb & 1) + 8 * (kb >> 1) : 16 * kb + 8 * s);
              const bool first = GROUP == 32 || (GROUP == 64 ? (BITS == 4 ? s % 2 == 0 : s == 0) : s == 0);
              const bool last = GROUP == 32 || (GROUP == 64 ? (BITS == 4 ? s % 2 == 1 : s == 1) : s == MUL - 1);
              const int g = ch * CH / GROUP + 32 * s / GROUP;
              const float4 x_sum = xs[32 * s / GROUP % NG];
              const u32x4_t av = *reinterpret_cast<const u32x4_t *>(xl + x_step * ((ch_slab * CH + k) * 2));
#pragma unroll
              for (int m = 0; m < NM; ++m) {
                u32x4_t bv;
                if constexpr (PAIRED && DT == 0) {
                  const uint32_t w = q[m][s], even = w & 0x0f0f0f0fu, odd = (w >> 4) & 0x0f0f0f0fu;
                  bv = u32x4_t{small_codes<0>(even), small_codes<0>(odd), small_codes<1>(even), small_codes<1>(odd)};
                } else if constexpr (PAIRED) {
                  const uint32_t w = q[m][s];
#pragma unroll
                  for (int i = 0; i < 4; ++i)
                    bv[i] = f16_centred<4>(__builtin_amdgcn_bitop3_b32(w >> (4 * i), 0x000f000fu, 0x64006400u, 0xEA));  // (a & b) | c
                } else if constexpr (DT == 1) {
#pragma unroll
                  for (int i = 0; i < 4; ++i)
                    bv[i] = f16_centred<8>(__builtin_amdgcn_perm(0x64646464u, q[m][2 * s + (i >> 1)], (i & 1) ? 0x07030702u : 0x07010700u));
                } else {
#pragma unroll
                  for (int i = 0; i < 4; i += 2) {
                    float v[4];
                    centred_codes(q[m][2 * s + (i >> 1)], v);
                    bv[i] = upper_halves(v[0], v[1]);
                    bv[i + 1] = upper_halves(v[2], v[3]);
                  }
                }
                acc[m] = mfma<DT>(av, bv, !first ? acc[m] : kStart ? f32x4_t{x_sum.x, x_sum.y, x_sum.z, x_sum.w} : f32x4_t{0.f, 0.f, 0.f, 0.f});
              }
              if (last) {  // (8-bit groups of 128: half a group, same scale)
                const bool with_bias = !(GROUP == 128 && BITS == 8) || (ch & 1) == 0;  // (once per group)
#pragma unroll
                for (int m = 0; m < NM; ++m) {
                  const uint32_t p = *reinterpret_cast<const uint32_t *>(my_pairs + m * 16 * L.pair_row + g * 4);
                  const float sc = as_f32(__builtin_bit_cast(T, (uint16_t)(p & 0xffffu)));
                  const float b = as_f32(__builtin_bit_cast(T, (uint16_t)(p >> 16)));
                  const float bi = !with_bias ? 0.f : kStart ? -__builtin_fmaf(1.0f / centre_of(BITS), b, sc) : __builtin_fmaf(centre_of(BITS), sc, b);
                  tot[m][0] = __builtin_fmaf(sc, acc[m][0], __builtin_fmaf(bi, x_sum.x, tot[m][0]));
                  tot[m][1] = __builtin_fmaf(sc, acc[m][1], __builtin_fmaf(bi, x_sum.y, tot[m][1]));
                  tot[m][2] = __builtin_fmaf(sc, acc[m][2], __builtin_fmaf(bi, x_sum.z, tot[m][2]));
                  tot[m][3] = __builtin_fmaf(sc, acc[m][3], __builtin_fmaf(bi, x_sum.w, tot[m][3]));
                }
              }
            }
          }
        }
      }
    }

    // ---- the K groups' sums, added in order, and the results: lane (c, kb) holds tokens 4 kb .. 4 kb + 3 of column c
    if constexpr (KW > 1) {
      float4 *const red = reinterpret_cast<float4 *>(lds + L.parts);
#pragma unroll
      for (int m = 0; m < NM; ++m) red[((wk * NW + wn) * NM + m) * 64 + lane] = make_float4(tot[m][0], tot[m][1], tot[m][2], tot[m][3]);
      __syncthreads();
      if (wk == 0)
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int w = 1; w < KW; ++w) {
            const float4 v = red[((w * NW + wn) * NM + m) * 64 + lane];
            tot[m][0] += v.x;
            tot[m][1] += v.y;
            tot[m][2] += v.z;
            tot[m][3] += v.w;
          }
    }
    if (wk == 0 && n0 + c < N) {
      const float lb = a.bias ? as_f32(static_cast<const T *>(a.bias)[n0 + c]) : 0.f;
      uint32_t again = 0;  // (bits: which of the four sums are not finite)
      auto put = [&](int r, float v, float up) __attribute__((always_inline)) {
        const int64_t rr = r0 + t0 + 4 * kb + r;
        const int64_t dst = a.dst_rows ? (int64_t)a.dst_rows[rr] : rr;
        if constexpr (GLU) v = v / (1.0f + __expf(-v)) * up;
        T o = rounded<T>(v);
        if (a.bias) o = rounded<T>(as_f32(o) + lb);
        static_cast<T *>(a.y)[dst * N + n0 + c] = o;
      };
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        if (4 * kb + r < nt) {
          put(r, tot[0][r], tot[NM - 1][r]);
          if (not_finite(tot[0][r]) || not_finite(tot[NM - 1][r])) again |= 1u << r;
        }
      }
      while (__builtin_expect(again != 0, 0)) {
        const int r = __builtin_ctz(again);
        again &= again - 1;
        const int64_t rr = r0 + t0 + 4 * kb + r, wrow = ebase + n0 + c;
        const T *const xr[1] = {static_cast<const T *>(a.x) + (a.src_rows ? (int64_t)a.src_rows[rr] : rr) * K};
        float v[NM][1];
#pragma unroll
        for (int m = 0; m < NM; ++m)
          plain_rows<BITS, 1, T>(xr, RowOrder::kPlain, (m ? a.w1 : a.w0) + wrow * (row_bytes / 4), static_cast<const T *>(m ? a.s1 : a.s0) + wrow * G,
                                 static_cast<const T *>(m ? a.b1 : a.b0) + wrow * G, K, GROUP, 1u, v[m]);
        put(r, v[0][0], v[NM - 1][0]);
      }
    }
  }
}

template <int DT, int BITS, int GROUP, bool GLU, int KW>
static hipError_t start_rows(const RowsArgs &a, int sk, int tt, hipStream_t st) {
  const RowsLds L(GROUP, GLU ? 2 : 1, KW, a.K, sk, tt);
  const auto kernel = &qmm_rows_kernel<DT, BITS, GROUP, GLU, KW>;
  if (L.bytes > 160 * 1024) return hipErrorInvalidConfiguration;
  if (L.bytes > 64 * 1024)
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, L.bytes);
        e != hipSuccess)
      return e;
  const dim3 grid((unsigned)((a.N + 16 * (4 / KW) - 1) / (16 * (4 / KW))), (unsigned)(a.work ? a.max_records ? a.max_records : a.max_active : 1));
  kernel<<<grid, 256, (size_t)L.bytes, st>>>(a, tt, sk);
  return hipGetLastError();
}

// How the launch is cut: K values of the token rows in LDS at a time (the whole row, or slabs that are a whole number of
// ring turns for every wave), token rows a pass, waves that share a row tile's K.
// The waves: with KW = 4 a block has 16 weight rows, so 1024 tiles are four blocks a CU, which is what the launch takes at once; from
// there on fewer and longer waves are better.  Measured, us of the kernel with 4 / 2 / 1 waves a tile at 2 and at 8 rows, K = 4096
// (1024 tiles and more: 2048): bf16 4-bit groups of 64, 128 tiles 6.8 / 8.8 / 12.6 and 11.4 / 13.1 / 17.5, 512 tiles 9.6 / 10.8 / 14.0 and 14.0 / 15.8 /
// 19.0, 1024 tiles 9.6 / 8.9 / 9.2 and 15.2 / 10.9 / 11.5, 2048 tiles 14.1 / 11.9 / 11.3 and 22.8 / 18.7 / 14.3, 4096 tiles 23.2 / 19.5 / 17.4 and
// 41.7 / 29.4 / 25.4; f16 8-bit, 512 tiles 12.8 / 15.6 / 20.8 and 18.5 / 21.6 / 26.5, 1024 tiles 10.8 / 11.0 / 12.6 and 17.9 / 13.8 / 15.4, 2048 tiles 18.6 /
// 15.3 / 16.1 and 27.4 / 24.9 / 18.9.
struct RowsCut {
  int kw, sk, tt;
};
static RowsCut cut_rows(const RowsArgs &a, int group, int bits, bool glu) {
  const int ch = bits == 4 ? 128 : 64, nm = glu ? 2 : 1;
  const int64_t longest = a.work ? a.max_rows : a.M;
  const int tt = (int)(longest < kTokens ? longest : kTokens);
  const int64_t tiles = (int64_t)((a.N + 15) / 16) * (a.work ? a.max_active : 1);
  int kw = tiles < 1024 ? 4 : (tiles < 2048 ? 2 : 1);
  for (;; kw /= 2) {
    const int unit = ch * kw * kRing;  // a slab: a multiple of this
    auto bytes = [&](int sk) { return RowsLds(group, nm, kw, a.K, sk, tt).bytes; };
    int sk = a.K;
    if (bytes(sk) > 64 * 1024) {  // (two blocks a CU at least)
      sk = a.K / unit * unit;
      while (sk > unit && bytes(sk) > 64 * 1024) sk -= unit;
      if (sk < unit) sk = a.K;
    }
    if (bytes(sk) <= 150 * 1024) return RowsCut{kw, sk, tt};
    if (kw == 1) return RowsCut{0, 0, 0};  // does not fit
  }
}

bool qmm_rows_applies(const RowsArgs &a, int group, int bits, int dt, bool glu) {
  return bits != 2 && dt != 2 && a.K % (bits == 4 ? 128 : 64) == 0 && a.K % group == 0 && (int64_t)a.N * a.K < (int64_t)1 << 31 &&
         cut_rows(a, group, bits, glu).kw > 0;
}

hipError_t launch_qmm_rows(const RowsArgs &a, int group, int bits, int dt, bool glu, hipStream_t st) {
  const RowsCut cut = cut_rows(a, group, bits, glu);
  if (cut.kw == 0) return hipErrorInvalidConfiguration;
  auto with_kw = [&](auto d, auto b, auto g, auto gl) {
    constexpr int DT = decltype(d)::value, BITS = decltype(b)::value, GROUP = decltype(g)::value;
    constexpr bool GLU = decltype(gl)::value;
    if (cut.kw == 4) return start_rows<DT, BITS, GROUP, GLU, 4>(a, cut.sk, cut.tt, st);
    if (cut.kw == 2) return start_rows<DT, BITS, GROUP, GLU, 2>(a, cut.sk, cut.tt, st);
    return start_rows<DT, BITS, GROUP, GLU, 1>(a, cut.sk, cut.tt, st);
  };
  auto with_glu = [&](auto d, auto b, auto g) {
    if constexpr (decltype(d)::value == 0 && decltype(g)::value != 64)  // (blocks with groups of 32 / 128)
      if (glu) return with_kw(d, b, g, std::true_type{});
    return with_kw(d, b, g, std::false_type{});
  };
  auto with_group = [&](auto d, auto b) {
    if (group == 32) return with_glu(d, b, std::integral_constant<int, 32>{});
    if (group == 64) return with_glu(d, b, std::integral_constant<int, 64>{});
    return with_glu(d, b, std::integral_constant<int, 128>{});
  };
  auto with_bits = [&](auto d) {
    return bits == 4 ? with_group(d, std::integral_constant<int, 4>{}) : with_group(d, std::integral_constant<int, 8>{});
  };
  if (glu && (dt != 0 || group == 64)) return hipErrorInvalidValue;
  if (dt == 0) return with_bits(std::integral_constant<int, 0>{});
  if (dt == 1) return with_bits(std::integral_constant<int, 1>{});
  return hipErrorInvalidValue;
}

}  // namespace mi_moe
