// Dense quantized product of float32 rows on the float32 matrix instructions: weights packed along K, 4- and 8-bit codes.
//
// Contract: mlx_quantized_matmul with transpose = true (mlx-rs/src/ops/quantization.rs:91-122).
//
// Arithmetic: weights dequantised as in the plain kernels, w = fma(s, q, b), and multiplied in float32 as they are.  What such a product loses is the order of its sums: one
// accumulator over all of K would lose several times what the plain kernel's 64 partial sums a result do.  So the matrix instructions add up eight values, four of those a run of
// 32, the runs of a wave its total, and the totals of the eight waves of a block meet in a tree.  Relative error against 64 bits (2-norm), here / plain kernel (rows x N x K): 64 x 1024 x 1024
// 0.995e-7 / 0.995e-7, 300 x 1536 x 2048 1.01e-7 / 1.21e-7, 1000 x 3072 x 3072 1.08e-7 / 1.38e-7, 777 x 4096 x 4096 1.15e-7 / 1.61e-7 (one chain of 32 values a run: 1.18e-7, 1.24e-7, 1.29e-7, 1.39e-7).
#include <atomic>
#include <type_traits>

#include "dense_rule.hpp"
#include "qmm_codes_dev.hpp"

namespace mi_moe {

struct F32Args {
  const float *x;
  const uint32_t *w;
  const float *s, *b;
  float *y;
  int N, K, group_log2;
  int64_t M;
};

// A block computes 32 MS rows x 32 NT columns with eight waves, each of which takes every eighth run of 32 K values.  v_mfma_f32_32x32x2_f32 multiplies one K value a half of the lanes, so a
// lane takes sixteen consecutive K values of its row (half l / 32 of the run): four 16-byte loads of x and 8 or 16 bytes of codes, straight into registers, a run ahead.
// What bounds it: the matrix unit, 64 cycles for 2048 products (157 TFLOP/s nominal, twice the vector unit's rate, which is what the plain
// kernel is bound by), and the last round of tiles.  us of the call, 4-bit, groups of 64, 1000 x 3072 x 3072: plain kernel 561, here 197 (96 TFLOP/s); 8-bit 1000 x 4096 x 4096 1082 / 335.
template <int BITS, int MS, int NT>
__global__ __launch_bounds__(512, 2) void qmm_f32_kernel(F32Args a, int n_mtiles, int n_ntiles) {
  constexpr int kWaves = 8, CW = BITS / 2;  // words of sixteen codes
  // Ids are dealt round-robin over the 8 XCDs: an XCD takes every eighth column tile and all row tiles of it, so its L2 holds those weights.
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3, nt = j / n_mtiles * 8 + xcd;
  if (nt >= n_ntiles) return;
  const int64_t row0 = (int64_t)(j % n_mtiles) * (32 * MS);
  const int n0 = nt * (32 * NT);
  const int lane = threadIdx.x & 63, ln = lane & 31, kb = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = a.N, K = a.K, G = K >> a.group_log2;
  const float *xr[MS];
#pragma unroll
  for (int m = 0; m < MS; ++m) {  // rows and columns outside: the last ones again, not stored
    const int64_t r = row0 + 32 * m + ln;
    xr[m] = a.x + (r < a.M ? r : a.M - 1) * K + 16 * kb;
  }
  const uint32_t *wr[NT];
  const float *sr[NT], *br[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int64_t n = n0 + 32 * t + ln < N ? n0 + 32 * t + ln : N - 1;
    wr[t] = a.w + n * (K * BITS / 32) + kb * CW;
    sr[t] = a.s + n * G;
    br[t] = a.b + n * G;
  }
  struct Run {
    float4 x[MS][4];
    uint32_t q[NT][CW];
    float s[NT], b[NT];
  };
  auto load = [&](int k, Run &R) __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int p = 0; p < 4; ++p) R.x[m][p] = reinterpret_cast<const float4 *>(xr[m] + k)[p];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
      for (int i = 0; i < CW; ++i) R.q[t][i] = wr[t][k * BITS / 32 + i];
      const int g = (k + 16 * kb) >> a.group_log2;
      R.s[t] = sr[t][g];
      R.b[t] = br[t][g];
    }
  };
  const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
  f32x16_t tot[MS][NT];
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) tot[m][t] = zero;
  Run next;
  if (wave * 32 < K) load(wave * 32, next);
#pragma unroll 1
  for (int k = wave * 32; k < K; k += kWaves * 32) {
    const Run R = next;
    load(k + kWaves * 32 < K ? k + kWaves * 32 : k, next);
    f32x16_t sum[MS][NT];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float w[NT][4];
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int c = 0; c < 4; ++c)
          w[t][c] = __builtin_fmaf(R.s[t], (float)((R.q[t][(4 * i + c) * BITS / 32] >> ((4 * i + c) * BITS % 32)) & ((1u << BITS) - 1u)), R.b[t]);
#pragma unroll
      for (int m = 0; m < MS; ++m) {
        const float4 p = R.x[m][i];
        const float xv[4] = {p.x, p.y, p.z, p.w};
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          f32x16_t part = zero;
#pragma unroll
          for (int c = 0; c < 4; ++c) part = __builtin_amdgcn_mfma_f32_32x32x2f32(xv[c], w[t][c], part, 0, 0, 0);
          sum[m][t] = i ? sum[m][t] + part : part;
        }
      }
    }
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t) tot[m][t] += sum[m][t];
  }
  // ---- the waves' totals, added in a tree; a thread stores consecutive columns' lanes
  constexpr int COLS = 32 * NT, CELLS = 32 * MS * COLS;
  extern __shared__ __align__(16) unsigned char lds_raw[];
  float *const parts = reinterpret_cast<float *>(lds_raw);  // [wave][row][column]
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) parts[wave * CELLS + (32 * m + 8 * (v >> 2) + 4 * kb + (v & 3)) * COLS + 32 * t + ln] = tot[m][t][v];
  __syncthreads();
#pragma unroll
  for (int i = 0; i < CELLS / 512; ++i) {
    const int cell = i * 512 + (int)threadIdx.x;
    float p[kWaves];
#pragma unroll
    for (int u = 0; u < kWaves; ++u) p[u] = parts[u * CELLS + cell];
    const int64_t row = row0 + cell / COLS;
    const int col = n0 + cell % COLS;
    if (row < a.M && col < N) a.y[row * N + col] = ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
  }
}

template <int BITS, int MS, int NT>
static hipError_t start_f32(const F32Args &a, hipStream_t st) {
  constexpr int lds = 8 * 32 * MS * 32 * NT * 4;
  const int n_ntiles = (a.N + 32 * NT - 1) / (32 * NT);
  const int64_t mtiles = (a.M + 32 * MS - 1) / (32 * MS), grid = (int64_t)((n_ntiles + 7) / 8) * 8 * mtiles;
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  const auto kernel = &qmm_f32_kernel<BITS, MS, NT>;
  static std::atomic<uint64_t> allowed{0};
  if (hipError_t e = allow_lds(reinterpret_cast<const void *>(kernel), lds, allowed); e != hipSuccess) return e;
  kernel<<<(unsigned)grid, 512, lds, st>>>(a, (int)mtiles, n_ntiles);
  return hipGetLastError();
}

hipError_t launch_qmm_f32(const float *x, const uint32_t *w, const float *s, const float *b, int64_t rows, int N, int K, int group, int bits, float *y, hipStream_t st) {
  const F32Args a{x, w, s, b, y, N, K, group == 32 ? 5 : group == 64 ? 6 : 7, rows};
  auto with_bits = [&](auto bb) {
    constexpr int BITS = decltype(bb)::value;
    if (tiles_of_an_xcd(rows, N, 32, 32) <= 32) return start_f32<BITS, 1, 1>(a, st);
    if (tiles_of_an_xcd(rows, N, 64, 32) <= 32) return start_f32<BITS, 2, 1>(a, st);
    return start_f32<BITS, 2, 2>(a, st);
  };
  return bits == 4 ? with_bits(std::integral_constant<int, 4>{}) : with_bits(std::integral_constant<int, 8>{});
}

}  // namespace mi_moe
