// Grouped quantized product of short pieces: a mixture-of-experts block with 4-bit codes in groups of 64, segments of a batch of up to sixty rows an expert in
// pieces of up to 64 token rows.
//
// Contract: mlx_gather_qmm with transpose = true (mlx-rs/src/ops/quantization.rs:160-230).  The same raw codes without a centre, prepared rows, group sums and
// bias product as qmm_pieces_kernel (qmm_tiles.hip).
#include "lds_copies.hpp"
#include "qmm_codes_dev.hpp"

namespace mi_moe {

constexpr int kWaves = 8, kHalf = kWaves / 2, kShortLds = 80 * 1024;  // two blocks share a CU

// LDS of a block: S stages of 128 K values (token rows of 256 bytes; 64 bytes of codes a weight row, 32 weight rows a wave) and a window's scales.
template <int MT>
struct ShortRing {
  static constexpr int S = MT <= 2 ? 3 : 2;
  static constexpr int X = 16 * MT * 256, W = 2048, STAGE = X + kWaves * W, WINDOW = 1024, BYTES = S * STAGE + kWaves * WINDOW;
  static constexpr int XALL = 4 * MT, XI = (XALL + kWaves - 1) / kWaves;  // copies of a stage's token rows, and of a wave (where they do not go round, waves make the same ones)
  static constexpr int COPIES = XI + 2;
};

// 16 MT token rows from sorted row `row0` (`rows` of them real) x 256 weight rows of expert e by eight waves of 32 weight rows each: GLU, 128 columns of h from n0:
// waves 0 to 3 the gate rows, 4 to 7 the up rows; else 256 columns from n0.
// A lane (weight row or token l % 16, quarter l / 16) multiplies 16 consecutive K values of a group in two steps of v_mfma_f32_16x16x32_bf16; the sums of a group
// are scaled once.
// What bounds it: at few rows an expert memory (128 experts, K = 2048, 1536 columns, 100 tokens: 226 MB in 47 us), then the latency of a stage, a chain of reads of LDS,
// unpacking and multiplies that four waves of a SIMD fill up for each other.  That is why it is four: tiles of 32 x 32 results (qmm_pieces_kernel, which
// took these pieces) want 250 registers and leave two, whose stages took 2700 cycles where their vector instructions are 1630.  And why the stages are written
// out one by one: 120 instructions of a stage of 16 rows, against 185 with the places and windows found at run time (49 us for 56 at 100 tokens).  Blocks of
// four waves and 128 weight rows, four a CU: token rows twice as often through L2, and no room for a third stage of 32 rows (203 tokens: 109 us a forward for 102).
// Blocks that take several tiles of a piece one after the other: slower, their own bookkeeping costs what the ends give.
template <bool GLU, int MT>
__device__ __forceinline__ void multiply_short(const CodesArgs &a, int e, int64_t row0, int rows, int n0, unsigned char *lds_raw) {
  typedef ShortRing<MT> R;
  constexpr int S = R::S;
  const int lane = threadIdx.x & 63, ln = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = a.N, K = a.K, G = K >> 6, row_bytes = K / 2, ext = padded_groups(G) * sum_slots(true);
  const int64_t ebase = (int64_t)e * N;
  const bool up = GLU && wave >= kHalf;
  const int col0 = n0 + 32 * (GLU ? wave % kHalf : wave);
  // weight row of place `at` (0 .. 31): in the order of h (CodesArgs::y_order) the place p of an 8-block takes the row whose result belongs there
  auto weight_row = [&](int at) __attribute__((always_inline)) { return col0 + (GLU ? (at & ~7) | value_at_place(a.y_order, at & 7) : at); };
  const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds_raw;
  const i32x4_t xr = words_of(a.x, (uint32_t)(a.x_rows * K * 2)), xsr = words_of(a.sums, (uint32_t)(a.x_rows * ext * 2));
  const i32x4_t wr = words_of((up ? a.w1 : a.w0) + ebase * (row_bytes / 4), (uint32_t)N * row_bytes);
  const i32x4_t sr = words_of(static_cast<const uint16_t *>(up ? a.s1 : a.s0) + ebase * G, (uint32_t)N * G * 2);
  const i32x4_t br = words_of(static_cast<const uint16_t *>(up ? a.b1 : a.b0) + ebase * G, (uint32_t)N * G * 2);

  // ---- what a lane copies.  Sixteen-byte pieces of a row are turned by the row's number, so that sixteen rows' pieces of one number lie in different banks.
  uint32_t x_off[R::XI], sums_off[R::XI], w_off[2], window_row;
#pragma unroll
  for (int c = 0; c < R::XI; ++c) {
    const int r = (wave * R::XI + c) % R::XALL * 4 + lane / 16, tr = r < rows ? r : rows - 1;  // rows past the end repeat the last one (never stored)
    const uint32_t row = a.src_rows ? a.src_rows[row0 + tr] : (uint32_t)(row0 + tr), piece = (uint32_t)((lane % 16) ^ (r & 15)) << 4;
    x_off[c] = row * (uint32_t)(K * 2) + piece;
    sums_off[c] = row * (uint32_t)(ext * 2) + piece;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) w_off[i] = (uint32_t)weight_row(16 * i + (lane >> 2)) * row_bytes + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  window_row = (uint32_t)weight_row(lane >> 1) * G * 2 + ((lane & 1) << 4);

  // ---- the stages: K in windows of 16 groups, each a stage of the bias product, which brings the window's scales, and then eight stages of codes, written out one by
  // one (nine stages, three places: a stage's place, and what it copies, is known when it is compiled).  Token rows are copied S - 1 stages ahead, a wave's weights
  // S: their place is the wave's own and free once its codes are read.  (Past the end the last values again.)
  const uint32_t x_at = ring_at + wave * R::XI % R::XALL * 1024, w_at = ring_at + R::X + wave * R::W;
  uint32_t turn = 0;  // two places: the window's first stage's (it takes turns)
  auto place = [&](int n) __attribute__((always_inline)) { return S == 3 ? (uint32_t)(n % 3 * R::STAGE) : n & 1 ? R::STAGE - turn : turn; };
  auto copy_weights = [&](int k, bool bias, uint32_t to) __attribute__((always_inline)) {
    const uint32_t at = bias ? (uint32_t)(k < K ? k : 0) >> 5 : (uint32_t)(k < K ? k : K - 128) >> 1;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      i32x4_t of;
#pragma unroll
      for (int w = 0; w < 4; ++w) of[w] = bias ? (i ? br : sr)[w] : wr[w];
      copy_to_lds(of, bias ? window_row : w_off[i], at, w_at + to + i * 1024);
    }
  };
  auto copy_rows = [&](int k, bool bias, uint32_t to) __attribute__((always_inline)) {
    const uint32_t at = bias ? (uint32_t)(k < K ? k : 0) >> 3 : (uint32_t)(k < K ? k : K - 128) << 1;
    i32x4_t of;
#pragma unroll
    for (int w = 0; w < 4; ++w) of[w] = bias ? xsr[w] : xr[w];
#pragma unroll
    for (int c = 0; c < R::XI; ++c) copy_to_lds(of, bias ? sums_off[c] : x_off[c], at, x_at + to + c * 1024);
  };
  // stage n of a window that begins at k: the bias product (0), or the codes from k + 128 (n - 1); n from 9 on: of the next window
  auto rows_of = [&](int k, int n) __attribute__((always_inline)) { copy_rows(n < 9 ? k + 128 * (n ? n - 1 : 0) : k + 1024 + 128 * (n > 9 ? n - 10 : 0), n % 9 == 0, place(n)); };
  auto weights_of = [&](int k, int n) __attribute__((always_inline)) { copy_weights(n < 9 ? k + 128 * (n ? n - 1 : 0) : k + 1024 + 128 * (n > 9 ? n - 10 : 0), n % 9 == 0, place(n)); };
  auto begin = [&]() __attribute__((always_inline)) {  // this stage's copies have arrived, in every wave, and its predecessor's rows are read
    wait_copies<2 + (S - 2) * R::COPIES>();
    block_barrier();
  };

  f32x4_t tot[2][MT];
  const f32x4_t zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int m = 0; m < MT; ++m) tot[j][m] = zero;
  weights_of(0, 0);
#pragma unroll
  for (int p = 0; p < S - 1; ++p) {
    rows_of(0, p);
    weights_of(0, p + 1);
  }
  unsigned char *const mine_at = lds_raw + R::X + wave * R::W, *const scales = lds_raw + S * R::STAGE + wave * R::WINDOW;  // [weight row][16]
  const unsigned char *f_at[4], *q_at[2];  // where a lane's pieces lie
#pragma unroll
  for (int i = 0; i < 4; ++i) f_at[i] = lds_raw + ln * 256 + (((8 * (i >> 1) + 2 * kq + (i & 1)) ^ ln) << 4);
#pragma unroll
  for (int g = 0; g < 2; ++g) q_at[g] = mine_at + ln * 64 + (((2 * g + (kq >> 1)) ^ ((ln >> 2) & 3)) << 4) + ((kq & 1) << 3);  // 16 K values: 8 bytes of a group's 32
  auto code_stage = [&](int k, int n) __attribute__((always_inline)) {
    const uint32_t from = place(n);
    begin();
    rows_of(k, n + S - 1);
    uint2 q[2][2];
    uint32_t s2[2];
    constexpr int AHEAD = MT < 3 ? MT : 2;  // sixteen rows fetched ahead
    u32x4_t F[AHEAD][2];
    auto fetch = [&](int i) __attribute__((always_inline)) {  // sixteen rows of a group
      if (i < 2 * MT)
#pragma unroll
        for (int h = 0; h < 2; ++h) F[i % AHEAD][h] = *reinterpret_cast<const u32x4_t *>(f_at[2 * (i / MT) + h] + from + i % MT * 4096);
    };
#pragma unroll
    for (int g = 0; g < 2; ++g)
#pragma unroll
      for (int j = 0; j < 2; ++j) q[g][j] = *reinterpret_cast<const uint2 *>(q_at[g] + from + j * 1024);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i);
#pragma unroll
    for (int j = 0; j < 2; ++j) s2[j] = *reinterpret_cast<const uint32_t *>(scales + (16 * j + ln) * 32 + 4 * (n - 1));
#pragma unroll
    for (int g = 0; g < 2; ++g) {
      u32x4_t op[2][2];
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        plain_codes(q[g][j].x, op[j][0]);
        plain_codes(q[g][j].y, op[j][1]);
      }
      if (g == 1) {  // (the stage's codes have been read: a copy out of L2 may overtake a read of LDS that waits its turn)
#pragma unroll
        for (int j = 0; j < 2; ++j) asm volatile("" : "+v"(op[j][0]), "+v"(op[j][1]));
        weights_of(k, n + S);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        f32x4_t acc[2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[j] = mfma<0>(F[(g * MT + m) % AHEAD][h], op[j][h], h ? acc[j] : zero);
        fetch(g * MT + m + AHEAD);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const float s = __uint_as_float(g ? s2[j] & 0xffff0000u : s2[j] << 16);
#pragma unroll
          for (int i = 0; i < 4; ++i) tot[j][m][i] = __builtin_fmaf(s, acc[j][i], tot[j][m][i]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m) asm volatile("" : "+v"(tot[j][m]));  // (added here, not where a stage ends the row: with every stage's sums kept until then they spill)
  };
#pragma unroll 1
  for (int k = 0; k < K; k += 1024) {
    {  // the bias product of the window: the group sums' three pieces against the bias, eight groups a multiply (real: groups from there on are not this row's)
      begin();
      rows_of(k, S - 1);
      const int real = G - (k >> 6);
      u32x4_t F[MT][2], o[2][2];
      const u32x4_t window = *reinterpret_cast<const u32x4_t *>(mine_at + place(0) + lane * 16);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
#pragma unroll
        for (int m = 0; m < MT; ++m) F[m][i] = *reinterpret_cast<const u32x4_t *>(lds_raw + place(0) + m * 4096 + ln * 256 + (((4 * i + kq) ^ ln) << 4));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int g = 8 * i + 2 * kq;
          const uint32_t b = g < real ? *reinterpret_cast<const uint32_t *>(mine_at + place(0) + 1024 + (16 * j + ln) * 32 + g * 2) : 0u;  // (an even number of groups)
          o[j][i] = u32x4_t{__builtin_amdgcn_perm(b, b, 0x01000100u), b & 0xffffu, __builtin_amdgcn_perm(b, b, 0x03020302u), b >> 16};
        }
      }
      *reinterpret_cast<u32x4_t *>(scales + lane * 16) = window;
      wait_reads();
      weights_of(k, S);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m) {
          f32x4_t sum = mfma<0>(F[m][0], o[j][0], zero);
          sum = mfma<0>(F[m][1], o[j][1], sum);
#pragma unroll
          for (int i = 0; i < 4; ++i) tot[j][m][i] += sum[i];
        }
    }
    const int stages = (K - k) >> 7;  // of codes, eight of them in this window
#pragma unroll
    for (int n = 1; n <= 8; ++n) {
      code_stage(k, n);
      if (n == stages) break;
    }
    if constexpr (S == 2) turn = R::STAGE - turn;
  }

  // ---- results: lane (column ln of half j, rows 16 m + 4 kq + 0 .. 3)
  const int my_row = lane >> 2;  // down: of 16, the row whose pieces this lane stores
  uint32_t dst[MT];
  if constexpr (!GLU) {
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      const int tr = 16 * m + my_row < rows ? 16 * m + my_row : rows - 1;
      dst[m] = a.dst_rows ? a.dst_rows[row0 + tr] : (uint32_t)(row0 + tr);
    }
  }
  wait_copies<0>();
  block_barrier();
  constexpr int ROWB = GLU ? 272 : 80;  // (16 bytes keep rows off each other's banks)
  constexpr int UP = 132;               // floats of an up row
  float *const ups = reinterpret_cast<float *>(lds_raw + 16 * MT * ROWB);
  unsigned char *const out = GLU ? lds_raw : lds_raw + wave * (16 * MT * ROWB);
  if constexpr (GLU) {
    if (up) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int i = 0; i < 4; ++i) ups[(16 * m + 4 * kq + i) * UP + 32 * (wave % kHalf) + 16 * j + ln] = tot[j][m][i];
    }
    __syncthreads();
  }
  if (!up) {
    uint32_t again = 0;  // results that are not finite (bit 4 (2 m + j) + i): computed again on the dequantised weights (see plain_rows)
    const int my_col = 32 * (GLU ? wave % kHalf : 0) + ln;
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * m + 4 * kq + i;
          float v = tot[j][m][i];
          bool bad = not_finite(v);
          if constexpr (GLU) {
            const float u = ups[r * UP + my_col + 16 * j];
            bad |= not_finite(u);
            v = gated(v, u);
          }
          again |= (bad && r < rows && (GLU || col0 < N) ? 1u : 0u) << (4 * (2 * m + j) + i);
          reinterpret_cast<uint16_t *>(out + r * ROWB)[my_col + 16 * j] = rounded<uint16_t>(v);
        }
    if (__builtin_expect(again != 0, 0)) {
#pragma unroll 1
      for (int at = 0; at < 2 * MT; ++at) {
        const int j = at & 1, m = at >> 1;
        const uint32_t open = again >> (4 * at) & 15u;
        if (!open) continue;
        const uint16_t *xs[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * m + 4 * kq + i, tr = r < rows ? r : rows - 1;
          xs[i] = static_cast<const uint16_t *>(a.x) + (int64_t)(a.src_rows ? a.src_rows[row0 + tr] : (uint32_t)(row0 + tr)) * K;
        }
        const int64_t wrow = ebase + weight_row(16 * j + ln);
        float v[GLU ? 2 : 1][4];
#pragma unroll
        for (int i = 0; i < (GLU ? 2 : 1); ++i)
          plain_rows<4, 4, uint16_t>(xs, RowOrder::kQuads, (i ? a.w1 : a.w0) + wrow * (row_bytes / 4), static_cast<const uint16_t *>(i ? a.s1 : a.s0) + wrow * G,
                                     static_cast<const uint16_t *>(i ? a.b1 : a.b0) + wrow * G, K, 64, open, v[i]);
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (open >> i & 1u) {
            const float o = GLU ? v[0][i] / (1.0f + __expf(-v[0][i])) * v[GLU ? 1 : 0][i] : v[0][i];
            reinterpret_cast<uint16_t *>(out + (16 * m + 4 * kq + i) * ROWB)[my_col + 16 * j] = rounded<uint16_t>(o);
          }
      }
    }
  }
  if constexpr (GLU) {
    __syncthreads();
    const int groups = N >> 6, padded = padded_groups(groups), piece = threadIdx.x & 15, g0 = (n0 >> 6) + (piece >> 3);  // sixteen lanes a row, eight a group
#pragma unroll
    for (int r0 = 0; r0 < 16 * MT; r0 += 4 * kWaves) {
      const int row = r0 + (int)(threadIdx.x >> 4);
      const u32x4_t w = *reinterpret_cast<const u32x4_t *>(out + row * ROWB + piece * 16);
      float sum = ((bf16lo_to_f32(w[0]) + bf16hi_to_f32(w[0])) + (bf16lo_to_f32(w[1]) + bf16hi_to_f32(w[1]))) +
                  ((bf16lo_to_f32(w[2]) + bf16hi_to_f32(w[2])) + (bf16lo_to_f32(w[3]) + bf16hi_to_f32(w[3])));
      sum += __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(sum)));
      sum += __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(sum)));
      sum += __uint_as_float(dpp_u32<kDppHalfMirror>(__float_as_uint(sum)));
      if (row < rows) {
        *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(a.y) + (row0 + row) * N + n0 + 8 * piece) = w;
        uint16_t *const sums = a.y_sums + (row0 + row) * padded * sum_slots(true);
        if ((piece & 7) == 0) put_sums(sums + g0 * sum_slots(true), sum_slots(true), sum);
        if (n0 + 128 >= N)  // the last block of a row writes the zeros behind its sums
          for (int g = groups + piece; g < padded; g += 16) put_sums(sums + g * sum_slots(true), sum_slots(true), 0.f);
      }
    }
  } else {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int m = 0; m < MT; ++m)
      if (16 * m + my_row < rows && col0 < N)
        *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(a.y) + (int64_t)dst[m] * N + col0 + 8 * (lane & 3)) =
            *reinterpret_cast<const u32x4_t *>(out + (16 * m + my_row) * ROWB + (lane & 3) * 16);
  }
}

// The pieces of a list (ShortTiles::piece = 64).  Ids are dealt round-robin over the 8 XCDs, whole pieces to each (the blocks of one share its gathered rows).
template <bool GLU>
__global__ __launch_bounds__(64 * kWaves, 4) void qmm_short_kernel(CodesArgs a, const uint32_t *__restrict__ list, int cap, int n_ntiles) {
  const uint32_t xcd = blockIdx.x & 7, j = blockIdx.x >> 3, id = j / (uint32_t)n_ntiles * 8u + xcd;
  const int n0 = (int)(j % (uint32_t)n_ntiles) * (GLU ? 128 : 256);
  const uint4 rec = reinterpret_cast<const uint4 *>(list)[1 + (id < (uint32_t)cap ? id : (uint32_t)cap - 1u)];  // (beside the count, not behind it)
  if (id >= list[0]) return;
  const int e = __builtin_amdgcn_readfirstlane((int)rec.x), rows = __builtin_amdgcn_readfirstlane((int)rec.z);
  const int64_t row0 = (int64_t)__builtin_amdgcn_readfirstlane((int)rec.y);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  static_assert(ShortRing<1>::BYTES <= kShortLds && ShortRing<2>::BYTES <= kShortLds && ShortRing<4>::BYTES <= kShortLds && 64 * (272 + 132 * 4) <= kShortLds, "two blocks share a CU");
  if (rows > 48) multiply_short<GLU, 4>(a, e, row0, rows, n0, lds_raw);
  else if (rows > 32) multiply_short<GLU, 3>(a, e, row0, rows, n0, lds_raw);
  else if (rows > 16) multiply_short<GLU, 2>(a, e, row0, rows, n0, lds_raw);
  else multiply_short<GLU, 1>(a, e, row0, rows, n0, lds_raw);
}

template <bool GLU>
static hipError_t start_short(const CodesArgs &a, const uint32_t *list, int cap, hipStream_t st) {
  constexpr int NI = GLU ? 128 : 256;
  const int n_ntiles = (a.N + NI - 1) / NI;
  const int64_t grid = ((int64_t)cap + 7) / 8 * 8 * n_ntiles;
  if (grid <= 0 || grid > INT32_MAX || a.N % 128 || a.K % 128) return hipErrorInvalidValue;
  static std::atomic<uint64_t> allowed{0};
  if (hipError_t e = allow_lds(reinterpret_cast<const void *>(&qmm_short_kernel<GLU>), kShortLds, allowed); e != hipSuccess) return e;
  launch_or_time(&qmm_short_kernel<GLU>, dim3((unsigned)grid), dim3(64 * kWaves), kShortLds, st, a, list, cap, n_ntiles);
  return hipGetLastError();
}
hipError_t launch_qmm_short(const CodesArgs &a, const uint32_t *list, int cap, bool glu, hipStream_t st) {
  return glu ? start_short<true>(a, list, cap, st) : start_short<false>(a, list, cap, st);
}

}  // namespace mi_moe
