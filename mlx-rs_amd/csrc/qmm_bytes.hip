// Grouped quantized product of long pieces with 8-bit codes: the segments of a mixture-of-experts block in pieces of up to 128 token rows, groups of 64.
//
// Contract: mlx_gather_qmm with transpose = true (mlx-rs/src/ops/quantization.rs:160-230).  Weights are dequantised in fp32 and rounded to bf16, as in the tiles of 256 weight
// rows (qmm_large.hip), which take the batches that do not come here; sums are fp32.
#include <type_traits>

#include "lds_copies.hpp"
#include "qmm_codes_dev.hpp"

namespace mi_moe {

constexpr int kBytesLds = 80 * 1024;
// What a block of 32 MS token rows and four waves holds in LDS: two places of 64 K values of token rows, the codes of 128 K values (32 NT weight rows a wave), and two
// windows of a wave's scales and biases (8 groups, 16 bytes a weight row each).
template <int MS, int NT>
struct Bytes {
  static constexpr int XROW = 128, X = 32 * MS * XROW, W = NT * 4096, WINDOW = 2048, LDS = 2 * X + 4 * W + 8 * WINDOW;
  static_assert(LDS <= kBytesLds, "two blocks share a CU");
};

// 32 MS token rows from sorted row `row0` (`rows` of them real) x 128 NT weight rows of expert e by four waves: GLU, 128 columns of h from n0, a wave 32 gate and the
// matching 32 up rows; else 128 NT columns from n0, 32 NT a wave.  A wave multiplies all the tile's token rows with its own weights, which it dequantises straight into
// the matrix instruction's operands: its codes go to no other wave, and a stage (64 K values) has one barrier, for the token rows.
//   operands  eight a stage (two sub-tiles of 32 weight rows, four multiplies of 16 K values).  K runs outside, token rows inside, so that two operands are free again
//             after every quarter of a stage; the next stage's are made there, four vector instructions behind each multiply (128 rows).
//   copies    straight into LDS: token rows a stage ahead; codes in whole lines of 128 bytes, two stages at once, one and a half ahead: they are read into
//             registers together, which frees their place.
// What bounds it: memory at few rows (8 experts, 4096 x 14336, 100 tokens: 1.4 GB in 360 us), then the clock and the copies.  36 pieces of 128 rows, gate/up (962 GFLOP): 1.8 M
// cycles an XCD at 1.7 GHz, matrix units busy 0.53 of them; without the dequantisation (8 vector instructions a word of codes, 4.5 a multiply) the same cycles at 2.0 GHz, with all
// copies out of L2 9 % fewer, with half the codes 14 %.  Codes copied in pieces of 64 bytes, a stage at a time: 1029 us for 975, down 606 for 556.
//   KW = 2    two groups of four waves share K, each with an LDS place of its own; the second one's sums go to the first through LDS at the end.
template <bool GLU, int MS, int KW, int NT>
__device__ __forceinline__ void multiply_bytes(const CodesArgs &a, int e, int64_t row0, int rows, int n0, unsigned char *block_lds) {
  typedef Bytes<MS, NT> R;
  static_assert(!GLU || NT == 2, "a gate and an up row's sub-tile");
  constexpr int NM = GLU ? 2 : 1;
  const int lane = threadIdx.x & 63, ln = lane & 31, kb = lane >> 5;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), wave = wave_all % 4, kg = wave_all / 4;
  const int N = a.N, K = a.K, G = K >> 6, k_first = kg * (K / KW), k_end = k_first + K / KW;
  unsigned char *const lds_raw = block_lds + kg * kBytesLds;
  const int64_t ebase = (int64_t)e * N;
  const uint32_t ring_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds_raw;
  constexpr int kCodes = 2 * R::X, kScales = kCodes + 4 * R::W;  // where the codes and the windows lie
  const i32x4_t xr = words_of(a.x, (uint32_t)(a.x_rows * K * 2));
  i32x4_t wr[NM], sr[NM], br[NM];
#pragma unroll
  for (int t = 0; t < NM; ++t) {
    wr[t] = words_of((t ? a.w1 : a.w0) + ebase * (K / 4), (uint32_t)N * K);
    sr[t] = words_of(static_cast<const uint16_t *>(t ? a.s1 : a.s0) + ebase * G, (uint32_t)N * G * 2);
    br[t] = words_of(static_cast<const uint16_t *>(t ? a.b1 : a.b0) + ebase * G, (uint32_t)N * G * 2);
  }
  const int col0 = n0 + (GLU ? 32 : 32 * NT) * wave, own0 = col0 < N ? col0 : N - 32 * NT;  // (columns past the end are others again, and never stored)
  // ---- what a lane copies.  Sixteen-byte pieces of a row are turned by a number of the row's, so that sixteen rows' pieces of one number lie in different banks.
  auto turned = [](int row) __attribute__((always_inline)) { return (row >> 1) & 7; };
  uint32_t x_off[MS], w_off[2];
#pragma unroll
  for (int i = 0; i < MS; ++i) {
    const int r = (wave * MS + i) * 8 + lane / 8, tr = r < rows ? r : rows - 1;  // rows past the end repeat the last one (never stored)
    x_off[i] = (a.src_rows ? a.src_rows[row0 + tr] : (uint32_t)(row0 + tr)) * (uint32_t)(K * 2) + ((uint32_t)((lane % 8) ^ turned(r)) << 4);
  }
#pragma unroll
  for (int i = 0; i < 2; ++i)  // rows 8 i + lane / 8; 16 rows on the pieces are turned alike
    w_off[i] = (uint32_t)(own0 + 8 * i + lane / 8) * (uint32_t)K + ((uint32_t)((lane % 8) ^ turned(8 * i + lane / 8)) << 4);
  const uint32_t window_off = (uint32_t)(own0 + (GLU || NT == 1 ? ln : lane)) * (uint32_t)(G * 2);
  auto copy_rows = [&](int k, uint32_t place) __attribute__((always_inline)) {  // (past the end the last values again)
#pragma unroll
    for (int c = 0; c < MS; ++c) copy_to_lds(xr, x_off[c], (k < K ? k : K - 64) * 2, ring_at + place * R::X + (wave * MS + c) * 1024);
  };
  auto copy_codes = [&](int k) __attribute__((always_inline)) {  // of 128 K values
#pragma unroll
    for (int i = 0; i < 4 * NT; ++i)
      copy_to_lds(wr[GLU ? i / 4 : 0], w_off[i & 1], (k < K ? k : K - 128) + ((i & 2) + (GLU ? 0 : i & 4)) * 8 * K, ring_at + kCodes + wave * R::W + i * 1024);
  };
  auto copy_window = [&](int k) __attribute__((always_inline)) {  // the 8 groups from K value k on: 16 bytes a weight row of scales, 1024 bytes behind them of biases
    const uint32_t to = ring_at + kScales + (wave * 2 + (k >> 9 & 1)) * R::WINDOW;
    const int from = (k < K ? k : 0) >> 6 << 1;
    if constexpr (GLU) {
#pragma unroll
      for (int t = 0; t < 2; ++t) {  // 32 rows of each matrix
        copy_half_to_lds(sr[t], window_off, from, to + t * 512);
        copy_half_to_lds(br[t], window_off, from, to + 1024 + t * 512);
      }
    } else if constexpr (NT == 1) {
      copy_half_to_lds(sr[0], window_off, from, to);
      copy_half_to_lds(br[0], window_off, from, to + 1024);
    } else {
      copy_to_lds(sr[0], window_off, from, to);
      copy_to_lds(br[0], window_off, from, to + 1024);
    }
  };

  f32x16_t tot[MS][NT];
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int v = 0; v < 16; ++v) tot[m][t][v] = 0.f;
  u32x4_t op[NT][4], q[2][2][NT];  // operands; sixteen codes of a weight row: of each of two stages, K values 0 .. 31 of it and those behind
  u32x2_t rest[NT];               // the codes of a pair's last multiply
  float scale[NT], offset[NT];
  uint32_t s_now[NT], b_now[NT];
  // Piece 2 kb + (h & 1) + 4 (h / 2) of a token row is multiply h's, piece 2 i + kb of a row of codes quarter i of a pair: made out of the first ones where they are wanted.
  uint32_t xa = ln * R::XROW + ((2 * kb ^ turned(ln)) << 4), wa = kCodes + wave * R::W + ln * 128 + ((kb ^ turned(ln)) << 4);
  // Two weights of a word of codes, behind the exponent of 1024 as f16 (exact) and back out of it in the fma that scales them.
  auto weights = [&](uint32_t codes, int pair, int t) __attribute__((always_inline)) {
    const half2_t v = __builtin_bit_cast(half2_t, __builtin_amdgcn_perm(0x64646464u, codes, pair ? 0x07030702u : 0x07010700u));
    return cvt_pk_bf16(__builtin_fmaf(scale[t], (float)v.x, offset[t]), __builtin_fmaf(scale[t], (float)v.y, offset[t]));
  };
  auto fetch_codes = [&]() __attribute__((always_inline)) {
    asm volatile("" : "+v"(wa));
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) q[i >> 1][i & 1][t] = *reinterpret_cast<const u32x4_t *>(lds_raw + (wa ^ i << 5) + t * 4096);
  };
  auto fetch_scales = [&](int k) __attribute__((always_inline)) {
    const unsigned char *const at = lds_raw + kScales + (wave * 2 + (k >> 9 & 1)) * R::WINDOW + (k >> 6 & 7) * 2 + ln * 16;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      s_now[t] = *reinterpret_cast<const uint16_t *>(at + t * 512);
      b_now[t] = *reinterpret_cast<const uint16_t *>(at + t * 512 + 1024);
    }
  };
  auto take_scales = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      scale[t] = __uint_as_float(s_now[t] << 16);
      offset[t] = __builtin_fmaf(-1024.0f, scale[t], __uint_as_float(b_now[t] << 16));
    }
  };
  // word i (0 .. 4 NT - 1) of the operands that quarter `made` of a pair's stage consumes
  auto make = [&](int stage, int made, int i) __attribute__((always_inline)) {
    const int t = i >> 2, w = i & 3;
    const uint32_t codes = stage == 1 && made == 3 ? rest[t][w >> 1] : q[stage][made >> 1][t][2 * (made & 1) + (w >> 1)];
    op[t][made][w] = weights(codes, w & 1, t);
  };
  // A stage from k on, from place STAGE of the token rows.  What its last quarter multiplies is made in its first one, what the next stage's other quarters do behind.
  auto multiply = [&](int k, auto of_pair) __attribute__((always_inline)) {
    constexpr int STAGE = decltype(of_pair)::value, STEPS = 4 * MS, AHEAD = MS == 1 ? 4 : 6;  // rows of a quarter, fetched ahead
    const unsigned char *const at = lds_raw + STAGE * R::X;
    u32x4_t F[AHEAD];
    asm volatile("" : "+v"(xa));
    auto fetch = [&](int j) __attribute__((always_inline)) {
      const int h = j / MS;
      F[j % AHEAD] = *reinterpret_cast<const u32x4_t *>(at + (xa ^ ((h & 1) | (h & 2) << 1) << 4) + j % MS * (32 * R::XROW));
    };
#pragma unroll
    for (int j = 0; j < AHEAD; ++j) fetch(j);
    fetch_scales(k + 64);
    if constexpr (STAGE == 1) fetch_codes();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < STEPS; ++j) {
      const int h = j / MS, m = j % MS;
      if (m == 0 && h == 1) take_scales();
      if (STAGE == 1 && m == 0 && h == 2) {
        wait_reads();  // (the codes' place is free)
        if ((k + 192 & 511) == 0) copy_window(k + 192);
        copy_codes(k + 192);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        tot[m][t] = mfma<0>(F[j % AHEAD], op[t][h], tot[m][t]);
        if (t == NT - 1 && j + AHEAD < STEPS) fetch(j + AHEAD);
        const int u = NT * m + t;
#pragma unroll
        for (int i = u * 4 / MS; i < (u + 1) * 4 / MS; ++i) make(h == 0 ? STAGE : STAGE ^ 1, (h + 3) & 3, i);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  };

  const std::integral_constant<int, 0> first{};
  const std::integral_constant<int, 1> second{};
  copy_window(k_first & ~511);
  copy_codes(k_first);
  copy_rows(k_first, 0);
  wait_copies<0>();
  fetch_scales(k_first);
  fetch_codes();
  take_scales();
#pragma unroll
  for (int i = 0; i < 12 * NT; ++i) make(0, i / (4 * NT), i % (4 * NT));
  wait_reads();
  if ((k_first + 128 & 511) == 0) copy_window(k_first + 128);
  copy_codes(k_first + 128);
#pragma unroll 1
  for (int k = k_first; k < k_end; k += 128) {
    wait_copies<4 * NT>();  // this stage's token rows have arrived, in every wave, and the place copied to next has been read; the next pair's codes may still be coming
    block_barrier();
    copy_rows(k + 64, 1);
    multiply(k, first);
#pragma unroll
    for (int t = 0; t < NT; ++t) rest[t] = u32x2_t{q[1][1][t][2], q[1][1][t][3]};
    wait_copies<0>();
    block_barrier();
    copy_rows(k + 128, 0);
    multiply(k + 64, second);
  }

  wait_copies<0>();
  block_barrier();
  if constexpr (KW == 2) {
    float4 *const parts = reinterpret_cast<float4 *>(block_lds) + wave * (MS * NT * 4 * 64) + lane;
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (kg == 1) parts[((m * NT + t) * 4 + r) * 64] = make_float4(tot[m][t][4 * r], tot[m][t][4 * r + 1], tot[m][t][4 * r + 2], tot[m][t][4 * r + 3]);
    __syncthreads();
    if (kg == 1) return;
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float4 v = parts[((m * NT + t) * 4 + r) * 64];
          tot[m][t][4 * r] += v.x;
          tot[m][t][4 * r + 1] += v.y;
          tot[m][t][4 * r + 2] += v.z;
          tot[m][t][4 * r + 3] += v.w;
        }
    __syncthreads();  // (of the waves that are left: the results' place is free)
  }

  // ---- results: lane (column ln of sub-tile t, rows 32 m + 8 (r / 4) + 4 kb + r % 4).  Two rows of a column become one register, neighbouring lanes swap halves, and
  // the rows are turned round in LDS: GLU: by the whole block, 256 bytes a row; else by each wave, 128 bytes a row.
  uint32_t dst[2] = {};
  if constexpr (!GLU) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const int64_t r = row0 + (64 * h + lane < rows ? 64 * h + lane : rows - 1);
      dst[h] = a.dst_rows ? a.dst_rows[r] : (uint32_t)r;
    }
  }
  constexpr int ROWB = GLU ? 272 : 64 * NT + 16, PIECES = 4 * NT;  // (16 bytes keep rows off each other's banks)
  static_assert((GLU ? 32 * MS * 272 : 4 * 32 * ROWB) <= R::LDS, "the results' place");
  unsigned char *const mine = GLU ? lds_raw + wave * 64 : lds_raw + wave * (32 * ROWB);
  float odd = 0.f;  // no number once a result was not finite
  auto turn = [&](int m, int at, auto plain) __attribute__((always_inline)) {
    auto value = [&](int t, int r) __attribute__((always_inline)) {
      if constexpr (!GLU) return tot[m][t][r];
      const float g = tot[m][0][r], u = tot[m][1][r];
      return decltype(plain)::value ? g / (1.0f + __expf(-g)) * u : gated(g, u);
    };
#pragma unroll
    for (int t = 0; t < (GLU ? 1 : NT); ++t)
#pragma unroll
      for (int r = 0; r < 16; r += 2) {
        const float v0 = value(t, r), v1 = value(t, r + 1);
        if (GLU) odd = __builtin_fmaf(v1, 0.f, __builtin_fmaf(v0, 0.f, odd));
        const uint32_t own = cvt_pk_bf16(v0, v1), theirs = dpp_u32<kDppXor1>(own);
        // even lane: row r of columns c, c + 1; odd lane: row r + 1
        const uint32_t both = __builtin_amdgcn_perm(theirs, own, (ln & 1) ? 0x03020706u : 0x05040100u);
        *reinterpret_cast<uint32_t *>(mine + (at + 8 * (r >> 2) + 4 * kb + (r & 3) + (ln & 1)) * ROWB + (32 * t + (ln & ~1)) * 2) = both;
      }
  };
  if constexpr (GLU) {
#pragma unroll
    for (int m = 0; m < MS; ++m) turn(m, 32 * m, std::false_type{});
    if (__builtin_expect(__any(odd != odd), 0)) {  // (gated gives no number for an infinite gate; the division does)
#pragma unroll
      for (int m = 0; m < MS; ++m) turn(m, 32 * m, std::true_type{});
    }
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2 * MS; ++i) {
      const int row = 16 * i + (int)(threadIdx.x >> 4), piece = threadIdx.x & 15;
      const u32x4_t w = *reinterpret_cast<const u32x4_t *>(lds_raw + row * ROWB + piece * 16);
      if (row < rows) *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(a.y) + (row0 + row) * N + n0 + 8 * piece) = w;
    }
  } else {
#pragma unroll
    for (int m = 0; m < MS; ++m) {
      turn(m, 0, std::false_type{});
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
      for (int i = 0; i < PIECES / 2; ++i) {
        const int row = 64 / PIECES * i + lane / PIECES, tr = 32 * m + row;
        const u32x4_t w = *reinterpret_cast<const u32x4_t *>(mine + row * ROWB + lane % PIECES * 16);
        const uint32_t to = (uint32_t)__shfl((int)dst[m / 2], tr & 63, 64);
        if (tr < rows && col0 < N) *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(a.y) + (int64_t)to * N + col0 + 8 * (lane % PIECES)) = w;
      }
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    }
  }
}

// The pieces of a list (ShortTiles::piece up to 128).  Ids are dealt round-robin over the 8 XCDs; an XCD takes the same columns of kRun pieces that follow each other
// in the list, mostly of one expert, so that its L2 holds their codes once: 8 experts, 4096 x 14336 at 512 / 2048 tokens 704 / 1721 us a forward, pieces each on their
// own 739 / 1745, two 720 / 1723, eight 737 / 1732.
constexpr uint32_t kRun = 4;
template <bool GLU, int KW, int NT>
__global__ __launch_bounds__(256 * KW, 2) void qmm_bytes_kernel(CodesArgs a, const uint32_t *__restrict__ list, int n_ntiles) {
  const uint32_t xcd = blockIdx.x & 7, j = blockIdx.x >> 3, unit = j / kRun * 8u + xcd;
  const uint32_t id = unit / (uint32_t)n_ntiles * kRun + j % kRun;
  if (id >= list[0]) return;
  const int n0 = (int)(unit % (uint32_t)n_ntiles) * (GLU ? 128 : 128 * NT);
  const uint4 rec = reinterpret_cast<const uint4 *>(list)[1 + id];
  const int e = __builtin_amdgcn_readfirstlane((int)rec.x), rows = __builtin_amdgcn_readfirstlane((int)rec.z);
  const int64_t row0 = (int64_t)__builtin_amdgcn_readfirstlane((int)rec.y);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  if (rows > 96) multiply_bytes<GLU, 4, KW, NT>(a, e, row0, rows, n0, lds_raw);
  else if (rows > 64) multiply_bytes<GLU, 3, KW, NT>(a, e, row0, rows, n0, lds_raw);
  else if (rows > 32) multiply_bytes<GLU, 2, KW, NT>(a, e, row0, rows, n0, lds_raw);
  else multiply_bytes<GLU, 1, KW, NT>(a, e, row0, rows, n0, lds_raw);
}

template <bool GLU, int KW, int NT>
static hipError_t start_bytes(const CodesArgs &a, const uint32_t *list, int cap, hipStream_t st) {
  constexpr int NI = GLU ? 128 : 128 * NT;
  const int n_ntiles = (a.N + NI - 1) / NI;
  const int64_t units = ((int64_t)cap + kRun - 1) / kRun * n_ntiles, grid = (units + 7) / 8 * 8 * kRun;
  if (grid <= 0 || grid > INT32_MAX || a.N % 128 || a.K % (128 * KW)) return hipErrorInvalidValue;
  const auto kernel = &qmm_bytes_kernel<GLU, KW, NT>;
  static std::atomic<uint64_t> allowed{0};
  if (hipError_t e = allow_lds(reinterpret_cast<const void *>(kernel), KW * kBytesLds, allowed); e != hipSuccess) return e;
  launch_or_time(kernel, dim3((unsigned)grid), dim3(256 * KW), KW * kBytesLds, st, a, list, n_ntiles);
  return hipGetLastError();
}
// Where no CU gets two blocks (a down product of few experts: 8 pieces are 128 blocks of 256 of 4096 columns), the length of a block's K is what counts, and two groups of waves
// share it; and where there are fewer blocks still, they are of 128 columns, so that more CUs have one.  8 experts, 4096 x 14336, us of a forward, K not shared / 256 columns / 128:
// 100 tokens 446 / 418 / 373, 200 476 / 446 / 400, 256 503 / 466 / 420, 400 574 / 546 / 474.  As many blocks as CUs (the list's capacity, which holds a second piece for every expert): a second
// piece of an expert then finds no CU left among blocks of 128, and K not shared leaves CUs with one block: 512 tokens 656 / 624 / 654, 540 735 / 694 / 737, Zipf-1.1 632 / 606 / 624 and
// 651 / 634 / 658; 16 experts, 4 a token, 2048 x 6400 at 512 / 543 tokens 322, 344 / 313, 335 / 319, 348, Zipf-1.1 376, 392 / 366, 383 / 375, 392.  More blocks: 576 and 700 tokens 761, 789 / 749,
// 780 / 803, 843, 1000 962 / 1002 / 1045; 16 experts, 4096 x 6400 at 512 / 600 tokens 548, 684 / 592, 726 / 595, 753.
template <bool GLU>
static hipError_t start_bytes(const CodesArgs &a, const uint32_t *list, int cap, hipStream_t st) {
  constexpr int NI = GLU ? 128 : 256;
  const int64_t blocks = (int64_t)cap * ((a.N + NI - 1) / NI);
  if (blocks > 256 || a.K % 256) return start_bytes<GLU, 1, 2>(a, list, cap, st);
  if constexpr (!GLU)
    if (blocks < 256) return start_bytes<GLU, 2, 1>(a, list, cap, st);
  return start_bytes<GLU, 2, 2>(a, list, cap, st);
}
hipError_t launch_qmm_bytes(const CodesArgs &a, const uint32_t *list, int cap, bool glu, hipStream_t st) {
  return glu ? start_bytes<true>(a, list, cap, st) : start_bytes<false>(a, list, cap, st);
}

}  // namespace mi_moe
