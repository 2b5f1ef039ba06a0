// Grouped quantized product of short pieces: the segments of a mixture-of-experts block in pieces of up to 64 token rows, 4- and 8-bit codes.
//
// Contract: mlx_gather_qmm with transpose = true (mlx-rs/src/ops/quantization.rs:160-230).  The arithmetic is qmm_tiles.hip's: raw codes, the scale applied to the sums
// of a group, the bias term a product of its own over the group sums.  4-bit codes in groups of 64 have no centre, others are centred on the way in (signed_codes,
// centred_codes).  Share of results that are not the float64 product's nearest value, tiles of 32 x 32 results, which had these pieces before / here, K = 1024, 2048,
// 4096 (1e-4): 4-bit groups of 32 0.93, 1.21, 1.63 / the same, of 128 0.71, 0.89, 1.18 / 0.51, 0.66, 0.92 (scaled once for 128 values); 8-bit, of 32 0.87, 1.24, 1.71 / the same, of 128 0.75,
// 1.00, 1.24 / 0.76, 1.00, 1.24.  4-bit codes as they are, in sums that start from -8 times the sum of x, lose more (0.99, 1.28, 1.71; 0.98, 1.21, 1.74) and are no faster: us of a
// forward, those / centred, 128 experts, hidden 2048, groups of 32 at 100 / 256 / 512 tokens, even 121, 130, 149 / 122, 134, 149, Zipf-1.1 83, 101, 143 / 86, 100, 143; of 128 92, 108, 119 /
// 93, 107, 118 and 69, 84, 113 / 71, 83, 115.
#include <type_traits>

#include "lds_copies.hpp"
#include "qmm_codes_dev.hpp"

namespace mi_moe {

constexpr int kWaves = 8, kHalf = kWaves / 2, kShortLds = 80 * 1024;  // two blocks share a CU

// What a block of 16 MT token rows is made of.  A stage is 64 bytes of codes a weight row, 32 weight rows a wave.
template <int BITS, int GROUP, int MT>
struct Short {
  static constexpr bool kPlain = BITS == 4 && GROUP == 64;  // no centre
  static constexpr int KS = BITS == 4 ? 128 : 64, XROW = KS * 2;                            // K values of a stage, bytes of a token row
  static constexpr int SUB = GROUP < KS ? GROUP : KS, NG = KS / SUB, H = SUB / 32;         // what is scaled at once, of a stage; multiplies of that
  // A window's groups: its scales are fetched 16 at a time, or from a word on where a row has an odd number of them (groups of 128), and its group sums
  // have to fit a token row's place.
  static constexpr int GW = BITS == 8 ? (GROUP == 128 ? 4 : 8) : (GROUP == 128 ? 8 : 16), NW = GW * GROUP / KS;
  static constexpr int SLOTS = sum_slots(kPlain);
  static constexpr int X = 16 * MT * XROW, W = 2048, STAGE = X + kWaves * W, WINDOW = 1024;
  static constexpr int S = 3 * STAGE + kWaves * WINDOW <= kShortLds ? 3 : 2;
  static constexpr int BYTES = S * STAGE + kWaves * WINDOW;
  static constexpr int XALL = X / 1024, XI = (XALL + kWaves - 1) / kWaves;  // copies of a stage's token rows, and of a wave (where they do not go round, waves make the same ones)
  static constexpr int COPIES = XI + 2;
  static_assert(BYTES <= kShortLds && 16 * MT * (272 + 132 * 4) <= kShortLds && (NW == 4 || NW == 8), "two blocks share a CU");
};

// 16 MT token rows from sorted row `row0` (`rows` of them real) x 256 weight rows of expert e by eight waves of 32 weight rows each: GLU, 128 columns of h from n0:
// waves 0 to 3 the gate rows, 4 to 7 the up rows; else 256 columns from n0.
// A lane (weight row or token l % 16, quarter l / 16) multiplies a quarter of the K values that are scaled at once in steps of eight, v_mfma_f32_16x16x32_bf16.
// What bounds it: at few rows an expert memory (128 experts, K = 2048, 1536 columns, 100 tokens: 226 MB in 47 us), then the latency of a stage, a chain of reads of LDS,
// unpacking and multiplies that four waves of a SIMD fill up for each other.  That is why it is four: tiles of 32 x 32 results (qmm_pieces_kernel, which
// took these pieces) want 250 registers and leave two, whose stages took 2700 cycles where their vector instructions are 1630.  And why the stages are written
// out one by one: 120 instructions of a stage of 16 rows, against 185 with the places and windows found at run time (49 us for 56 at 100 tokens).  Blocks of
// four waves and 128 weight rows, four a CU: token rows twice as often through L2, and no room for a third stage of 32 rows (203 tokens: 109 us a forward for 102).
// Blocks that take several tiles of a piece one after the other: slower, their own bookkeeping costs what the ends give.
template <int BITS, int GROUP, bool GLU, int MT>
__device__ __forceinline__ void multiply_short(const CodesArgs &a, int e, int64_t row0, int rows, int n0, unsigned char *lds_raw) {
  typedef Short<BITS, GROUP, MT> R;
  constexpr int S = R::S, KS = R::KS, XROW = R::XROW, XP = XROW / 16, NG = R::NG, H = R::H, NW = R::NW, GLOG = GROUP == 32 ? 5 : GROUP == 64 ? 6 : 7;
  const int lane = threadIdx.x & 63, ln = lane & 15, kq = lane >> 4;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = a.N, K = a.K, G = K >> GLOG, row_bytes = K * BITS / 8, ext = padded_groups(G) * R::SLOTS;
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

  // ---- what a lane copies.  Sixteen-byte pieces of a row are turned by a number of the row's, so that sixteen rows' pieces of one number lie in different banks.
  auto turned = [](int row) __attribute__((always_inline)) { return XP == 16 ? row & 15 : (row >> 1) & 7; };
  uint32_t x_off[R::XI], sums_off[R::XI], w_off[2], window_row;
#pragma unroll
  for (int c = 0; c < R::XI; ++c) {
    const int r = (wave * R::XI + c) % R::XALL * (64 / XP) + lane / XP, tr = r < rows ? r : rows - 1;  // rows past the end repeat the last one (never stored)
    const uint32_t row = a.src_rows ? a.src_rows[row0 + tr] : (uint32_t)(row0 + tr), piece = (uint32_t)((lane % XP) ^ turned(r)) << 4;
    x_off[c] = row * (uint32_t)(K * 2) + piece;
    sums_off[c] = row * (uint32_t)(ext * 2) + piece;
  }
#pragma unroll
  for (int i = 0; i < 2; ++i) w_off[i] = (uint32_t)weight_row(16 * i + (lane >> 2)) * row_bytes + (((lane & 3) ^ ((lane >> 4) & 3)) << 4);
  window_row = ((uint32_t)weight_row(lane >> 1) * G * 2 & ~3u) + ((lane & 1) << 4);

  // ---- the stages: K in windows of GW groups, each a stage of the bias product, which brings the window's scales, and then NW stages of codes, written out one by
  // one.  Token rows are copied S - 1 stages ahead, a wave's weights S: their place is the wave's own and free once its codes are read.  (Past the end the last
  // values again.)
  const uint32_t x_at = ring_at + wave * R::XI % R::XALL * 1024, w_at = ring_at + R::X + wave * R::W;
  uint32_t turn[S];  // the places of a window's stages
#pragma unroll
  for (int i = 0; i < S; ++i) turn[i] = i * R::STAGE;
  auto place = [&](int n) __attribute__((always_inline)) { return (NW + 1) % S == 0 ? (uint32_t)(n % S * R::STAGE) : turn[n % S]; };
  // stage n of a window that begins at k: the bias product (0), or codes; n from NW + 1 on: of the next window
  auto weights_of = [&](int k, int n) __attribute__((always_inline)) {
    const bool bias = n % (NW + 1) == 0;
    const int at = n <= NW ? k + KS * (n ? n - 1 : 0) : k + KS * (NW + (bias ? 0 : n - NW - 2)), from = bias ? (at < K ? at : 0) >> GLOG << 1 : (at < K ? at : K - KS) * BITS / 8;
#pragma unroll
    for (int i = 0; i < 2; ++i) copy_to_lds(!bias ? wr : i ? br : sr, bias ? window_row : w_off[i], from, w_at + place(n) + i * 1024);
  };
  auto rows_of = [&](int k, int n) __attribute__((always_inline)) {
    const bool bias = n % (NW + 1) == 0;
    const int at = n <= NW ? k + KS * (n ? n - 1 : 0) : k + KS * (NW + (bias ? 0 : n - NW - 2)), from = bias ? ((at < K ? at : 0) >> GLOG) * (2 * R::SLOTS) : (at < K ? at : K - KS) * 2;
#pragma unroll
    for (int c = 0; c < R::XI; ++c) copy_to_lds(bias ? xsr : xr, bias ? sums_off[c] : x_off[c], from, x_at + place(n) + c * 1024);
  };
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
  // Where a lane's pieces lie, each in a register whose parts the compiler does not see: constants beyond 64 KB of LDS would each take one of their own.
  uint32_t f_at[NG * H], q_at[NG], s_at[2];
#pragma unroll
  for (int i = 0; i < NG * H; ++i) f_at[i] = ln * XROW + (((i / H * (R::SUB / 8) + kq * H + i % H) ^ turned(ln)) << 4);
#pragma unroll
  for (int g = 0; g < NG; ++g) {  // 8 H of the SUB values at once
    const int byte = g * (R::SUB * BITS / 8) + kq * (H * BITS);
    q_at[g] = R::X + wave * R::W + ln * 64 + (((byte >> 4) ^ ((ln >> 2) & 3)) << 4) + (byte & 15);
  }
  int late[2];  // groups of 128: a row's first scale lies behind another row's in its word
#pragma unroll
  for (int j = 0; j < 2; ++j) {
    late[j] = GROUP == 128 ? weight_row(16 * j + ln) & G & 1 : 0;
    s_at[j] = S * R::STAGE + wave * R::WINDOW + (16 * j + ln) * 32 + late[j] * 2;
    asm volatile("" : "+v"(s_at[j]));
  }
#pragma unroll
  for (int i = 0; i < NG * H; ++i) asm volatile("" : "+v"(f_at[i]));
#pragma unroll
  for (int g = 0; g < NG; ++g) asm volatile("" : "+v"(q_at[g]));
  auto code_stage = [&](int k, int n) __attribute__((always_inline)) {
    uint32_t from = place(n);
    if constexpr ((NW + 1) % S != 0) asm volatile("" : "+s"(from));  // (added where it is wanted: every stage's addresses at once do not fit the registers)
    begin();
    rows_of(k, n + S - 1);
    constexpr int STEPS = NG * MT, AHEAD = (MT < 2 && H == 2) || H == 4 ? 1 : 2;  // sixteen rows of SUB values each; fetched ahead
    uint32_t q[2][4], s2[2][2];
    u32x4_t F[AHEAD][H];
    auto fetch = [&](int i) __attribute__((always_inline)) {
      if (i >= STEPS) return;
      const int g = i / MT, m = i % MT;
#pragma unroll
      for (int h = 0; h < H; ++h) F[i % AHEAD][h] = *reinterpret_cast<const u32x4_t *>(lds_raw + f_at[g * H + h] + from + m * (16 * XROW));
    };
#pragma unroll
    for (int g = 0; g < NG; ++g)
#pragma unroll
      for (int j = 0; j < 2; ++j) __builtin_memcpy(&q[j][g * 4 / NG], __builtin_assume_aligned(lds_raw + q_at[g] + from + j * 1024, 16 / NG), 16 / NG);
#pragma unroll
    for (int i = 0; i < AHEAD; ++i) fetch(i);
#pragma unroll
    for (int j = 0; j < 2; ++j) {  // the stage's scales, in the upper or lower half of a word each
      if constexpr (NG == 4) __builtin_memcpy(s2[j], __builtin_assume_aligned(lds_raw + s_at[j] + 8 * (n - 1), 8), 8);
      else if constexpr (NG * GROUP == KS && NG == 2) s2[j][0] = *reinterpret_cast<const uint32_t *>(lds_raw + s_at[j] + 4 * (n - 1));
      else s2[j][0] = *reinterpret_cast<const uint16_t *>(lds_raw + s_at[j] + 2 * ((n - 1) * KS / GROUP));
    }
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      u32x4_t op[2][H];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int h = 0; h < H; ++h) {
          const int i = g * H + h;
          if constexpr (BITS == 4) {
            if constexpr (R::kPlain) plain_codes(q[j][i], op[j][h]);
            else signed_codes(q[j][i], op[j][h]);
          } else {
#pragma unroll
            for (int w = 0; w < 2; ++w) {
              float v[4];
              centred_codes(q[j][2 * i + w], v);
              op[j][h][2 * w] = upper_halves(v[0], v[1]);
              op[j][h][2 * w + 1] = upper_halves(v[2], v[3]);
            }
          }
        }
      if (g == NG - 1) {  // (the stage's codes have been read: a copy out of L2 may overtake a read of LDS that waits its turn)
#pragma unroll
        for (int j = 0; j < 2; ++j)
#pragma unroll
          for (int h = 0; h < H; ++h) asm volatile("" : "+v"(op[j][h]));
        weights_of(k, n + S);
      }
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const int i = g * MT + m;
        f32x4_t acc[2];
#pragma unroll
        for (int h = 0; h < H; ++h)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[j] = mfma<0>(F[i % AHEAD][h], op[j][h], h ? acc[j] : zero);
        fetch(i + AHEAD);
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const uint32_t w = s2[j][NG == 4 ? g / 2 : 0];
          const float s = __uint_as_float(NG * GROUP == KS && (g & 1) ? w & 0xffff0000u : w << 16);
#pragma unroll
          for (int r = 0; r < 4; ++r) tot[j][m][r] = __builtin_fmaf(s, acc[j][r], tot[j][m][r]);
        }
      }
    }
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int m = 0; m < MT; ++m) asm volatile("" : "+v"(tot[j][m]));  // (added here, not where a stage ends the row: with every stage's sums kept until then they spill)
  };
#pragma unroll 1
  for (int k = 0; k < K; k += NW * KS) {
    {  // the bias product of the window (real: groups from there on are not this row's)
      begin();
      rows_of(k, S - 1);
      const int real = G - (k >> GLOG);
      // groups of a multiply, multiplies; the four groups of 128 of a window are added with the next one's, by every other window (one rounding for two)
      constexpr int PER = 32 / R::SLOTS, NB = (R::GW + PER - 1) / PER, MOST = R::GW == 4 ? 2 * NB : NB;
      const int here = MOST == NB ? NB : k & NW * KS ? 0 : MOST;
      const unsigned char *const rows_at = lds_raw + place(0), *const mine = mine_at + place(0);
      f32x4_t sum[2][MT];
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m) sum[j][m] = zero;
#pragma unroll
      for (int i = 0; i < MOST; ++i) {
        if (i >= here) break;
        u32x4_t F[MT], o[2];
#pragma unroll
        for (int m = 0; m < MT; ++m) F[m] = *reinterpret_cast<const u32x4_t *>(rows_at + m * (16 * XROW) + ln * XROW + (((4 * i + kq) ^ turned(ln)) << 4));
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const unsigned char *const at = mine + (16 * j + ln) * 32;
          if constexpr (R::kPlain) {  // the sums' three pieces against the bias, a bf16 as it is
            const int g = 8 * i + 2 * kq;
            const uint32_t b = g < real ? *reinterpret_cast<const uint32_t *>(at + 1024 + g * 2) : 0u;  // (an even number of groups)
            o[j] = u32x4_t{__builtin_amdgcn_perm(b, b, 0x01000100u), b & 0xffffu, __builtin_amdgcn_perm(b, b, 0x03020302u), b >> 16};
          } else {  // against three pieces of the bias and the centre's share of it
            const int g = 4 * i + kq;
            const float sv = as_f32(*reinterpret_cast<const uint16_t *>(at + (g + late[j]) * 2)), bv = as_f32(*reinterpret_cast<const uint16_t *>(at + 1024 + (g + late[j]) * 2));
            const Pieces p = split3(g < real ? __builtin_fmaf(centre_of(BITS), sv, bv) : 0.f);
            o[j] = u32x4_t{p.h | p.h << 16, p.h | p.m << 16, p.m | p.l << 16, 0u};
          }
        }
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int j = 0; j < 2; ++j) sum[j][m] = mfma<0>(F[m], o[j], sum[j][m]);
      }
      *reinterpret_cast<u32x4_t *>(scales + lane * 16) = *reinterpret_cast<const u32x4_t *>(mine + lane * 16);
      wait_reads();
      weights_of(k, S);
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int m = 0; m < MT; ++m)
#pragma unroll
          for (int r = 0; r < 4; ++r) tot[j][m][r] += sum[j][m][r];
    }
    const int stages = (K - k) / KS;  // of codes, NW of them in this window
#pragma unroll
    for (int n = 1; n <= NW; ++n) {
      code_stage(k, n);
      if (n == stages) break;
    }
    uint32_t was[S];
#pragma unroll
    for (int i = 0; i < S; ++i) was[i] = turn[i];
#pragma unroll
    for (int i = 0; i < S; ++i) turn[i] = was[(i + NW + 1) % S];
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
          plain_rows<BITS, 4, uint16_t>(xs, BITS == 4 ? RowOrder::kQuads : RowOrder::kPlain, (i ? a.w1 : a.w0) + wrow * (row_bytes / 4), static_cast<const uint16_t *>(i ? a.s1 : a.s0) + wrow * G,
                                     static_cast<const uint16_t *>(i ? a.b1 : a.b0) + wrow * G, K, GROUP, open, v[i]);
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
    constexpr int LANES = GROUP / 8;  // of a group; sixteen of a row
    const int groups = N >> GLOG, padded = padded_groups(groups), piece = threadIdx.x & 15, g0 = (n0 >> GLOG) + piece / LANES;
#pragma unroll
    for (int r0 = 0; r0 < 16 * MT; r0 += 4 * kWaves) {
      const int row = r0 + (int)(threadIdx.x >> 4);
      const u32x4_t w = *reinterpret_cast<const u32x4_t *>(out + row * ROWB + piece * 16);
      float sum = ((bf16lo_to_f32(w[0]) + bf16hi_to_f32(w[0])) + (bf16lo_to_f32(w[1]) + bf16hi_to_f32(w[1]))) +
                  ((bf16lo_to_f32(w[2]) + bf16hi_to_f32(w[2])) + (bf16lo_to_f32(w[3]) + bf16hi_to_f32(w[3])));
      sum += __uint_as_float(dpp_u32<kDppXor1>(__float_as_uint(sum)));
      sum += __uint_as_float(dpp_u32<kDppXor2>(__float_as_uint(sum)));
      if (GROUP >= 64) sum += __uint_as_float(dpp_u32<kDppHalfMirror>(__float_as_uint(sum)));
      if (GROUP == 128) sum += __uint_as_float(dpp_u32<kDppMirror>(__float_as_uint(sum)));
      if (row < rows) {
        *reinterpret_cast<u32x4_t *>(static_cast<uint16_t *>(a.y) + (row0 + row) * N + n0 + 8 * piece) = w;
        uint16_t *const sums = a.y_sums + (row0 + row) * padded * R::SLOTS;
        if (piece % LANES == 0) put_sums(sums + g0 * R::SLOTS, R::SLOTS, sum);
        if (n0 + 128 >= N)  // the last block of a row writes the zeros behind its sums
          for (int g = groups + piece; g < padded; g += 16) put_sums(sums + g * R::SLOTS, R::SLOTS, 0.f);
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
template <int BITS, int GROUP, bool GLU>
__global__ __launch_bounds__(64 * kWaves, 4) void qmm_short_kernel(CodesArgs a, const uint32_t *__restrict__ list, int cap, int n_ntiles) {
  const uint32_t xcd = blockIdx.x & 7, j = blockIdx.x >> 3, id = j / (uint32_t)n_ntiles * 8u + xcd;
  const int n0 = (int)(j % (uint32_t)n_ntiles) * (GLU ? 128 : 256);
  const uint4 rec = reinterpret_cast<const uint4 *>(list)[1 + (id < (uint32_t)cap ? id : (uint32_t)cap - 1u)];  // (beside the count, not behind it)
  if (id >= list[0]) return;
  const int e = __builtin_amdgcn_readfirstlane((int)rec.x), rows = __builtin_amdgcn_readfirstlane((int)rec.z);
  const int64_t row0 = (int64_t)__builtin_amdgcn_readfirstlane((int)rec.y);
  extern __shared__ __align__(16) unsigned char lds_raw[];
  if (rows > 48) multiply_short<BITS, GROUP, GLU, 4>(a, e, row0, rows, n0, lds_raw);
  else if (rows > 32) multiply_short<BITS, GROUP, GLU, 3>(a, e, row0, rows, n0, lds_raw);
  else if (rows > 16) multiply_short<BITS, GROUP, GLU, 2>(a, e, row0, rows, n0, lds_raw);
  else multiply_short<BITS, GROUP, GLU, 1>(a, e, row0, rows, n0, lds_raw);
}

template <int BITS, int GROUP, bool GLU>
static hipError_t start_short(const CodesArgs &a, const uint32_t *list, int cap, hipStream_t st) {
  constexpr int NI = GLU ? 128 : 256;
  const int n_ntiles = (a.N + NI - 1) / NI;
  const int64_t grid = ((int64_t)cap + 7) / 8 * 8 * n_ntiles;
  if (grid <= 0 || grid > INT32_MAX || a.N % 128 || a.K % 128) return hipErrorInvalidValue;
  const auto kernel = &qmm_short_kernel<BITS, GROUP, GLU>;
  static std::atomic<uint64_t> allowed{0};
  if (hipError_t e = allow_lds(reinterpret_cast<const void *>(kernel), kShortLds, allowed); e != hipSuccess) return e;
  launch_or_time(kernel, dim3((unsigned)grid), dim3(64 * kWaves), kShortLds, st, a, list, cap, n_ntiles);
  return hipGetLastError();
}
hipError_t launch_qmm_short(const CodesArgs &a, const uint32_t *list, int cap, int group, int bits, bool glu, hipStream_t st) {
  auto run = [&](auto b, auto g) {
    constexpr int BITS = decltype(b)::value, GROUP = decltype(g)::value;
    return glu ? start_short<BITS, GROUP, true>(a, list, cap, st) : start_short<BITS, GROUP, false>(a, list, cap, st);
  };
  auto with_group = [&](auto b) {
    if (group == 32) return run(b, std::integral_constant<int, 32>{});
    return group == 64 ? run(b, std::integral_constant<int, 64>{}) : run(b, std::integral_constant<int, 128>{});
  };
  return bits == 4 ? with_group(std::integral_constant<int, 4>{}) : with_group(std::integral_constant<int, 8>{});
}

}  // namespace mi_moe
