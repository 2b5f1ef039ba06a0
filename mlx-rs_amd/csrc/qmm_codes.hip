// The middle of the range of dense products on raw codes (which: dense_rule.hpp; contract, arithmetic and prepared rows: qmm_tiles.hip, with
// c = 8 or 128): tiles of 64 x 128, and of 32 x 64 for bf16 and 8-bit codes in groups of 32, whose waves load their codes straight into the registers that unpack them.
#include <type_traits>

#include "qmm_codes_dev.hpp"

namespace mi_moe {

namespace {

constexpr int kStep = 64;      // K values per step; two steps between barriers
constexpr int kRow = 17;       // LDS row stride in 16-byte units: 128 values and 16 bytes that keep rows off each other's banks
constexpr uint32_t kOutside = 0x80000000u;  // an offset past every descriptor here: such a load returns zeros
constexpr int kWeave = 7;  // vector instructions between two matrix instructions
constexpr size_t kLdsAtLeast = 4 * 32 * (32 * 2 + 16);  // the epilogue's staging

typedef uint32_t u32x3_t __attribute__((ext_vector_type(3)));

// a multiply function together with how it deals K values to its four multiplies (see qmm_codes_kernel)
template <bool SPLIT, class F>
struct Split : F {
  static constexpr bool split = SPLIT;
  __device__ __forceinline__ Split(F f) : F(f) {}
};
template <bool SPLIT, class F>
__device__ __forceinline__ Split<SPLIT, F> with_split(F f) { return Split<SPLIT, F>(f); }

}  // namespace

// A block computes 32 MS token rows x 32 WN weight rows with WN KW waves.  A wave owns 32 weight
// rows for all the block's token rows, so it loads its own codes straight
// into the lanes that multiply them and unpacks them in registers: nothing of the weights passes through LDS, and no
// wave unpacks what another one does.  A lane (weight row l % 32, half l / 32) loads 16 bytes; which K values its
// eight codes of a multiply stand for is free as long as the token operand agrees:
//   4-bit, groups >= 64: 16 bytes are 32 codes, half h holds K values 32 h ..: multiply t takes word t of both halves;
//   4-bit, groups of 32: two v_permlane32_swap deal the words so that a multiply stays inside one group;
//   8-bit: 16 bytes are 16 codes, two loads a step, groups of 32 stay apart by themselves.
// Token rows pass through LDS (128 K values between two barriers, double-buffered).
// A step takes one 32 x 32 sub-tile after the other: its four multiplies follow each other in one accumulator, and the
// scaled addition of the sub-tile before it (16 fma) and the unpacking of the next step's codes (10 to 15 instructions a
// multiply) run between them, which is as much vector work as fits beside the matrix cores.
// What bounds it (777 x 4096 x 4096, f16, 8-bit; 26 GFLOP): 54 us for the call = 480 TFLOP/s (the plain kernel
// 3160 us); the matrix cores alone would take 18.  Taken apart at one block a CU (cycles per 64 K values of 128 x 32 a
// wave, 512 of them matrix work): multiplies and barriers 575, with the vector work 640, with the reads of LDS 840, with
// the loads 1350.  The loads cost their line visits: a wave's codes sit in 32 rows.
// KW > 1: the block's waves form KW groups that share K among them, each with LDS buffers of its own; their sums meet in
// LDS at the end, added in group order.  For launches that give a CU one block or less.
// DT: 0 bf16, 1 f16.  G32: groups of 32; otherwise a group is one or two steps (scale_shift).
template <int DT, int BITS, bool G32, int MS, int WN, int KW>
__global__ __launch_bounds__(64 * WN * KW) __attribute__((amdgpu_waves_per_eu(2, 4))) void qmm_codes_kernel(
    CodesArgs a, int n_mtiles, int n_ntiles, int scale_shift) {
  typedef typename ElemOf<DT>::type T;
  constexpr int BM = 32 * MS, NT = 1;        // (weight tiles of a wave)
  constexpr int NI = 32 * WN;                // output columns per block
  constexpr int NA = BM * 8 / (64 * WN);     // 16-byte activation loads per thread, piece and step
  constexpr int RS = 8 * WN;                 // rows one such load of a group covers
  constexpr int NQ = BITS == 4 ? 1 : 2;      // 16-byte code loads per lane, tile and step
  constexpr int NS = G32 ? 2 : 1;            // scaled additions per sub-tile and step
  constexpr bool SPLIT = BITS == 8 || G32;   // which K values a multiply takes: see chunk below
  constexpr float kUnit = BITS == 4 && DT == 0 ? 0.0625f : 1.0f;  // the codes are multiplied as (q - centre) / kUnit
  constexpr int A_SZ = BM * kRow, BUF = A_SZ;                      // 16-byte units
  static_assert(BM % RS == 0, "whole loads");

  // block -> (M tile, N tile).  Ids are dealt round-robin over the 8 XCDs: an XCD takes every eighth N tile and all M tiles of it, so its
  // L2 holds the weights of a few N tiles and x streams through.
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int nt = j / n_mtiles * 8 + xcd;
  if (nt >= n_ntiles) return;
  const int64_t row0 = (int64_t)(j % n_mtiles) * BM;
  const int rows = a.M - row0 < BM ? (int)(a.M - row0) : BM;

  const int lane = threadIdx.x & 63;
  const int wave_all = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = wave_all % WN, kg = wave_all / WN;  // column tile, K group
  const int tid = wave * 64 + lane;                    // within the K group
  const int N = a.N, K = a.K;
  const int n0 = nt * NI;
  const int G = K / (G32 ? 32 : 64 << scale_shift), row_bytes = K * BITS / 8;

  extern __shared__ __align__(16) unsigned char lds_raw[];
  u32x4_t *const lds = reinterpret_cast<u32x4_t *>(lds_raw) + kg * (2 * BUF);

  // ---- what a thread stages: chunk acp (8 K values) of token rows arg, arg + RS, ...  Offsets are 32 bits: the host
  // takes this kernel for operands below 4 GiB only.
  const int acp = tid & 7, arg = tid >> 3;
  const int pg = padded_groups(G), ext = pg * kSlots;
  const __amdgpu_buffer_rsrc_t xr = rsrc_of(a.x, (uint32_t)(a.x_rows * K * sizeof(T))), xsr = rsrc_of(a.sums, (uint32_t)(a.x_rows * ext * 2));
  uint32_t x_voff[NA], xs_voff[NA];
#pragma unroll
  for (int i = 0; i < NA; ++i) {
    int tr = arg + RS * i;
    tr = tr < rows ? tr : rows - 1;  // rows past the end repeat the last one (never stored)
    const uint32_t r = (uint32_t)(row0 + tr);
    x_voff[i] = (r * (uint32_t)K + acp * 8) * sizeof(T);
    xs_voff[i] = (r * (uint32_t)ext + acp * 8) * 2;
  }
  // ---- the weight rows of this lane
  const int ln = lane & 31, kb = lane >> 5;
  const int w_row[NT] = {n0 + 32 * wave + ln < N ? n0 + 32 * wave + ln : N - 1};  // columns past the end repeat the last one (never stored)
  const __amdgpu_buffer_rsrc_t wr[NT] = {rsrc_of(a.w0, (uint32_t)N * row_bytes)};
  const __amdgpu_buffer_rsrc_t sr[NT] = {rsrc_of(a.s0, (uint32_t)N * G * sizeof(T))};  // (read in words: the host takes an even number of them)
  const __amdgpu_buffer_rsrc_t br[NT] = {rsrc_of(a.b0, (uint32_t)N * G * sizeof(T))};
  const uint32_t w_voff[NT] = {(uint32_t)w_row[0] * row_bytes + kb * 16}, s_voff[NT] = {(uint32_t)(w_row[0] * G * (int)sizeof(T))};

  f32x16_t tot[MS][NT];
  const f32x16_t zero = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t) tot[m][t] = zero;

  struct StageA {  // a thread's share of a step's token rows
    u32x4_t v[NA];
  };
  struct Operand {  // a step's weight operand: eight values a lane and multiply
    u32x4_t v[NT][4];
  };
  auto nk_share = [](int nk) __attribute__((always_inline)) { return (nk / 2 + KW - 1) / KW * 2; };  // steps of a K group
  // One pipelined pass of nk steps (an even number), dealt to the K groups in even shares (what a share has past the
  // last step is multiplied with zeros).  Two steps at a time: while they are multiplied out of one LDS buffer, the
  // token rows of the next two are on their way into registers, the codes run two steps ahead and are unpacked one
  // step ahead.
  // window_steps, window: called ahead of every so many steps.
  // Inside a step the sub-tiles follow each other, each with the reads of the next one's token rows ahead of its
  // multiplies and its share of the unpacking between them; nothing moves across a sub-tile.
  auto pass = [&](int nk, auto b_type, auto load_a, auto load_b, auto unpack, auto begin, auto multiply, int window_steps, auto window) __attribute__((always_inline)) {
    StageA RA[2];
    decltype(b_type) RB[2];
    auto put = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int d = 0; d < 2; ++d)
#pragma unroll
        for (int i = 0; i < NA; ++i) lds[buf * BUF + (arg + RS * i) * kRow + 8 * d + acp] = RA[d].v[i];
    };
    const int share = nk_share(nk);  // the same number of barriers for every group
    const int k0 = kg * share, k1 = k0 + share < nk ? k0 + share : nk;
    auto clamped = [&](int ks) __attribute__((always_inline)) { return ks < nk ? ks : nk - 1; };
    load_b(clamped(k0), RB[0]);
    load_a(clamped(k0), k0 < k1, RA[0]);
    load_a(clamped(k0 + 1), k0 < k1, RA[1]);
    load_b(clamped(k0 + 1), RB[1]);
    Operand op[2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int h = 0; h < 4; ++h) unpack(RB[0], op[0], t, h);
    put(0);
    __syncthreads();
    u32x4_t F[2][4];  // the token operand of a sub-tile row, and of the next
    auto fetch = [&](const u32x4_t *At, int m, bool split, u32x4_t (&to)[4]) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 4; ++h)
        to[h] = At[(32 * m + ln) * kRow + (split ? 4 * (h >> 1) + 2 * kb + (h & 1) : 4 * kb + h)];  // the chunk multiply h takes
    };
    int buf = 0;
    for (int kw = k0; kw < k0 + share; kw += window_steps) {
      window(kw);
      for (int kq = kw; kq < k0 + share && kq < kw + window_steps; kq += 2) {
        const u32x4_t *const At = lds + buf * BUF;
        buf ^= 1;
        fetch(At, 0, decltype(multiply)::split, F[0]);
#pragma unroll
        for (int d = 0; d < 2; ++d) {
          load_b(clamped(kq + d + 2), RB[d]);
          if (d == 0) {
            load_a(clamped(kq + 2), kq + 2 < k1, RA[0]);
            load_a(clamped(kq + 3), kq + 2 < k1, RA[1]);
          }
          begin(kq + d, d);
          __builtin_amdgcn_sched_barrier(0);  // (the loads stay at the head of the step)
#pragma unroll
          for (int m = 0; m < MS; ++m)
#pragma unroll
            for (int t = 0; t < NT; ++t) {
              if (t == 0 && m + 1 < MS) fetch(At + 8 * d, m + 1, decltype(multiply)::split, F[(d * MS + m + 1) & 1]);
              if (t == 0 && m + 1 == MS && d == 0) fetch(At + 8, 0, decltype(multiply)::split, F[MS & 1]);
              multiply(F[(d * MS + m) & 1], op[d], d, m, t);
              constexpr int UNITS = 4 * NT, TILES = MS * NT;
#pragma unroll
              for (int u = UNITS * (m * NT + t) / TILES; u < UNITS * (m * NT + t + 1) / TILES; ++u) unpack(RB[d ^ 1], op[d ^ 1], u / 4, u % 4);
              if (t == 0 && (m + 1 < MS || d == 0)) __builtin_amdgcn_sched_group_barrier(0x100, 4, 0);
#pragma unroll
              for (int i = 0; i < 4; ++i) {
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                __builtin_amdgcn_sched_group_barrier(0x002, kWeave, 0);
              }
              __builtin_amdgcn_sched_barrier(0);
            }
          if (d == 1) {
            put(buf);
            __syncthreads();
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };

  // ---- the bias product: group sums of x against b + centre s, accumulated into the result
  {
    // A lane's four groups of a step are three words, as a row may start between two.  Groups past the row's end are another
    // row's or zeros: their sums are zero.
    struct StageB {
      u32x3_t s[NT], b[NT];
    };
    auto load_a = [&](int ks, bool real, StageA &R) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NA; ++i)
        R.v[i] = __builtin_amdgcn_raw_buffer_load_b128(xsr, KW == 1 || real ? xs_voff[i] : kOutside, ks * (kStep * 2), 0);
    };
    auto load_b = [&](int ks, StageB &R) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const uint32_t off = (s_voff[t] + (ks * 8 + 4 * kb) * (uint32_t)sizeof(T)) & ~3u;
        R.s[t] = __builtin_amdgcn_raw_buffer_load_b96(sr[t], off, 0, 0);
        R.b[t] = __builtin_amdgcn_raw_buffer_load_b96(br[t], off, 0, 0);
      }
    };
    auto unpack = [&](const StageB &R, Operand &o, int t, int h) __attribute__((always_inline)) {
      const auto group = [&](const u32x3_t &v) __attribute__((always_inline)) {  // (row starts are even numbers of bytes)
        const uint32_t pair = __builtin_amdgcn_alignbyte(v[h / 2 + 1], v[h / 2], s_voff[t]);
        return as_f32(__builtin_bit_cast(T, (uint16_t)(h % 2 ? pair >> 16 : pair)));
      };
      const Pieces p = split3(__builtin_fmaf(centre_of(BITS), group(R.s[t]), group(R.b[t])));
      o.v[t][h] = u32x4_t{p.h | p.h << 16, p.h | p.m << 16, p.m | p.l << 16, 0u};
    };
    auto body = [&](const u32x4_t (&av)[4], const Operand &o, int, int m, int t) __attribute__((always_inline)) {
#pragma unroll
      for (int h = 0; h < 4; ++h) tot[m][t] = mfma<0>(av[h], o.v[t][h], tot[m][t]);
    };
    pass(pg / 8, StageB{}, load_a, load_b, unpack, [](int, int) {},
         with_split<false>(body), 1 << 30, [](int) {});
  }

  // ---- the product of the codes
  {
    struct StageB {
      u32x4_t q[NT][NQ];
    };
    f32x16_t acc[2];  // the group of a sub-tile being multiplied, and the one before it
    float acc_s[2];
    acc[1] = zero;  // (nothing is pending yet)
    acc_s[1] = 0.f;
    auto add_scaled = [&](int which, int tile) __attribute__((always_inline)) {
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[tile / NT][tile % NT][r] = __builtin_fmaf(acc_s[which], acc[which][r], tot[tile / NT][tile % NT][r]);
    };
    auto load_a = [&](int ks, bool real, StageA &R) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NA; ++i)
        R.v[i] = __builtin_amdgcn_raw_buffer_load_b128(xr, KW == 1 || real ? x_voff[i] : kOutside, ks * (kStep * (uint32_t)sizeof(T)), 0);
    };
    auto load_b = [&](int ks, StageB &R) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int h = 0; h < NQ; ++h)
          R.q[t][h] = __builtin_amdgcn_raw_buffer_load_b128(wr[t], w_voff[t], ks * (kStep * BITS / 8) + 32 * h, 0);
      }
    };
    auto unpack = [&](StageB &R, Operand &o, int t, int h) __attribute__((always_inline)) {
      if constexpr (BITS == 4 && G32) {
        if (h == 0) {
#pragma unroll
          for (int w = 0; w < 2; ++w) {
            const auto r = __builtin_amdgcn_permlane32_swap(R.q[t][0][w], R.q[t][0][w + 2], false, false);
            R.q[t][0][w] = r[0];
            R.q[t][0][w + 2] = r[1];
          }
        }
      }
      if constexpr (BITS == 4 && DT == 0) {
        float v[8];
        centred_codes(R.q[t][0][h], v);
#pragma unroll
        for (int i = 0; i < 4; ++i) o.v[t][h][i] = upper_halves(v[i], v[i + 4]);
      } else if constexpr (BITS == 4) {
        const uint32_t w = R.q[t][0][h];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (i % 2 == 0) {
            o.v[t][h][i] = f16_centred<4>(__builtin_amdgcn_bitop3_b32(w >> (4 * i), 0x000f000fu, 0x64006400u, 0xEA));  // (a & b) | c
          } else {  // 1024 + 16 q -> q - 8, exact as well: one shift serves two nibbles
            const half2_t v = __builtin_bit_cast(half2_t, __builtin_amdgcn_bitop3_b32(w >> (4 * (i - 1)), 0x00f000f0u, 0x64006400u, 0xEA));
            o.v[t][h][i] = __builtin_bit_cast(uint32_t, __builtin_elementwise_fma(v, half2_t{(_Float16)0.0625f, (_Float16)0.0625f}, half2_t{(_Float16)-72.0f, (_Float16)-72.0f}));
          }
        }
      } else if constexpr (DT == 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i)  // bytes 2 i, 2 i + 1 under the exponent of 1024
          o.v[t][h][i] = f16_centred<8>(__builtin_amdgcn_perm(0x64646464u, R.q[t][h >> 1][2 * (h & 1) + (i >> 1)],
                                                              (i & 1) ? 0x07030702u : 0x07010700u));
      } else {
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          float v[4];
          centred_codes(R.q[t][h >> 1][2 * (h & 1) + (i >> 1)], v);
          o.v[t][h][i] = upper_halves(v[0], v[1]);
          o.v[t][h][i + 1] = upper_halves(v[2], v[3]);
        }
      }
    };
    // The scales of this wave's rows pass through LDS a window at a time: a lane fetches 16 bytes of its row (half kb of
    // the window) one window ahead, and reads one value per group back.  One 2-byte load per group from a row each
    // touches as many lines as the codes themselves (measured: a quarter of the kernel's time).
    // The fetch is aligned down to 4 bytes.  Where a window can start between two words (an odd number of 2-byte scales
    // per row, or per K group: groups of 128), the sixteenth scale would lie behind the fetch: windows of eight then.
    const int first_group = (nk_share(K / kStep) * kg) * (G32 ? 2 : 1) >> scale_shift, share_groups = nk_share(K / kStep) * (G32 ? 2 : 1) >> scale_shift;
    const int win = ((G | share_groups) & 1) ? 8 : 16;  // scales of a window
    constexpr int SROW = 32 + 16;                  // bytes per row of the window
    unsigned char *const swin = reinterpret_cast<unsigned char *>(lds_raw) + 2 * KW * BUF * 16 + wave_all * (NT * 32 * SROW);
    u32x4_t swin_next[NT];
    auto load_window = [&](int g) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
        swin_next[t] = __builtin_amdgcn_raw_buffer_load_b128(sr[t], ((s_voff[t] + g * (uint32_t)sizeof(T)) & ~3u) + kb * 16, 0, 0);
    };
    load_window(first_group);
    int gw = first_group;        // first group of the window in LDS
    const unsigned char *s_at[NT];  // this lane's scale of that group
    auto window = [&](int ks) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t) *reinterpret_cast<u32x4_t *>(swin + (t * 32 + ln) * SROW + kb * 16) = swin_next[t];
      gw = (ks * (G32 ? 2 : 1)) >> scale_shift;
      load_window(gw + win);
#pragma unroll
      for (int t = 0; t < NT; ++t) s_at[t] = swin + (t * 32 + ln) * SROW + ((s_voff[t] + gw * (uint32_t)sizeof(T)) & 3u);
      __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
      __builtin_amdgcn_wave_barrier();
      __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    };
    float step_s[2][NT][NS];
    auto begin = [&](int ks, int d) __attribute__((always_inline)) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int i = 0; i < NS; ++i)
          step_s[d][t][i] = kUnit * as_f32(*reinterpret_cast<const T *>(s_at[t] + ((G32 ? 2 * ks + i : ks >> scale_shift) - gw) * (int)sizeof(T)));
    };
    auto body = [&](const u32x4_t (&av)[4], const Operand &o, int d, int m, int t) __attribute__((always_inline)) {
      const int tile = m * NT + t;
#pragma unroll
      for (int i = 0; i < NS; ++i) {
        const int which = ((d * MS * NT + tile) * NS + i) & 1;
#pragma unroll
        for (int h = 4 / NS * i; h < 4 / NS * (i + 1); ++h)
          acc[which] = mfma<DT>(av[h], o.v[t][h], h == 4 / NS * i ? zero : acc[which]);
        acc_s[which] = step_s[d][t][i];
        add_scaled(which ^ 1, i > 0 ? tile : tile > 0 ? tile - 1 : MS * NT - 1);
      }
    };
    pass(K / kStep, StageB{}, load_a, load_b, unpack, begin, with_split<SPLIT>(body),
         (win >> (G32 ? 1 : 0)) << scale_shift, window);
    add_scaled(1, MS * NT - 1);  // an even number of steps ends in accumulator 1
  }

  if constexpr (KW > 1) {  // (the passes end in a barrier: LDS is free)
    float *const parts = reinterpret_cast<float *>(lds_raw) + (wave * 64 + lane) * 4;  // 16-byte pieces, lane by lane
    constexpr int kPiece = 64 * WN * 4;
#pragma unroll
    for (int g = 1; g < KW; ++g) {
      if (kg == g) {
#pragma unroll
        for (int m = 0; m < MS; ++m)
#pragma unroll
          for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int r = 0; r < 4; ++r)
              *reinterpret_cast<float4 *>(parts + ((m * NT + t) * 4 + r) * kPiece) =
                  make_float4(tot[m][t][4 * r], tot[m][t][4 * r + 1], tot[m][t][4 * r + 2], tot[m][t][4 * r + 3]);
      }
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

  // ---- epilogue: a wave turns its 32 x 32 sub-tiles round in a private piece of LDS and stores 16 bytes a lane
  constexpr int ROWB = 32 * (int)sizeof(T) + 16;
  constexpr int PV = 16 / (int)sizeof(T);             // values per 16-byte piece
  constexpr int CPR = 32 / PV;                        // pieces per row
  constexpr int RPI = 64 / CPR;                       // rows one store instruction covers
  static_assert(WN * 32 * ROWB <= kLdsAtLeast, "staging does not fit");
  unsigned char *const mine = lds_raw + wave * (32 * ROWB);
  const int my_piece = lane % CPR, my_row = lane / CPR;
  const bool vec = N % PV == 0;
#pragma unroll
  for (int m = 0; m < MS; ++m) {
    const int col0 = n0 + 32 * wave;
    const int bc = col0 + ln < N ? col0 + ln : N - 1;
    const float lb = a.bias ? as_f32(static_cast<const T *>(a.bias)[bc]) : 0.f;
    auto put = [&](int r, float v) __attribute__((always_inline)) {
      T o = rounded<T>(v);
      if (a.bias) o = rounded<T>(as_f32(o) + lb);
      reinterpret_cast<T *>(mine + (8 * (r >> 2) + 4 * kb + (r & 3)) * ROWB)[ln] = o;
    };
    uint32_t again = 0;  // (bits: which of the sixteen sums are not finite)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      put(r, tot[m][0][r]);
      again |= (not_finite(tot[m][0][r]) ? 1u : 0u) << r;
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
      plain_rows<BITS, 4, T>(xs, row_order(BITS), a.w0 + (int64_t)w_row[0] * (row_bytes / 4), static_cast<const T *>(a.s0) + (int64_t)w_row[0] * G,
                             static_cast<const T *>(a.b0) + (int64_t)w_row[0] * G, K, K / G, open, v);
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (open >> i & 1u) put(4 * quad + i, v[i]);
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    const int my_col = col0 + PV * my_piece;
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

template <int DT, int BITS, bool G32, int MS, int WN, int KW>
static hipError_t start_codes(const CodesArgs &a, int scale_shift, hipStream_t st) {
  constexpr int NI = 32 * WN, BM = 32 * MS;
  constexpr size_t bufs = (size_t)2 * KW * BM * kRow * 16 + WN * KW * 32 * 48, sums = KW > 1 ? (size_t)BM * 32 * WN * 4 : 0;
  constexpr size_t most = bufs > sums ? bufs : sums, lds = most > kLdsAtLeast ? most : kLdsAtLeast;
  static_assert(lds <= 160 * 1024, "more LDS than a CU has");
  const int n_ntiles = (a.N + NI - 1) / NI, mtiles = (int)((a.M + BM - 1) / BM);
  const int64_t grid = (int64_t)((n_ntiles + 7) / 8) * 8 * mtiles;
  if (grid <= 0 || grid > INT32_MAX) return hipErrorInvalidValue;
  const auto kernel = &qmm_codes_kernel<DT, BITS, G32, MS, WN, KW>;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> allowed{0};
    if (hipError_t e = allow_lds(reinterpret_cast<const void *>(kernel), (int)lds, allowed); e != hipSuccess) return e;
  }
  kernel<<<(unsigned)grid, 64 * WN * KW, lds, st>>>(a, mtiles, n_ntiles, scale_shift);
  return hipGetLastError();
}

hipError_t launch_qmm_codes_small(const CodesArgs &a, hipStream_t st) { return start_codes<0, 8, true, 1, 2, 4>(a, 0, st); }

hipError_t launch_qmm_codes_middle(const CodesArgs &a, bool share, int group, int bits, int dt, hipStream_t st) {
  auto with_group = [&](auto d, auto b) {
    constexpr int DT = decltype(d)::value, BITS = decltype(b)::value;
    if (group == 32) return share ? start_codes<DT, BITS, true, 2, 4, 2>(a, 0, st) : start_codes<DT, BITS, true, 2, 4, 1>(a, 0, st);
    return share ? start_codes<DT, BITS, false, 2, 4, 2>(a, group == 128, st) : start_codes<DT, BITS, false, 2, 4, 1>(a, group == 128, st);
  };
  auto with_bits = [&](auto d) {
    return bits == 4 ? with_group(d, std::integral_constant<int, 4>{}) : with_group(d, std::integral_constant<int, 8>{});
  };
  if (dt == 0) return with_bits(std::integral_constant<int, 0>{});
  if (dt == 1) return with_bits(std::integral_constant<int, 1>{});
  return hipErrorInvalidValue;
}

}  // namespace mi_moe
