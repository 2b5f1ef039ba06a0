// Tiled quantized product over weights that are packed along the output columns: y [M, N] = x [M, K] w [K, N], each row
// of w quantised along N.  This is the gradient of a quantized linear layer with respect to its input.
//
// Contract: mlx_quantized_matmul with transpose = false (mlx-rs/src/ops/quantization.rs:91-122).
//
// Arithmetic: a group has a scale of its own for every k, so nothing can be taken out of the sum; the weights are
// dequantised, w = fma(s, q, b) in fp32, and enter the matrix cores in pieces (each the rounded rest of the ones before
// it), as do f32 rows of x:
//   bf16  x as it is, w in two pieces: 2 products
//   f16   x as it is, 2^10 w in two f16 pieces (the factor keeps every piece clear of the smallest numbers: w is a multiple of 2^-24,
//         and leaves |w| < 64 without an overflow): 2 products
//   f32   x in three pieces (exact), w in three (exact): the 6 products down to 2^-18 of the first
// Two pieces hold 17 bits (f16: 23), which is all of w unless its bias is some 2^9 (f16: 2^12) times its scale or more; groups whose values
// have both signs keep it below 2^4 (4-bit codes) and 2^8 (8-bit).  A wave that met such a scale goes over its K once more, for the
// third pieces (another step inside the loop would spill): the weights are those of the plain product in every case.
// A result that is not finite is computed again the plain way, one fma per k: pieces of an infinity are no numbers, and
// where nothing but a piece has overflowed that gives the number.  That is a lane's own chain over K, for eight results at a time.
// us of the call with finite rows / one infinity in one row / one in each (before the weights left LDS): 1000 x 2048 x 4096 bf16 48 / 425 / 960 (a thread per packed word 1360;
// one result at a time 50 / 1620 / 11700); 20 rows f16 20 / 256 / 270, weights beyond 64 270 (4120).
#include <type_traits>

#include "dense_rule.hpp"
#include "lds_copies.hpp"
#include "qmm_dev.hpp"

namespace mi_moe {

namespace {

constexpr int kStep = 32;                   // K values per step
constexpr uint32_t kOutside = 0x80000000u;  // an offset past every descriptor here: such a load returns zeros

constexpr int pieces_of_x(int dt) { return dt == 2 ? 3 : 1; }
constexpr int pieces_of_w(int dt) { return dt == 2 ? 3 : 2; }
constexpr float factor_of_w(int dt) { return dt == 1 ? 1024.0f : 1.0f; }

// the pieces of two values, P registers: the first piece of both, the next one of what it left, ...
template <int DT, int P>
__device__ __forceinline__ void split_pair(float v0, float v1, uint32_t (&to)[P]) {
#pragma unroll
  for (int p = 0; p < P; ++p) {
    if constexpr (DT == 1) {
      const half2_t h = __builtin_convertvector(f32x2_t{v0, v1}, half2_t);
      to[p] = __builtin_bit_cast(uint32_t, h);
      v0 -= (float)h.x;
      v1 -= (float)h.y;
    } else {
      to[p] = cvt_pk_bf16(v0, v1);
      v0 -= bf16lo_to_f32(to[p]);
      v1 -= bf16hi_to_f32(to[p]);
    }
  }
}

// LDS of a wave: x [pieces, or two steps in turn][32 MS rows][32 K values], (s, b) of 32 K values of two groups.  A row is four 16-byte chunks; chunk c of row r sits at c ^ (r / 4 % 4), so that the 16 lanes of one LDS
// cycle, which read one chunk of 16 rows or write four chunks of four, meet 16 different places.
constexpr int kRowPieces = 4;
__device__ __forceinline__ int at(int row, int chunk) { return row * kRowPieces + (chunk ^ ((row >> 2) & 3)); }
constexpr int kScaleRow = 32 * 8 + 16;  // bytes of one group's (s, b) pairs
constexpr bool rows_copied(int dt, int nt) { return dt != 2 && nt == 2; }
constexpr int wave_lds(int dt, int ms, int nt) {
  return (rows_copied(dt, nt) ? 2 : pieces_of_x(dt)) * ms * 32 * kRowPieces * 16 + 2 * kScaleRow;
}

}  // namespace

// A block computes 32 MS rows x 32 NT columns; its KW waves share K among them, each on LDS of its own, and meet only to
// add their sums: no wave waits for another in the loop, so the unpacking of one runs beside the multiplies of the other
// on its SIMD.  A lane unpacks eight K values of 2 NT consecutive columns (a byte to a word of eight rows): the eight
// values of a column are then one 16-byte chunk of a weight operand.  Sixteen lanes hold an octet of K values, a multiply takes octets 2 h and 2 h + 1, and
// an exchange of sixteen lanes between two columns' registers (v_permlane16_swap) brings each where it is multiplied: the weights never
// pass through LDS.  The columns are dealt to the sub-tiles so that a lane ends up with NT
// consecutive ones: column n = 2 NT u + j goes to place 16 (j % NT * 2 + j / NT) + u, that is
// sub-tile j % NT, lane 16 (j / NT) + u.
// What bounds it (128 x 64 tiles, bf16): a step of a wave is 1024 cycles of matrix work (two products) beside about 800 of
// unpacking and 16 KB of rows through LDS.  1000 x 2048 x 4096, 4-bit, groups of 64: 41.5 us for the call, 400 TFLOP/s of the product
// (weights through LDS as well, rows by way of registers 46.5, of which unpacking was 6, the second product 7, the rows' LDS traffic 9).  Unpacking the next step between the multiplies of this one: 41.5 too.
// 1 row 17.8 us (19.1), f32 118 (124).
// Error: share of results that are not the float64 product's nearest value, here / a thread per packed word: 300 x 2048 x 2048 bf16 1.1e-4
// to 2.2e-4 / 1.8e-4 to 5.4e-4, f16 1.2e-3 / 3.6e-3; groups at 1 + q / 2^13 and rows that sum to zero, bf16, 3e-3 to 1.1e-2 / 1.4e-3 to
// 3.2e-3 (two pieces alone: 0.11 to 0.14); f32 against 64 bits 4.9e-7 / 1.07e-6.  What looking at the scales cost: 1 us of 47.
template <int DT, int BITS, int MS, int NT, int KW>
__global__ __launch_bounds__(64 * KW) void qmm_cols_kernel(ColsArgs a, int n_mtiles, int n_ntiles, int group_log2) {
  typedef typename ElemOf<DT>::type T;
  typedef typename std::conditional<BITS * NT == 4, uint8_t, typename std::conditional<BITS * NT == 16, uint32_t, uint16_t>::type>::type Codes;
  constexpr int PX = pieces_of_x(DT), PW = pieces_of_w(DT);
  constexpr float kFactor = factor_of_w(DT);
  constexpr bool kCopied = rows_copied(DT, NT);
  constexpr int CN = 2 * NT;          // columns a lane unpacks
  constexpr int NX = 2 * MS;          // 16-row pieces of the token rows
  constexpr int XP = DT == 2 ? 2 : 1; // 16-byte pieces of eight values of x
  constexpr int X_SZ = 32 * MS * kRowPieces;
  static_assert(sizeof(Codes) * 8 == BITS * CN, "a lane's columns of one row are one load");

  // block -> tile.  Ids are dealt round-robin over the 8 XCDs: an XCD takes every eighth column tile and all row tiles
  // of it, so its L2 holds those weights.
  const int xcd = blockIdx.x & 7, j = blockIdx.x >> 3;
  const int nt = j / n_mtiles * 8 + xcd;
  if (nt >= n_ntiles) return;
  const int64_t row0 = (int64_t)(j % n_mtiles) * (32 * MS);
  const int rows = a.M - row0 < 32 * MS ? (int)(a.M - row0) : 32 * MS;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int N = a.N, K = a.K, n0 = nt * (32 * NT);
  const int row_bytes = N / 8 * BITS, G = N >> group_log2;

  extern __shared__ __align__(16) unsigned char lds_raw[];
  u32x4_t *const Xs = reinterpret_cast<u32x4_t *>(lds_raw + wave * wave_lds(DT, MS, NT));
  unsigned char *const Ss = reinterpret_cast<unsigned char *>(Xs + (kCopied ? 2 : PX) * X_SZ);

  // ---- this lane's share of a step: rows xrow + 16 i and chunk oct of x; columns CN u .. and rows 8 oct .. of the codes;
  // row lane % 32 of the scales and biases, of the tile's first (lane / 32 = 0) or second 32 columns
  const int xrow = lane >> 2, xoct = lane & 3;
  const int u = lane & 15, oct = (lane >> 4 & 1) * 2 + (lane >> 5);
  int wcol = n0 + CN * u;
  wcol = wcol < N ? wcol : N - CN;  // columns past the end repeat the last ones (never stored)
  const int skl = lane & 31;
  int sgroup = (n0 + 32 * (lane >> 5)) >> group_log2;
  sgroup = sgroup < G ? sgroup : G - 1;
  const T *const sp = static_cast<const T *>(a.s), *const bp = static_cast<const T *>(a.b);

  const uint32_t x_at = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) unsigned char *)lds_raw + (uint32_t)(wave * wave_lds(DT, MS, NT));
  // Rows of the tiles of 64 columns are copied straight into LDS, a step ahead of the one that is multiplied, whose multiplies cover the copies; narrower
  // tiles' do not (32 x 32 tiles, one row x 2048 x 4096 17.8 us, copied 27.0), and f32 rows are split on the way.
  auto copy_rows = [&](int ks, int place) __attribute__((always_inline)) {
    const int k = ks * kStep;
    const i32x4_t from = words_of(static_cast<const T *>(a.x) + row0 * K + k, ((uint32_t)rows * K - k) * (uint32_t)sizeof(T));
#pragma unroll
    for (int i = 0; i < NX; ++i) {
      const int row = xrow + 16 * i, chunk = xoct ^ (row >> 2 & 3);
      copy_to_lds(from, k + 8 * chunk < K ? (row * (uint32_t)K + 8 * chunk) * (uint32_t)sizeof(T) : kOutside, 0, x_at + place * (X_SZ * 16) + i * 1024);
    }
  };
  struct Stage {
    u32x4_t x[kCopied ? 1 : NX][XP];
    uint32_t q[8];
    T s, b;
  };
  auto load = [&](int ks, Stage &R) __attribute__((always_inline)) {
    const int k = ks * kStep;
    // rows past the end are past the descriptor, K values past the end are sent there: both read zeros
    if constexpr (!kCopied) {
      const __amdgpu_buffer_rsrc_t xr = rsrc_of(static_cast<const T *>(a.x) + row0 * K + k, ((uint32_t)rows * K - k) * (uint32_t)sizeof(T));
#pragma unroll
      for (int i = 0; i < NX; ++i)
#pragma unroll
        for (int p = 0; p < XP; ++p) {
          const uint32_t off = ((xrow + 16 * i) * (uint32_t)K + 8 * xoct) * (uint32_t)sizeof(T) + 16 * p;
          R.x[i][p] = __builtin_amdgcn_raw_buffer_load_b128(xr, k + 8 * xoct < K ? off : kOutside, 0, 0);
        }
    }
    const int left = K - k < kStep ? K - k : kStep;  // rows past the end read zeros, with a scale and a bias of zero
    const __amdgpu_buffer_rsrc_t wr = rsrc_of(reinterpret_cast<const unsigned char *>(a.w) + (int64_t)k * row_bytes, (uint32_t)left * row_bytes);
#pragma unroll
    for (int r = 0; r < 8; ++r) {
      const uint32_t off = (uint32_t)(8 * oct + r) * row_bytes + wcol * BITS / 8;
      if constexpr (sizeof(Codes) == 1) R.q[r] = __builtin_amdgcn_raw_buffer_load_b8(wr, off, 0, 0);
      else if constexpr (sizeof(Codes) == 2) R.q[r] = __builtin_amdgcn_raw_buffer_load_b16(wr, off, 0, 0);
      else R.q[r] = __builtin_amdgcn_raw_buffer_load_b32(wr, off, 0, 0);
    }
    const bool on = skl < left;
    const int64_t sat = (int64_t)(k + (on ? skl : 0)) * G + sgroup;
    const T s = sp[sat], b = bp[sat];
    R.s = on ? s : T{};
    R.b = on ? b : T{};
  };
  auto wave_fence = [&]() __attribute__((always_inline)) {  // LDS serves a wave in order: this pins the program's order
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
  };
  // By how many powers of two a bias is ahead of its scale, at most and at least, in the exponent's place.  Weights have two pieces'
  // bits, from the leading one of the largest value (at most 2 max(|b|, 2^BITS |s|)) down to the last one of scale or bias, while
  // that is at most kBits and at least BITS - kBits.
  constexpr int kBits = DT == 1 ? 11 : 8;  // of s, b and a piece
  int most = 0, least = 0;
  auto see_scale = [&](const Stage &R) __attribute__((always_inline)) {
    const uint32_t s = __float_as_uint(as_f32(R.s)), b = __float_as_uint(as_f32(R.b));
    const int ahead = (int)(b & 0x7f800000u) - (int)(s & 0x7f800000u);
    most = ahead > most ? ahead : most;
    least = b << 1 != 0u && ahead < least ? ahead : least;
  };
  u32x4_t op[2][NT][PW];  // the weights of a step as operands of its two multiplies
  // rows, and pieces FIRST .. FIRST + COUNT - 1 of the weights
  auto put = [&](const Stage &R, auto first, auto count) __attribute__((always_inline)) {
    constexpr int FIRST = decltype(first)::value, COUNT = decltype(count)::value;
    *reinterpret_cast<float2 *>(Ss + (lane >> 5) * kScaleRow + skl * 8) = make_float2(kFactor * as_f32(R.s), kFactor * as_f32(R.b));
    if constexpr (!kCopied) {
#pragma unroll
      for (int i = 0; i < NX; ++i) {
        u32x4_t *const to = Xs + at(xrow + 16 * i, xoct);
        if constexpr (DT != 2) {
          *to = R.x[i][0];
        } else {
          u32x4_t o[PX];
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            uint32_t pc[PX];
            split_pair<DT, PX>(__uint_as_float(R.x[i][c >> 1][2 * (c & 1)]), __uint_as_float(R.x[i][c >> 1][2 * (c & 1) + 1]), pc);
#pragma unroll
            for (int p = 0; p < PX; ++p) o[p][c] = pc[p];
          }
#pragma unroll
          for (int p = 0; p < PX; ++p) to[p * X_SZ] = o[p];
        }
      }
    }
    wave_fence();
    const float4 *const pairs = reinterpret_cast<const float4 *>(Ss + (CN * u / 32) * kScaleRow + oct * 64);
    u32x4_t o[CN][COUNT];
#pragma unroll
    for (int r = 0; r < 4; ++r) {  // two rows
      const float4 sb = pairs[r];
      const uint32_t q0 = R.q[2 * r], q1 = R.q[2 * r + 1];
#pragma unroll
      for (int c = 0; c < CN; ++c) {
        const float v0 = __builtin_fmaf(sb.x, (float)((q0 >> (BITS * c)) & ((1u << BITS) - 1u)), sb.y);
        const float v1 = __builtin_fmaf(sb.z, (float)((q1 >> (BITS * c)) & ((1u << BITS) - 1u)), sb.w);
        uint32_t pc[FIRST + COUNT];
        split_pair<DT, FIRST + COUNT>(v0, v1, pc);
#pragma unroll
        for (int p = 0; p < COUNT; ++p) o[c][p][r] = pc[FIRST + p];
      }
    }
    // columns t and NT + t of the lanes of octets 0 and 2 (1 and 3): an exchange of sixteen lanes leaves each octet in the half that multiplies it
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int p = 0; p < COUNT; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const auto v = __builtin_amdgcn_permlane16_swap(o[t][p][r], o[NT + t][p][r], false, false);
          op[0][t][p][r] = v[0];
          op[1][t][p][r] = v[1];
        }
  };

  f32x16_t tot[MS][NT];
#pragma unroll
  for (int m = 0; m < MS; ++m)
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int r = 0; r < 16; ++r) tot[m][t][r] = 0.f;
  const int ln = lane & 31, kb = lane >> 5;
  auto multiply = [&](auto pieces, int place) __attribute__((always_inline)) {
    constexpr int COUNT = decltype(pieces)::value;  // of the weights
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
      for (int m = 0; m < MS; ++m) {
        u32x4_t xv[PX];
#pragma unroll
        for (int p = 0; p < PX; ++p) xv[p] = Xs[(p + place) * X_SZ + at(32 * m + ln, 2 * h + kb)];
#pragma unroll
        for (int px = PX - 1; px >= 0; --px)
#pragma unroll
          for (int pw = COUNT - 1; pw >= 0; --pw)
            if (px + pw < PW)
#pragma unroll
              for (int t = 0; t < NT; ++t) tot[m][t] = mfma<DT>(xv[px], op[h][t][pw], tot[m][t]);
      }
    }
    wave_fence();
  };

  const int steps = (K + kStep - 1) / kStep, share = (steps + KW - 1) / KW;
  const int k0 = wave * share, k1 = k0 + share < steps ? k0 + share : steps;
  auto pass = [&](auto first, auto count) __attribute__((always_inline)) {
    Stage R;
    load(k0, R);
    if constexpr (kCopied) copy_rows(k0, 0);
    int place = 0;
    for (int ks = k0; ks < k1; ++ks) {
      if constexpr (kCopied) wait_copies<0>();  // this step's, asked for ahead of the multiplies before it
      if constexpr (DT != 2) see_scale(R);
      put(R, first, count);
      load(ks + 1 < k1 ? ks + 1 : ks, R);
      if constexpr (kCopied) copy_rows(ks + 1 < k1 ? ks + 1 : ks, place ^ 1);
      multiply(count, place);
      if constexpr (kCopied) place ^= 1;
    }
    if constexpr (kCopied) wait_copies<0>();
  };
  if (k0 < k1) {
    pass(std::integral_constant<int, 0>{}, std::integral_constant<int, PW>{});
    if constexpr (DT != 2)
      if (__ballot((most >> 23) > kBits || (least >> 23) < BITS - kBits)) pass(std::integral_constant<int, PW>{}, std::integral_constant<int, 1>{});
  }

  // ---- the waves' sums: the second half of the waves hands its sums to the first, whose sums every wave then adds for a
  // share of the rows, in a fixed order
  constexpr int HALF = KW / 2, PIECES = MS * NT * 4;
  float4 *const parts = reinterpret_cast<float4 *>(lds_raw);
  auto give = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          parts[((wave % HALF) * PIECES + (m * 4 + r) * NT + t) * 64 + lane] =
              make_float4(tot[m][t][4 * r], tot[m][t][4 * r + 1], tot[m][t][4 * r + 2], tot[m][t][4 * r + 3]);
  };
  __syncthreads();
  if (wave >= HALF) give();
  __syncthreads();
  if (wave < HALF) {
#pragma unroll
    for (int m = 0; m < MS; ++m)
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const float4 v = parts[(wave * PIECES + (m * 4 + r) * NT + t) * 64 + lane];
          tot[m][t][4 * r] += v.x;
          tot[m][t][4 * r + 1] += v.y;
          tot[m][t][4 * r + 2] += v.z;
          tot[m][t][4 * r + 3] += v.w;
        }
    give();  // (its own slot, which only this wave has read)
  }
  __syncthreads();

  const int col = n0 + CN * (ln & 15) + NT * (ln >> 4);
  for (int piece = wave; piece < MS * 4; piece += KW) {  // rows 32 (piece / 4) + 8 (piece % 4) + 4 kb + 0 .. 3
    float v[NT][4];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      float4 sum = parts[(piece * NT + t) * 64 + lane];
#pragma unroll
      for (int w = 1; w < HALF; ++w) {
        const float4 more = parts[(w * PIECES + piece * NT + t) * 64 + lane];
        sum.x += more.x;
        sum.y += more.y;
        sum.z += more.z;
        sum.w += more.w;
      }
      v[t][0] = sum.x;
      v[t][1] = sum.y;
      v[t][2] = sum.z;
      v[t][3] = sum.w;
    }
    if (col >= N) continue;
    const int r_first = 32 * (piece >> 2) + 8 * (piece & 3) + 4 * kb;
    uint32_t again = 0;  // (bits: which of the sums are not finite)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        v[t][r] *= 1.0f / kFactor;
        again |= (r_first + r < rows && not_finite(v[t][r]) ? 1u : 0u) << (r * NT + t);
      }
    if (__builtin_expect(again != 0, 0)) {  // all of the lane's sums in one pass over K, eight values at a time: it costs the latency of their loads
      float f[4][NT] = {};
      uint32_t open = again;
      for (int k = 0; k < K && open; k += 8) {  // (no number stays none)
        T xv[4][8], sv[8], bv[8];
        uint32_t word[8];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = r_first + r < rows ? r_first + r : rows - 1;
          __builtin_memcpy(xv[r], __builtin_assume_aligned(static_cast<const T *>(a.x) + (row0 + row) * K + k, 16), sizeof xv[r]);
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int64_t g = (int64_t)(k + i) * G + (col >> group_log2);
          word[i] = a.w[(int64_t)(k + i) * (row_bytes / 4) + col * BITS / 32] >> (col * BITS % 32);  // (a lane's columns lie in one word)
          sv[i] = sp[g];
          bv[i] = bp[g];
        }
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
          for (int t = 0; t < NT; ++t) {
            const float wv = __builtin_fmaf(as_f32(sv[i]), (float)((word[i] >> (BITS * t)) & ((1u << BITS) - 1u)), as_f32(bv[i]));
#pragma unroll
            for (int r = 0; r < 4; ++r) f[r][t] = __builtin_fmaf(as_f32(xv[r][i]), wv, f[r][t]);
          }
#pragma unroll
        for (int i = 0; i < 4 * NT; ++i)
          if (f[i / NT][i % NT] != f[i / NT][i % NT]) open &= ~(1u << i);
      }
#pragma unroll
      for (int i = 0; i < 4 * NT; ++i)
        if (again >> i & 1u) v[i % NT][i / NT] = f[i / NT][i % NT];
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      if (r_first + r >= rows) continue;
      T o[NT];
#pragma unroll
      for (int t = 0; t < NT; ++t) o[t] = rounded<T>(v[t][r]);
      T *const to = static_cast<T *>(a.y) + (row0 + r_first + r) * N + col;
      __builtin_memcpy(__builtin_assume_aligned(to, NT * sizeof(T)), o, sizeof o);
    }
  }
}

template <int DT, int BITS, int MS, int NT, int KW>
static hipError_t start_cols(const ColsArgs &a, int group_log2, hipStream_t st) {
  constexpr int loop = KW * wave_lds(DT, MS, NT), sums = KW / 2 * MS * NT * 32 * 32 * 4, lds = loop > sums ? loop : sums;
  static_assert(lds <= 160 * 1024, "more LDS than a CU has");
  const int n_ntiles = (a.N + 32 * NT - 1) / (32 * NT);
  const int64_t mtiles = (a.M + 32 * MS - 1) / (32 * MS), grid = (int64_t)((n_ntiles + 7) / 8) * 8 * mtiles;
  if (grid > INT32_MAX) return hipErrorInvalidValue;
  const auto kernel = &qmm_cols_kernel<DT, BITS, MS, NT, KW>;
  if (lds > 64 * 1024)
    if (hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, lds);
        e != hipSuccess)
      return e;
  kernel<<<(unsigned)grid, 64 * KW, lds, st>>>(a, (int)mtiles, n_ntiles, group_log2);
  return hipGetLastError();
}

// Whole 16-byte pieces of x, offsets that fit their 32 bits, no 2-bit codes; every other shape stays with the plain kernel.
bool qmm_cols_applies(const ColsArgs &a, int bits, int dt) {
  const int64_t elem = dt == 2 ? 4 : 2, most = (int64_t)1 << 31;
  return bits != 2 && a.K % 8 == 0 && 128 * (int64_t)a.K * elem < most && 32 * (int64_t)a.N * bits / 8 < most && a.N % 32 == 0;
}

// Which tile: the smallest one of which the fullest XCD gets at most one a CU; a CU's time is that of its unpacking and
// multiplies, so a second tile on some CUs costs a whole further round (700 x 1408 x 2944: 242 tiles of 64 x 64, but 33 on some XCDs, 39.2 us, of 128 x 64
// 24.3; 48 shapes at that line 1.14 to 1.45 times as fast as with 256 tiles counted).  Measured, 4-bit, groups of 64, bf16, N = 2048,
// K = 4096, us of the call with 32 x 32 / 64 x 32 / 64 x 64 / 128 x 64 tiles at 64 / 130 / 300 / 1000 rows, before the weights went through no LDS:
// 21.0, 26.2, 28.4, 37.0 / 32.2, 21.6, 29.4, 38.0 / 47.9, 40.8, 31.3, 39.8 / 136, 86.7, 65.9, 46.3 (f16 the same to 5 %).
// f32 holds three times the rows in LDS and multiplies three times as much: at 64 / 130 / 300 / 1000 rows 27.8, 38.5,
// 80.2, 118 / 54.2, 40.7, 88.0, 121 / 85.2, 78.0, 91.0, 121 / 249, 174, 196, 141, so 64 x 32 for two rounds of the chip (counted by XCD: 259 x 3200 x 4096
// 113.6 for 104.8), and 128 x 64 beyond (K shared by four waves there: what LDS holds).
template <int DT, int BITS>
static hipError_t pick_cols(const ColsArgs &a, int group_log2, hipStream_t st) {
  auto fits = [&](int ms, int nt) { return tiles_of_an_xcd(a.M, a.N, 32 * ms, 32 * nt) <= 32; };
  if (fits(1, 1)) return start_cols<DT, BITS, 1, 1, 8>(a, group_log2, st);
  if constexpr (DT == 2) {
    if ((a.M + 63) / 64 * ((a.N + 31) / 32) <= 512) return start_cols<DT, BITS, 2, 1, 8>(a, group_log2, st);
  } else {
    if (fits(2, 1)) return start_cols<DT, BITS, 2, 1, 8>(a, group_log2, st);
    if (fits(2, 2)) return start_cols<DT, BITS, 2, 2, 8>(a, group_log2, st);
  }
  return start_cols<DT, BITS, 4, 2, DT == 2 ? 4 : 8>(a, group_log2, st);
}

hipError_t launch_qmm_cols(const ColsArgs &a, int group, int bits, int dt, hipStream_t st) {
  if (a.M == 0) return hipSuccess;
  const int gl = group == 32 ? 5 : (group == 64 ? 6 : 7);
  auto with_bits = [&](auto d) {
    constexpr int DT = decltype(d)::value;
    return bits == 4 ? pick_cols<DT, 4>(a, gl, st) : pick_cols<DT, 8>(a, gl, st);
  };
  if (dt == 0) return with_bits(std::integral_constant<int, 0>{});
  if (dt == 1) return with_bits(std::integral_constant<int, 1>{});
  return with_bits(std::integral_constant<int, 2>{});
}

}  // namespace mi_moe
