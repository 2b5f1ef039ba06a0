// Which tile a dense product on raw codes takes, and how it shares K among the waves of a block: arithmetic alone, for host and device code.
#pragma once
#include <cstdint>

namespace mi_moe {

// K values of each of n shares: even, in whole 128s or (pairs) 256s.
constexpr int share_of_k(int K, int n, bool pairs) {
  const int even = (K / 128 + n - 1) / n;
  return (pairs ? (even + 1) & ~1 : even) * 128;
}

// Tiles (rows x cols) of the fullest XCD: it takes every eighth column of tiles, with all its rows, for 32 CUs.  A launch is as long as that one's:
// 12 x 18 tiles are fewer than 256, but two XCDs get 36 of them and run two rounds where a CU holds one block.
constexpr int64_t tiles_of_an_xcd(int64_t M, int N, int rows, int cols) {
  return (int64_t)(((N + cols - 1) / cols + 7) / 8) * ((M + rows - 1) / rows);
}

// The tiles (token rows x weight rows) and the groups of waves that share K.
enum class DenseTile {
  k32x64,            // four groups (qmm_tiles.hip): one block a CU with 4-bit codes, two with 8-bit ones
  kRegisters32x64,   // four groups, codes loaded into registers (qmm_codes.hip), bf16 and 8-bit codes in groups of 32: one block
  k32x128,           // four groups, 4-bit: one block
  k64x256,           // two groups, one block (4-bit); one group, two blocks (8-bit)
  kRegisters64x128,  // codes in registers, one group: several blocks
  kRegisters64x128Shared,  // two groups: one block
};

// Measured, us of the kernels from graph replays, with the tiles of the fullest XCD (x of 64 x 128 unless another is named):
//   4-bit, K shared by four in 32 x 128 against registers: f16, 567 x 1280 x 3840, 36 of 32 x 128, 42.9 / 32.8; bf16 367 x 2304 x 2944, 36,
//     38.9 / 28.7; bf16 414 x 1760 x 2944, 26, 24.1 / 28.5; f16 483 x 1664 x 3456 in groups of 32, 32, 31.0 / 36.6.  32 x 64 / 32 x 128: bf16
//     221 x 2080 x 1408, 35 of 32 x 64, 20.1 / 16.2.
//   4-bit, 64 x 256 against registers, one round of 64 x 256 (x = 52 to 64): K = 1024 25.0 / 21.9 (f16), 1408 29.4 / 27.9, 2560 42.1 / 40.0, 3072
//     43.7 / 45.6 and 46.0 / 46.2, 4096 55.1 / 58.9 and 51.0 / 54.5; in groups of 32 2560 48.8 / 46.5, 3584 58.5 / 59.5, 4096 66.0 / 68.0;
//     two rounds: 1535 x 3504 x 2688 (x = 96) 75.6 / 60.8, 1874 x 2576 x 4096 (90) 104 / 80.8, 1580 x 3968 x 3584 in groups of 128 (100) 83.7 / 87.1,
//     1692 x 3504 x 4096 in groups of 32 (108) 119 / 126; more, in which registers' blocks, several on a CU, fill the gaps: 2345 x 3952 x 3584
//     (148, three) 138 / 125, 3423 x 3264 x 3968 in groups of 128 (216, four) 189 / 160, 3784 x 3520 x 4096 (240, four) 195 / 206.
//   8-bit, 32 x 64 against registers by its own tiles of an XCD: 50 20.5 / 23.4, 55 22.7 / 25.4, 64 27.4 / 33.1; 66 20.4 / 17.8, 70 23.4 / 19.6, 80
//     21.9 / 18.0.
//   8-bit, 64 x 256 against registers, with the most blocks of it on a CU, two at a time: 3872 x 1888 x 2688 (x = 122, two) 77.9 / 86.2, 3336 x 1424 x 1024
//     (106, two) 32.7 / 36.3, 2706 x 3552 x 2560 in groups of 128 (172, three) 94.5 / 107, 3126 x 3456 x 2176 (196, four) 107 / 112, 2738 x 1488 x 3712
//     (86, two) 84.2 / 77.0, 2544 x 2272 x 4096 (120, three) 142 / 111; in groups of 32 3146 x 1712 x 3840 (100, two) 114 / 127, 3683 x 4000 x 3328
//     (232, four) 208 / 225, 1993 x 2928 x 2944 (96, two) 98.3 / 84.3, 3498 x 4080 x 1024 (220, four) 82.0 / 74.4.
//   8-bit, groups of 32, bf16, 32 x 64 against registers: K = 1024 10.8 / 11.7, 1152 12.2 / 12.3, 1408 12.8 / 12.7, 2560 16.7 / 16.0, 3328 20.3 / 19.0, 4096 22.8 / 21.3
//     (stages of 64 K values hold two groups, each with a scaling of its sums and a conversion to float of every code; registers take 128 K
//     values between two barriers); f16, whose codes need no conversion, 12.0 / 12.4 at K = 1408, 19.7 / 19.6 at 3712.
//   Registers, K shared by two / by one: f16 8-bit 743 x 2672 x 3072 (x = 36) 52.2 / 38.8; bf16 4-bit 998 x 1168 x 3840 (32) 36.2 / 38.7.
constexpr DenseTile dense_tile(int64_t M, int N, int K, int bits, int group, bool bf16) {
  const int64_t x = tiles_of_an_xcd(M, N, 64, 128), wide = tiles_of_an_xcd(M, N, 64, 256);
  const int64_t least = tiles_of_an_xcd(M, N, 32, 64);
  if (bf16 && bits == 8 && group == 32 && K >= 1280 && least <= 32) return DenseTile::kRegisters32x64;
  if (least <= (bits == 4 ? 32 : 64)) return DenseTile::k32x64;
  if (bits == 4) {
    if (tiles_of_an_xcd(M, N, 32, 128) <= 32) return DenseTile::k32x128;
    const int64_t rounds = (wide + 31) / 32;
    if (K >= (group == 32 || rounds > 2 ? 3584 : rounds == 2 ? 3328 : 3072) && x >= (rounds <= 2 ? 50 : 60) * rounds) return DenseTile::k64x256;
  } else {
    const int64_t blocks = (wide + 31) / 32;
    if (blocks >= 2 && x >= 49 * blocks && (group != 32 || K >= 1536)) return DenseTile::k64x256;
  }
  return x <= 32 ? DenseTile::kRegisters64x128Shared : DenseTile::kRegisters64x128;
}

// Tiles of 96 or 128 token rows x 128 weight rows, K shared by two groups of waves, one block a CU (qmm_tiles.hip): where they fill the chip in one round and
// tiles of 64 x 128 would give some CUs two blocks and others one.  0: dense_tile's.  Measured, us of the call, dense_tile's / these (84 shapes of 96 rows with
// 4-bit codes, 64 with 8-bit ones, 1.00 to 1.33 times as fast, longer K more):
//   96 rows   bf16 4-bit 640 x 4096 x 4096 53.2 / 41.1, 650 x 2864 x 1152 22.1 / 20.8, 902 x 2288 x 3584 49.1 / 39.2, in groups of 32 926 x 2928 x 3584 58.6 / 48.0,
//             542 x 3248 x 1152 24.9 / 24.1, of 128 549 x 3888 x 3840 48.6 / 36.6; f16 8-bit 868 x 2944 x 2688 35.7 / 30.9, in groups of 32 718 x 4016 x 1152
//             23.3 / 23.5, of 128 562 x 3760 x 3456 40.7 / 32.8
//   128 rows  8-bit: K = 3072 43.8 / 42.5, 40.0 / 36.8, 44.3 / 42.0 (128), 55.1 / 51.9 (32), 3328 44.2 / 41.5, 4096 51.1 / 46.3, 62.0 / 59.3 (32); below
//             that 1664 26.8 / 27.3, 2688 38.7 / 38.3, 43.3 / 45.3 (32), 1152 21.2 / 22.1, 1280 24.2 / 27.2 (32).  4-bit: two groups' stages are more LDS than a CU has
constexpr int long_tile_rows(int64_t M, int N, int K, int bits) {
  if (K < 1024 || tiles_of_an_xcd(M, N, 64, 128) <= 32) return 0;
  if (tiles_of_an_xcd(M, N, 96, 128) <= 32) return 96;
  return bits == 8 && K >= 3072 && tiles_of_an_xcd(M, N, 128, 128) <= 32 ? 128 : 0;
}

// Dense float32 rows: tiles on the float32 matrix instructions (qmm_f32.hip), or the plain kernel (quantize.hip).  A launch of tiles takes as long as the fullest XCD's rounds, whatever share of
// a round there is: at K = 4096 28 us for one of 32 x 32, 47 of 64 x 32, 86 a round of 64 x 64.  The plain kernel's time is that of its blocks, of 8 rows (4 with 8-bit codes) x 16
// columns here: up to 1024 of them run at once in 20 to 30 us, 2048 take 49 to 60, then 0.024 us each and, where rows are no multiple of 1024 values (K = 4096 apart), a third more; with
// 8-bit codes 0.017.  The lines lie where the two meet: of 2000 shapes and group sizes (64 to 9000 rows, 16 to 4096 columns, K = 1024 to 16384) the tiles take 900, and are slower than the plain
// kernel in three, by 2 %.  Us, plain / tiles, 4-bit unless named:
//   tiles  64 / 250 / 1000 x 3072 x 3072 38.9, 112, 561 / 22.1, 67.5, 197; 96 x 1536 x 2048 20 / 16; 192 x 1024 x 4096 42 / 28; 700 x 256 x 8192 81 / 55; 116 x 1176 x 3712 40 / 25; 700 x 1024 x 4096
//          132 / 86; 8-bit 64 / 1000 x 4096 x 4096 74, 1082 / 28, 335; 96 x 1024 x 4096 32 / 28; 1000 x 128 x 2048 20 / 16
//   plain  64 x 256 x 16384 20 / 105; 72 x 256 x 8192 17 / 53; 64 x 1024 x 4096 18 / 28; 2228 x 104 x 5632 90 / 226; 2510 x 136 x 1280 39 / 60; 400 x 64 x 8192 21 / 54; 8-bit 72 x 512 x 8192 32 / 53
//   fewer rows, which keep a row's sums whatever their number: 24 / 32 / 48 x 3072 x 3072 22, 22, 37 / 25, 26, 27
// Shorter K keeps the plain sums for their error: at K = 384 and 8-bit codes the plain kernel's 64 sums of six values lose 3 % less.
constexpr bool float32_tiles(int64_t rows, int N, int K, int bits) {
  if (rows < 64 || K < 1024) return false;
  const int64_t plain = (bits == 4 ? (rows + 7) / 8 : (rows + 3) / 4) * ((N + 15) / 16), rounds = (tiles_of_an_xcd(rows, N, 64, 64) + 31) / 32;
  const int size = tiles_of_an_xcd(rows, N, 32, 32) <= 32 ? 0 : tiles_of_an_xcd(rows, N, 64, 32) <= 32 ? 1 : 2;
  if (bits == 8) return plain > (size == 0 ? 1350 : size == 1 ? 2500 : 5300 * rounds);
  return K % 1024 == 0 ? plain > (size == 0 ? 1024 : size == 1 ? 1700 : 3600 * rounds) : plain > (size == 0 ? 900 : size == 1 ? 1550 : 2750 * rounds);
}

}  // namespace mi_moe
