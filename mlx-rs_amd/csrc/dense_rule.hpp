// How a product on raw codes shares K among the waves of a block: arithmetic alone, for host and device code.
#pragma once
#include <cstdint>

namespace mi_moe {

// K values of each of n shares: even, in whole 128s or (pairs) 256s.
constexpr int share_of_k(int K, int n, bool pairs) {
  const int even = (K / 128 + n - 1) / n;
  return (pairs ? (even + 1) & ~1 : even) * 128;
}

}  // namespace mi_moe
