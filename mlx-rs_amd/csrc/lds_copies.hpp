// Copies from memory straight into LDS (qmm_tiles.hip, qmm_cols.hip).
#pragma once
#include "common.hpp"

namespace mi_moe {

// Written out because the compiler waits for every copy in flight ahead of any read of LDS; it knows nothing of these, and the
// kernel counts them itself.  (The compiler's own counts of loads in flight stay safe: with loads it does not know of in
// between it waits for more than it has to.)  A lane's 16 bytes go to LDS at `to` + 16 lane; what lies past the descriptor's end is zeros.
// The wait states are the instruction's own: a load must not follow a vector instruction that wrote one of its scalar registers (a
// spilled descriptor comes back through v_readlane) by less than five, which the compiler minds for the loads it knows.  They cost 0.3 to 2 % of a
// product (96 x 4096 x 4096 bf16 4-bit 17.8 us, 18.0 with them).
// Measured out of L2, bytes a cycle and CU: pieces of 64 consecutive bytes 31, of 128 and more 60; 32 bytes a row, as matrix operands
// loaded straight into registers are, 18.
typedef int32_t i32x4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ i32x4_t words_of(const void *base, uint32_t bytes) {
  const uint64_t p = reinterpret_cast<uint64_t>(base);
  return i32x4_t{(int32_t)(uint32_t)p, (int32_t)(uint32_t)(p >> 32), (int32_t)bytes, 0x00020000};
}
__device__ __forceinline__ void copy_to_lds(i32x4_t rsrc, uint32_t voff, uint32_t soff, uint32_t to) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds" ::"s"(to), "v"(voff), "s"(rsrc), "s"(soff) : "m0", "memory");
}
// The same by lanes 0 to 31, where all lanes are active: no branch, in which the compiler may hold a scalar operand in a vector register.
__device__ __forceinline__ void copy_half_to_lds(i32x4_t rsrc, uint32_t voff, uint32_t soff, uint32_t to) {
  asm volatile("s_mov_b32 exec_hi, 0\n\ts_mov_b32 m0, %0\n\ts_nop 3\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds\n\ts_mov_b32 exec_hi, -1" ::"s"(to), "v"(voff), "s"(rsrc), "s"(soff) : "m0", "memory");
}
template <int N>
__device__ __forceinline__ void wait_copies() {  // all but the last N have arrived; LDS reads are done
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ void wait_reads() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }  // of LDS, and writes to it
__device__ __forceinline__ void block_barrier() { asm volatile("s_barrier" ::: "memory"); }

}  // namespace mi_moe
