// What the 256 x 256 matrix tiles share: LDS-DMA and MFMA as inline asm.
#pragma once
#include "common.h"

namespace nga {

// 16 bytes a lane from base + off to lds + 16 lane, without an output, so that the kernel counts them itself: behind the builtin the
// compiler waits for all DMAs under way before each transpose read. m0 needs one cycle.
__device__ __forceinline__ void tile_dma(const uint16_t* base, uint32_t off, uint16_t* lds) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"((uint32_t)(uintptr_t)(lptr_t)lds), "v"(off), "s"(base)
               : "memory", "m0");
}

// acc += a b, the sums in accumulation registers throughout: with the builtin the compiler moves a good part of 256 of them to and
// fro in every round; with the builtin and sums pinned to those registers it does not, and the loop is slower by a fifth all the
// same (1,024 x 4,096 of K 28,672: 247 us, so 192). The wait covers operands that the instruction before has written.
__device__ __forceinline__ void tile_mfma(f32x4& acc, bf16x8 a, bf16x8 b) {
  asm("s_nop 1\n\tv_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// Before the first look at sums: behind the last product, and before anything that reads them, until its result is there
template <int A, int B>
__device__ __forceinline__ void tile_pin(f32x4 (&acc)[A][B]) {
#pragma unroll
  for (int i = 0; i < A; ++i)
#pragma unroll
    for (int j = 0; j < B; ++j) asm volatile("" : "+a"(acc[i][j]));
}
template <int A, int B>
__device__ __forceinline__ void tile_settle(f32x4 (&acc)[A][B]) {
  tile_pin(acc);
  asm volatile("s_nop 15\n\ts_nop 7" ::: "memory");
  tile_pin(acc);
}

}  // namespace nga
