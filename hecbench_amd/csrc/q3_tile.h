// What the tiled kernels of the batched 3-bit product share (q3_prefill.hip, q3_direct.hip): loads straight into LDS, the
// step's wait, and a quarter of a k-group's codes as matrix operands.
#pragma once

#include "q3_recipe.h"

namespace hq_q3 {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef float f4v __attribute__((ext_vector_type(4)));
typedef float f2v __attribute__((ext_vector_type(2)));
typedef uint32_t u4v __attribute__((ext_vector_type(4)));
typedef uint32_t u2v __attribute__((ext_vector_type(2)));

// 64 lanes x 16 bytes from base + voff (per lane) to LDS bytes lds .. lds + 1023.  Assembly, as the compiler would wait
// for every load in flight before the first LDS read behind one; the waits are the loop's own.
#pragma clang diagnostic push
#pragma clang diagnostic ignored "-Winline-asm"  // that m0 is the compiler's own is why it is listed
__device__ __forceinline__ void load_lds(uint32_t lds, uint32_t voff, const void* base) {
  lds = __builtin_amdgcn_readfirstlane(lds);  // wave-uniform, whatever registers the compiler computed it in
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds), "v"(voff), "s"(base) : "memory", "m0");
}
#pragma clang diagnostic pop
template <int N>
__device__ __forceinline__ void wait_loads_and_meet() {
  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(N) : "memory");
}

// Quarter J of one column's k-group: operand registers 4J .. 4J+3 of q3_recipe.h, eight of its 32 codes.
template <int J>
__device__ __forceinline__ u4v unpack_quarter(uint32_t w0, uint32_t w1, uint32_t w2) {
  u4v f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    constexpr int kOffsets[7] = {0, 4, 10, 32, 41, 64, 71};
    const int off = kOffsets[kRecipe[4 * J + i].window];
    const uint32_t win = off == 0 ? w0 : off == 32 ? w1 : off == 64 ? w2 : off == 71 ? w2 >> 7
                         : off < 32 ? __builtin_amdgcn_alignbit(w1, w0, off) : __builtin_amdgcn_alignbit(w2, w1, off - 32);
    f[i] = win & mask_of(4 * J + i);
  }
  return f;
}

}  // namespace hq_q3
