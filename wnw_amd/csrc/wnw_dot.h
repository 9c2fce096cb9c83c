// Row dot products on matrix instructions, for scores that rank tokens by
// softmax weights: no less exact than short chains of scalar multiply-adds.
#pragma once

#include <type_traits>

#include "wnw_common.h"

namespace wnw {

// 16 rows x 16 heads of q . K: A = the rows' 16-byte chunks, B = q's, lane
// (lq, lc) = (lane / 16, lane % 16) holding chunk 4 c + lq of row / head lc;
// the sum's lane holds rows 4 lq + i of head lc.  Every matrix instruction
// (32 exact 16-bit products, or 4 fp32 ones) starts from zero and the results
// are added pairwise, N of them from number LO on, so that no rounding meets
// more of the sum than in a tree of short scalar chains: error of a dot of 128
// over its size 4.7e-8 in bf16, 7.3e-8 in fp32 (as one chain 6.0e-8 and 2.0e-7,
// as four 4.7e-8 and 1.1e-7; a tree of chains of 8 / 4 fused multiply-adds
// 4.8e-8 and 7.3e-8).  fused_score_accumulate, 8 items of 7,564 rows, 4 heads,
// D = 128, both passes: bf16 12.3 us either way, fp32 17.5 -> 19.0 us.
// PER: fp32 matrix instructions in one chain at the leaves.
template <typename T, int LO, int N, int PER>
__device__ __forceinline__ f32x4 dot_tree(const u32x4* a, const u32x4* b) {
  f32x4 c = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (N > PER) {
    return dot_tree<T, LO, N / 2, PER>(a, b) + dot_tree<T, LO + N / 2, N / 2, PER>(a, b);
  } else if constexpr (sizeof(T) == 4) {
#pragma unroll
    for (int i = LO; i < LO + N; ++i)
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(a[i / 4][i % 4]), __uint_as_float(b[i / 4][i % 4]), c, 0,
                                               0, 0);
    return c;
  } else {
#pragma unroll
    for (int i = LO; i < LO + N; ++i)
      if constexpr (std::is_same<T, bf16_t>::value)
        c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[i]), __builtin_bit_cast(bf16x8, b[i]),
                                                    c, 0, 0, 0);
      else
        c = __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a[i]), __builtin_bit_cast(f16x8, b[i]), c,
                                                   0, 0, 0);
    return c;
  }
}
// The dots of NC chunks.  fp32: 8 results at a time, ordered by passing the
// next chunks through an empty instruction that takes the last 8's sum (all
// 64 at D = 256 at once would leave one wave per SIMD, and that one spilling).
template <typename T, int NC, int PER = 1>
__device__ __forceinline__ f32x4 dot_rows(u32x4* a, const u32x4* b) {
  if constexpr (sizeof(T) == 4) {
    constexpr int CG = 2 * PER, NG = NC / CG;  // chunks of a group, groups
    f32x4 y[NG];
#pragma unroll
    for (int g = 0; g < NG; ++g) {
      if (g > 0) {
#pragma unroll
        for (int c = 0; c < CG; ++c) asm volatile("" : "+v"(a[CG * g + c]) : "v"(y[g - 1]));
      }
      y[g] = dot_tree<T, 0, 8 * PER, PER>(a + CG * g, b + CG * g);
    }
#pragma unroll
    for (int o = 1; o < NG; o *= 2)
#pragma unroll
      for (int g = 0; g + o < NG; g += 2 * o) y[g] += y[g + o];
    return y[0];
  } else {
    return dot_tree<T, 0, NC, PER>(a, b);
  }
}

}  // namespace wnw
