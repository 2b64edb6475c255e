// The exponentials of 16-bit attention, shared by its kernels so that they give the same bits.
//
// exp(x - m) is exp2(x k - sh) with k = log2 e (times the scale where that is folded in) and sh =
// round(m k): one fused multiply-add and one exponential per score.  The rounding of sh is a common
// factor of a row's terms and cancels in the division by the row sum, as long as
//   - a step that leaves the maximum as it was rescales the sum by exactly 1: the difference of the
//     maxima comes first (exp2(m k - sh) is that common factor, and a row of many steps would
//     collect its powers: with fp16 scores and 2048 keys a tenth of the outputs changed);
//   - the product stays moderate.  Additive masks can make it huge (padding written as the type's
//     lowest value or as -1e9, of which a row or its first keys have nothing else): m k overflows,
//     or the common factor does.  With an additive mask (ADD), bf16 maxima of 2^16 and more use
//     k = 1, sh = m, which is exact: neighbouring bf16 values differ by 2^8 and more there, so
//     every term is 1 (x = m) or 0 either way (fp16 ends at 65504).
#pragma once

#include <type_traits>

#include "rowops.h"

namespace biops {

// scale = 2^k with -8 <= k <= 0: the bf16 kernels without an additive mask keep their scores in
// units of round(S) and fold the scale into the exponentials (attention_fused.hip).
int pow2_scale(float scale);

struct ExpBase {
  float m, k, sh;  // exp(x - m) = exp2(x * k - sh)
};

// m: the maximum so far, -inf while no key is visible (every term is then exp(-inf) = 0).
template <typename T, bool ADD>
__device__ __forceinline__ ExpBase attn_exp_base(float m, float kexp) {
  const float mm = m == -INFINITY ? 0.f : m;
  if constexpr (ADD && std::is_same<T, bf16_t>::value) {
    const bool exact = fabsf(mm) >= 65536.f;
    return ExpBase{mm, exact ? 1.f : kexp, exact ? mm : mm * kexp};
  }
  return ExpBase{mm, kexp, mm * kexp};
}
__device__ __forceinline__ float attn_exp(float x, const ExpBase& b) {
  return __builtin_amdgcn_exp2f(__builtin_fmaf(x, b.k, -b.sh));
}
// Factor of the sum so far when the maximum goes from m to that of base b.
__device__ __forceinline__ float attn_rescale(float m, const ExpBase& b) {
  return __builtin_amdgcn_exp2f((m - b.m) * b.k);
}

}  // namespace biops
