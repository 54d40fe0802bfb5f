// The softmax arithmetic that the attention kernels share, so that whichever of them serves a call gives the
// same bits.
#pragma once
#include "common.h"

namespace gptmi {

// The softmax arithmetic, in three forms.
// ACC = false, SCALED = false (fp16 storage): running max on the raw scores, scale * log2(e) folded
// into one fused multiply-add in front of the hardware's exp2, a reciprocal for the denominator -- the
// same real-number formula as the reference, two VALU operations per score fewer.
// SCALED = true: the running max is that of the scaled scores, as in the reference, so that what the
// weights subtract and what the rescaling divides are the same number.  Where a tile leaves the max
// in place its difference is 0 and the rescaling exactly 1.  Formed from the products instead
// (old * c - m * c), the compiler fuses one of the two and every key tile multiplies by exp of a
// rounding error (fp32, d = 128, scaled scores of 700, 16 tiles: up to 5.2e-4 of the output); with the
// product rounded per max, tiles of different max disagree by that rounding (fp16, scaled scores of
// 500000: 3.6e-3).
//   ACC = true (fp32 storage, and the fp16 copies of q, k, v that the block functions of fp32 models
//   hand on): library exp and a true division, so fewer fp16 rounding flips of P against the
//   reference's np.exp.  (Argument reductions of fewer operations were less exact: 0.95 ulp against expf's 0.85.)
//   ACC = false (fp16 storage with dropout): the hardware's exp2.
template <bool ACC, bool SCALED = ACC>
struct Softmax {
  float c;  // SCALED: scale; otherwise scale * log2(e)
  __device__ __forceinline__ explicit Softmax(float scale)
      : c(SCALED ? scale : scale * 1.4426950408889634f) {}
  // what the running max is taken of
  __device__ __forceinline__ float score(float s) const { return SCALED ? s * c : s; }
  // what weight() subtracts for the running max m
  __device__ __forceinline__ float base(float m) const { return SCALED ? m : m * c; }
  // the weight of score s = score(.) for base b = base(m)
  __device__ __forceinline__ float weight(float s, float b) const {
    if constexpr (SCALED) return ACC ? expf(s - b) : __expf(s - b);
    else return __builtin_amdgcn_exp2f(fmaf(s, c, -b));
  }
  // the rescaling when the running max goes from `old` to m
  __device__ __forceinline__ float rescale(float old, float m) const {
    if constexpr (SCALED) return ACC ? expf(old - m) : __expf(old - m);
    else return __builtin_amdgcn_exp2f((old - m) * c);
  }
};

// o / den for a whole row: ACC divides, otherwise the reciprocal (1 ulp of fp32) is taken once
template <bool ACC>
struct Normalise {
  float d;
  __device__ __forceinline__ explicit Normalise(float den) : d(ACC ? den : __builtin_amdgcn_rcpf(den)) {}
  __device__ __forceinline__ float operator()(float o) const { return ACC ? o / d : o * d; }
};

// The same for a result that is rounded to fp16: the reciprocal is taken once, and the remainder of the first
// quotient corrects it to the bits of the division (P. Markstein, IBM J. Res. Dev. 34, 1990; quotients whose
// remainder is no normal number are far below fp16's smallest; div_fixup: infinities, NaN and 0).  4
// operations instead of 10, 32 times a query's lane: fp32 attention of 32 x 12 pairs of 300 rows 32.1 -> 28.8 us.
template <bool ACC>
struct NormaliseHalf {
  float d, inv;
  __device__ __forceinline__ explicit NormaliseHalf(float den)
      : d(den), inv(ACC ? 1.0f / den : __builtin_amdgcn_rcpf(den)) {}
  __device__ __forceinline__ float operator()(float o) const {
    const float q = o * inv;
    return ACC ? __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, d, o), inv, q), d, o) : q;
  }
};

}  // namespace gptmi
