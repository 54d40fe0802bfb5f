// The arithmetic of one LayerNorm row (reference: fused_layer_norm_kernel, kernels.py:104-145),
// in one place so that every kernel that normalises a row gives the same bits: the LayerNorm
// kernel, the embedding kernel that emits the first LayerNorm, and the GEMM whose operand
// prologue normalises its rows.
#pragma once
#include "common.h"

namespace gptmi {

// What bounds a row is VALU instructions, not memory, where few rows are normalised by every column
// tile of a product (gemm_tile.hip, LNA): some 11 an element, of which 5 are left.
//   * fp16 rows stay packed: v_fma_mix_f32 takes a half as it stands (x * 1 + s is s + x and
//     x * 1 - mean is x - mean, rounded once, so the values are those of a conversion in front);
//   * FULL: rows that are whole shares of 32 lanes (256 and 768 halves) need no masks in the operand prologue;
//   * the divisions by H are a product with its reciprocal and one correction by the remainder, which
//     is the correctly rounded quotient (P. Markstein, IBM J. Res. Dev. 34, 1990) unless the remainder
//     is subnormal; a mean that is not finite makes the row NaN either way, a variance beyond 2^100 is
//     divided;
//   * 1 / sqrt is the hardware's reciprocal square root (1 ulp) and a Newton step, nearer to the exact
//     value than a root and a division, which are left to arguments outside 2^-100 .. 2^100.
// LayerNorm -> qkv / ffn1 at 128 rows of 768: 7.5 / 7.9 us with 11, 6.9 / 7.3 with 5; at 24 rows 6.1 / 6.1
// and 5.6 / 5.7.  Error against 64 bits over nine widths and five scales: never larger than with 11 (256
// floats 6.33e-8 -> 5.84e-8).
#pragma clang fp contract(off)
template <int J>
__device__ __forceinline__ unsigned half_pair(h8 v) {
  return __builtin_bit_cast(u4, v)[J / 2];
}
// x[J] + c in one instruction
template <int J>
__device__ __forceinline__ float half_plus(h8 x, float c) {
  float r;
  const unsigned u = half_pair<J>(x);
  if constexpr (J % 2 == 0)
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel_hi:[1,0,0]" : "=v"(r) : "v"(u), "v"(c));
  else
    asm("v_fma_mix_f32 %0, %1, 1.0, %2 op_sel:[1,0,0] op_sel_hi:[1,0,0]" : "=v"(r) : "v"(u), "v"(c));
  return r;
}
template <int J = 0>
__device__ __forceinline__ float chunk_sum(h8 x, float s) {
  s = half_plus<J>(x, s);
  if constexpr (J < 7) s = chunk_sum<J + 1>(x, s);
  return s;
}
__device__ __forceinline__ float chunk_sum(f4 x, float s) {
#pragma unroll
  for (int j = 0; j < 4; ++j) s += x[j];
  return s;
}
template <int J = 0>
__device__ __forceinline__ void chunk_minus(h8 x, float mean, float (&d)[8]) {
  d[J] = half_plus<J>(x, -mean);
  if constexpr (J < 7) chunk_minus<J + 1>(x, mean, d);
}
__device__ __forceinline__ void chunk_minus(f4 x, float mean, float (&d)[4]) {
#pragma unroll
  for (int j = 0; j < 4; ++j) d[j] = x[j] - mean;
}
__device__ __forceinline__ float over(float s, float n, float inv_n) {
  const float q = s * inv_n;
  return __builtin_fmaf(__builtin_fmaf(-q, n, s), inv_n, q);
}

// A row is spread over LPR lanes: lane l holds the 16-byte chunks l, l + LPR, ... of the row's nchunks
// (VN elements each; zeros in the places past the end).  fp32 mean, then the centred biased variance;
// d: the elements less the mean.  Each lane adds its elements in that order.  Contraction is spelled
// out (fmaf where a multiply-add is fused, none elsewhere): left to the compiler, two kernels were
// fused differently.
template <int CH, int VN, int LPR, bool FULL, typename V>
__device__ __forceinline__ void layernorm_stats(const V (&x)[CH], int lane, int nchunks, int H, float eps,
                                                float (&d)[CH][VN], float& rstd) {
  const float n = (float)H, inv_n = 1.0f / n;
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) s = chunk_sum(x[i], s);
  const float mean = over(group_sum<LPR>(s), n, inv_n);
  float q = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    chunk_minus(x[i], mean, d[i]);
    if (FULL || lane + i * LPR < nchunks) {
#pragma unroll
      for (int j = 0; j < VN; ++j) q = __builtin_fmaf(d[i][j], d[i][j], q);
    }
  }
  q = group_sum<LPR>(q);
  float v;
  if (__builtin_expect(q <= 0x1p100f, 1)) v = over(q, n, inv_n) + eps;
  else v = q / n + eps;
  if (__builtin_expect(v >= 0x1p-100f && v <= 0x1p100f, 1)) {
    const float y = __builtin_amdgcn_rsqf(v);
    rstd = __builtin_fmaf(__builtin_fmaf(-v * y, y, 1.0f), 0.5f * y, y);
  } else {
    rstd = 1.0f / sqrtf(v);
  }
}
// (x - mean) * rstd * w + b
__device__ __forceinline__ float layernorm_apply(float d, float rstd, float w, float b) {
  const float z = d * rstd;
  float r = __builtin_fmaf(z, w, b);
  // The result is an fp32 number that the caller rounds to the storage type (the reference's
  // fp32 arithmetic followed by a cast).  Without this fence the compiler may merge the
  // multiply-add and the conversion into one mixed-precision instruction that rounds the exact
  // result once, straight to fp16 -- in some kernels and not in others.
  asm("" : "+v"(r));
  return r;
}
#pragma clang fp contract(fast)

// Lanes per row for rows of `nchunks` 16-byte chunks: 32 if that leaves fewer idle lane slots
// than 64 (96 chunks: 3 passes of 32 against 2 passes of 64 with a quarter empty), but not beyond 4
// chunks a lane: longer shares fetch the LayerNorm's parameters behind the statistics instead of with
// the row (1280 and 1600 halves; 8 rows of 1600: 4.2 -> 2.9 us, 65536 rows 68.8 -> 64.8).
inline int lanes_per_row(int nchunks) {
  const int slots32 = (nchunks + 31) / 32 * 32, slots64 = (nchunks + 63) / 64 * 64;
  return slots32 < slots64 && nchunks <= 128 ? 32 : 64;
}

}  // namespace gptmi
