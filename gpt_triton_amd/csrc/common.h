// Shared device/host helpers for the gfx950 kernels of libgptmi.
#pragma once
#include <hip/hip_runtime.h>
#include <hip/hip_fp16.h>
#include <stdint.h>

#include "launch.h"

namespace gptmi {

typedef _Float16 h8 __attribute__((ext_vector_type(8)));
typedef _Float16 h4 __attribute__((ext_vector_type(4)));
typedef _Float16 h2 __attribute__((ext_vector_type(2)));
typedef float f4 __attribute__((ext_vector_type(4)));
typedef float f16v __attribute__((ext_vector_type(16)));
typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef uint32_t u2 __attribute__((ext_vector_type(2)));

constexpr int kWave = 64;

// Stores that write through: the line goes to memory at once instead of staying dirty in the XCD's L2
// until the kernel ends, when the write-back of all of it stands between this launch and the next
// (behind 29 MB of plain stores 3.0 us from the last wavefront to the first of the next launch, 1.1
// without).  The memory-side cache keeps the line for the next kernel; non-temporal stores, which are as
// fast by themselves, send it to HBM (124M forward, 16 x 300 tokens: plain 1907, non-temporal 1858,
// these 1813 us; 2 x 64 tokens captured: 412, 424, 410).  In assembly, since no builtin stores 16
// bytes this way: the trailing s_nop keeps the next VALU instruction from overwriting data registers
// that a store of more than 64 bits reads a little after issue.
template <typename V>
__device__ __forceinline__ void store_through(V* p, V v) {
  static_assert(sizeof(V) == 8 || sizeof(V) == 16, "8 or 16 bytes");
  if constexpr (sizeof(V) == 16)
    asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" : : "v"(p), "v"(v) : "memory");
  else
    asm volatile("global_store_dwordx2 %0, %1, off sc0 sc1" : : "v"(p), "v"(v) : "memory");
}

// The transposing LDS load: within a block of 16 lanes, lane i receives element i % 4 of the 8 bytes that
// lanes i / 4, i / 4 + 4, + 8 and + 12 point at -- with lane s pointing at the 4 columns 4 (s % 4).. of row s / 4 of
// a row-major matrix, column i of 4 rows.
typedef short s4v __attribute__((__vector_size__(4 * sizeof(short))));
__device__ __forceinline__ h4 lds_read_tr16(const char* p) {
  const s4v r = __builtin_amdgcn_ds_read_tr16_b64_v4i16(
      (__attribute__((address_space(3))) s4v*)(uintptr_t)p);
  return __builtin_bit_cast(h4, r);
}

// Workgroups for what a launch requests ahead, behind its `workers`: the CUs that these leave idle, or 128 that find room as the
// last of them end (64 gain less: 28 x 300 tokens of 124M none / 64 / 128 2072 / 1923 / 1901 us, 32 x 300 in fp32
// 2440 / 2266 / 2268, 16 x 512 2054 / 1922 / 1899, 64 x 300 3977 / 3940 / 3928; 1024 wide 8 x 1024 6024 / 5661 /
// 5623, 1280 wide 4 x 700 5855 / 5514 / 5361).
inline int prefetch_workgroups(const Prefetch* ahead, int64_t workers, int cus) {
  return ahead == nullptr || ahead->empty() ? 0 : workers <= cus - 64 ? cus - (int)workers : 128;
}
// The workgroups from `first` on of a launch: a word of each 128-byte line, and a thread has 8 loads on their way at a
// time.  As loops over the four matrices, each load was waited for before the next was made, a microsecond or two
// apiece: forwards, weights from HBM, 60 x 24 tokens of 124M 729 -> 717 us, 21 x 64 644 -> 628, 28 x 300 2020 -> 2006, 1024 wide
// 15 x 300 3778 -> 3738, 1600 wide 1 x 200 2759 -> 2733, 4 x 512 8812 -> 8706; others equal.
template <int NT>
__device__ __forceinline__ void prefetch_lines(const PrefetchArgs& pf, int first) {
  typedef const __attribute__((address_space(1))) unsigned* Word;
  const unsigned xcd = blockIdx.x & 7, skipped = (xcd - (unsigned)first) & 7;  // ids in front of the XCD's first one
  const unsigned block = (blockIdx.x - (unsigned)first) >> 3, blocks = (gridDim.x - (unsigned)first - skipped + 7) >> 3;
  const AheadLines lines(pf, xcd);
  unsigned sink = 0;
  constexpr unsigned B = 8;
  const unsigned step = blocks * NT;
  for (unsigned i = block * NT + threadIdx.x; i < lines.all(); i += B * step) {
    unsigned w[B];
#pragma unroll
    for (unsigned j = 0; j < B; ++j) {
      const unsigned n = i + j * step;
      w[j] = *(Word)(uintptr_t)lines.at(n < lines.all() ? n : lines.all() - 1);
    }
#pragma unroll
    for (unsigned j = 0; j < B; ++j) sink ^= w[j];
  }
  asm volatile("" : : "v"(sink));
}

// Cross-lane steps without the LDS: an xor shuffle compiles to ds_bpermute, ~100 cycles of latency
// per step of a reduction, and the reductions of a LayerNorm row (twelve steps) or of a softmax tile
// sit on the critical path of their kernels.  The swaps and row rotations are VALU instructions.
//   half_swap(v): v of lane % 32 (a) and of lane % 32 + 32 (b), for both lanes in this order (the attention kernel with 16
//                 queries a wavefront adds in it)
struct LanePair {
  float a, b;
};
__device__ __forceinline__ LanePair half_swap(float v) {
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane32_swap(u, u, false, false);
  const unsigned x = r[0], y = r[1];
  return {__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)};
}
__device__ __forceinline__ LanePair row_swap(float v) {  // a: of the lane without its bit 4, b: with it
  const unsigned u = __builtin_bit_cast(unsigned, v);
  const auto r = __builtin_amdgcn_permlane16_swap(u, u, false, false);
  const unsigned x = r[0], y = r[1];
  return {__builtin_bit_cast(float, x), __builtin_bit_cast(float, y)};
}
template <int N>
__device__ __forceinline__ float row_rotate(float v) {  // within rows of 16 lanes
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x120 | N,
                                                               0xf, 0xf, true));
}
// The other lane of xor-8, 4, 2, 1 steps taken in this order: behind the step of distance 2 N all
// lanes that differ in the higher bits hold the same value, so rotating by N finds the value of lane ^ N.
template <int G, typename Op>
__device__ __forceinline__ float group_reduce(float v, Op op) {
  static_assert(G == 64 || G == 32, "a wavefront or its halves");
  if constexpr (G == 64) {
    const LanePair p = half_swap(v);
    v = op(p.a, p.b);
  }
  const LanePair p = row_swap(v);
  v = op(p.a, p.b);
  v = op(v, row_rotate<8>(v));
  v = op(v, row_rotate<4>(v));
  v = op(v, row_rotate<2>(v));
  return op(v, row_rotate<1>(v));
}
// Sum / max over aligned groups of G lanes (G = 64: the wavefront; G = 32: each half on its own);
// every lane gets the result.
template <int G>
__device__ __forceinline__ float group_sum(float v) {
  return group_reduce<G>(v, [](float a, float b) { return a + b; });
}
template <int G>
__device__ __forceinline__ float group_max(float v) {
  return group_reduce<G>(v, [](float a, float b) { return fmaxf(a, b); });
}
__device__ __forceinline__ float wave_sum(float v) { return group_sum<kWave>(v); }
__device__ __forceinline__ float wave_max(float v) { return group_max<kWave>(v); }
// Sum / max of this lane's value and that of lane ^ 32.
__device__ __forceinline__ float half_sum(float v) {
  const LanePair p = half_swap(v);
  return p.a + p.b;
}
__device__ __forceinline__ float half_max(float v) {
  const LanePair p = half_swap(v);
  return fmaxf(p.a, p.b);
}

// tanh-form GELU of the reference (kernels.py:15-26): 0.5 x (1 + tanh(u)) with
// tanh(u) = 2 sigmoid(2u) - 1, u = sqrt(2/pi) (x + 0.044715 x^3).  Algebraically
// that is x * sigmoid(2u) = x / (1 + exp(-2u)); evaluated here as one exp2 and
// one hardware reciprocal (1 ulp), ~1e-7 relative from the reference's form.
__device__ __forceinline__ float gelu_new(float x) {
  // k = -2 * sqrt(2/pi) * log2(e), folded into the cubic's coefficients: exp(-2u) = exp2(x (k +
  // 0.044715 k x^2)) -- one multiplication fewer per element of a GELU epilogue
  constexpr float k = -2.0f * 0.7978845608028654f * 1.4426950408889634f;
  const float e = __builtin_amdgcn_exp2f(x * fmaf(0.044715f * k, x * x, k));
  return x * __builtin_amdgcn_rcpf(1.0f + e);
}

// ---------------------------------------------------------------------------
// Dropout of the reference (kernels.py:31-34): keep where tl.rand(seed, offset) > p, scaled
// by a true division by (1 - p).  tl.rand is Philox-4x32-10 with counter (offset, 0, 0, 0) and
// the 64-bit seed as key; the first output word, read as int32 with negatives folded by
// -x-1, times 4.6566127342e-10 gives the uniform in [0, 1).  NCH independent offsets share
// one rolled round loop so that a call site stays a few dozen instructions.
//
// Bound by the 32 x 32 -> 64 bit products (quarter rate).  Of the 20 of the general form 17 are left,
// one of them uniform: three counter words start as 0, so round 1 has one product and round 2's
// second is the same for every offset, and of rounds 9 and 10 only what reaches the first word is
// formed.
// ---------------------------------------------------------------------------
struct DropoutArgs {
  float p;
  unsigned seed_lo, seed_hi;
};

__device__ __forceinline__ unsigned xor3(unsigned a, unsigned b, unsigned c) {
  return __builtin_amdgcn_bitop3_b32(a, b, c, 0x96);
}

template <int NCH>
__device__ __forceinline__ void philox_uniform(const DropoutArgs& d, const unsigned (&offset)[NCH],
                                               float (&u)[NCH]) {
  constexpr unsigned A = 0xD2511F53u, B = 0xCD9E8D57u, W0 = 0x9E3779B9u, W1 = 0xBB67AE85u;
  unsigned c0[NCH], c1[NCH], c2[NCH], c3[NCH];
  unsigned k0 = d.seed_lo, k1 = d.seed_hi;
  const uint64_t seed_a = (uint64_t)A * k0;  // round 2's product of word 0, which round 1 makes k0
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const uint64_t a = (uint64_t)A * offset[i];
    c2[i] = (unsigned)(a >> 32) ^ k1;
    c3[i] = (unsigned)a;
  }
  k0 += W0;
  k1 += W1;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const uint64_t b = (uint64_t)B * c2[i];
    c0[i] = (unsigned)(b >> 32) ^ k0;
    c1[i] = (unsigned)b;
    c2[i] = xor3((unsigned)(seed_a >> 32), c3[i], k1);
    c3[i] = (unsigned)seed_a;
  }
#pragma unroll 1
  for (int r = 0; r < 6; ++r) {
    k0 += W0;
    k1 += W1;
#pragma unroll
    for (int i = 0; i < NCH; ++i) {
      const uint64_t b = (uint64_t)B * c2[i], a = (uint64_t)A * c0[i];
      c0[i] = xor3((unsigned)(b >> 32), c1[i], k0);
      c2[i] = xor3((unsigned)(a >> 32), c3[i], k1);
      c1[i] = (unsigned)b;
      c3[i] = (unsigned)a;
    }
  }
  k0 += W0;
  k1 += W1;
#pragma unroll
  for (int i = 0; i < NCH; ++i) {
    const unsigned n2 = xor3(__umulhi(A, c0[i]), c3[i], k1), n1 = B * c2[i];
    const unsigned w = xor3(__umulhi(B, n2), n1, k0 + W0);
    const int x = (int)w;
    u[i] = (float)(x ^ (x >> 31)) * 4.6566127342e-10f;  // ~x = -x-1 for negative words
  }
}

// x / keep for the kept values.  Division by one number: its reciprocal is taken once, and the
// remainder of the first quotient corrects it (correctly rounded for a correctly rounded reciprocal,
// P. Markstein, IBM J. Res. Dev. 34, 1990).  That takes a quotient that is finite and a remainder
// that is no subnormal number, 24 bits below x: |x| from 2^-100 to 2^127 keep.  Values among which
// there are others (infinities, NaN and 0 count) are divided; asked once for the N values of a thread
// (MLP block of 4800 x 768 with the mask at hand: 77.1 us; 79.3 asked per value, 76.3 never).
struct KeepScale {
  float keep, inv;
  __device__ __forceinline__ explicit KeepScale(float p) : keep(1.0f - p), inv(1.0f / (1.0f - p)) {}
  template <int N>
  __device__ __forceinline__ void apply(float (&x)[N]) const {
    float lo = __builtin_fabsf(x[0]), hi = lo;
#pragma unroll
    for (int i = 1; i < N; ++i) {
      lo = fminf(lo, __builtin_fabsf(x[i]));
      hi = fmaxf(hi, __builtin_fabsf(x[i]));
    }
    if (__builtin_expect(lo >= 0x1p-100f && hi <= 0x1p127f * keep, 1)) {
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = finite(x[i]);
    } else {
#pragma unroll
      for (int i = 0; i < N; ++i) x[i] = x[i] / keep;
    }
  }
  // for an x that is an fp16 number: no range to ask for, div_fixup passes infinities, NaN and 0 through
  __device__ __forceinline__ float of_half(float x) const {
    const float q = x * inv;
    return __builtin_amdgcn_div_fixupf(fmaf(fmaf(-q, keep, x), inv, q), keep, x);
  }
  // for an x that is rounded to fp16 afterwards and no infinity (the quotients that `finite` would
  // round otherwise are far below fp16's smallest)
  __device__ __forceinline__ float finite(float x) const {
    const float q = x * inv;
    float r = fmaf(fmaf(-q, keep, x), inv, q);
    asm("" : "+v"(r));  // rounded to fp32 before it is to fp16, not by one mixed-precision fma
    return r;
  }
};

template <int NCH>
__device__ __forceinline__ void dropout_apply(const DropoutArgs& d, const unsigned (&offset)[NCH],
                                              float (&x)[NCH]) {
  float u[NCH];
  philox_uniform<NCH>(d, offset, u);
  KeepScale(d.p).apply(x);
#pragma unroll
  for (int i = 0; i < NCH; ++i) x[i] = u[i] > d.p ? x[i] : 0.0f;
}

// v where bit `b` of `bits` is set, +0 elsewhere (v's bits under a mask: one bit-field extract, one and).
__device__ __forceinline__ float keep_if(unsigned bits, int b, float v) {
  return __int_as_float(__builtin_amdgcn_sbfe((int)bits, (unsigned)b, 1u) & __float_as_int(v));
}

void set_error(const char* fmt, ...);

}  // namespace gptmi
