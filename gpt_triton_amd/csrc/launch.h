// Host-side launchers implemented by the kernel translation units and called
// by the C ABI in capi.cpp.  All of them only enqueue work on `st`.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "weights_ahead.h"

namespace gptmi {

// Dropout of one launch: probability p (0 = none) and the 64-bit seed of the generator.
struct Dropout {
  float p;
  uint64_t seed;
  const void* keep = nullptr;  // the mask's bits, if the caller has them (launch_dropout_mask)
};

// Bit o % 32 of word o / 32 of `mask`: whether offset o is kept, for all o below 32 * words.
void launch_dropout_mask(void* mask, int64_t words, Dropout drop, hipStream_t st);

int launch_embed(const int64_t* ids, const void* wte, const void* wpe, void* out,
                 int64_t rows, int64_t L, int64_t V, int H, Dropout drop, bool f16, hipStream_t st);
bool launch_embed_layernorm(const int64_t* ids, const void* wte, const void* wpe, const void* w,
                            const void* b, void* emb, void* out, int64_t rows, int64_t L,
                            int64_t V, int H, float eps, bool f16, hipStream_t st);
// out_f16 with fp32 rows: the result rounded to fp16, as the GEMM rounds its operands
int launch_layernorm(const void* x, const void* w, const void* b, void* out,
                     int64_t M, int H, float eps, bool f16, bool out_f16, hipStream_t st);
int launch_softmax(const void* x, void* out, int64_t M, int H, bool f16,
                   hipStream_t st);
void launch_pack_rows(const void* src, void* dst, int64_t R, int K, int Kp, bool f16,
                      hipStream_t st);
void launch_pack_transpose(const void* src, void* dst, int K, int N, int Kp, bool f16,
                           hipStream_t st);
// two weights, K1 and K2 multiples of 64; N1 or N2 may be 0
void launch_pack_transpose_pair(const void* s1, void* d1, int K1, int N1, const void* s2, void* d2, int K2,
                                int N2, bool f16, hipStream_t st);

// launch_layernorm to fp16 and launch_pack_transpose_pair, which do not depend on each other, in one launch
// where their sizes and alignments allow it.
void launch_layernorm_pack_pair(const void* x, const void* w, const void* b, void* out, int64_t M, int H,
                                float eps, const void* s1, void* d1, int K1, int N1, const void* s2, void* d2,
                                int K2, int N2, bool f16, hipStream_t st);
// whether fp16 rows of this width leave room for that
bool layernorm_packs(int H);

// Epilogue description of one GEMM launch: out = gelu?(acc + bias) + residual,
// stored either as a plain [M][N] matrix or scattered into q/k/v [B][heads][L][d].
struct GemmEpilogue {
  const void* bias;      // [N] in the storage dtype, or nullptr
  const void* residual;  // [M][N] in the storage dtype, or nullptr
  void* out;             // [M][N] (plain mode)
  void* q;               // qkv mode: three [B][heads][L][d] tensors
  void* k;
  void* v;
  int64_t L;      // qkv mode: rows per sequence
  int heads;      // qkv mode
  int d;          // qkv mode: head size
  int gelu;       // apply tanh-GELU after the bias
  Dropout drop;   // after the GELU, before the residual (plain mode only)
  bool qkv;       // scatter mode
  bool f16;       // storage dtype of bias / residual / outputs
  bool out_f16;   // fp32 storage: outputs rounded to fp16 all the same (the next product's operand)
};

// C[M][N] = A[M][Kp] . Bt[N][Kp]^T with fp16 operands (Kp % 64 == 0), fp32
// accumulation and the fused epilogue above.
int launch_gemm(const void* A, const void* Bt, int64_t M, int N, int Kp,
                const GemmEpilogue& ep, hipStream_t st);

// The same product, fp16 storage, with the weight as the caller has it, W [K][N]: no packed image.  Same kernels,
// same division of the rows, same bits.  gemm_reads_kn says where that is taken (and is the faster way).
bool gemm_reads_kn(const void* W, int64_t M, int N, int K, const GemmEpilogue& ep);
int launch_gemm_kn(const void* A, const void* W, int64_t M, int N, int K, const GemmEpilogue& ep, hipStream_t st);

// The same product with A = LayerNorm(x; ln_w, ln_b, eps), x [M][H] in the storage type with H = K a multiple
// of 64: every workgroup normalises the rows of its tile in its operand prologue (the bits of
// launch_layernorm's fp16 output) and the normalised matrix never goes to memory.  fp16 output, no residual,
// no dropout; meant for few rows, where a LayerNorm launch costs more than normalising the rows
// once per column tile.  gemm_layernorm_supported says whether (M, H) is taken.
bool gemm_layernorm_supported(int64_t M, int H, bool f16 = true);
int launch_gemm_layernorm(const void* x, const void* ln_w, const void* ln_b, float eps,
                          const void* Bt, int64_t M, int N, int H, const GemmEpilogue& ep,
                          hipStream_t st);

// LayerNorm (unless x is normed), q, k, v product (packed weight image Bt [3h][h]) and causal attention of short
// sequences in one launch: fp16, head size 64, out [B][L][heads][64], the bits of the launches it stands for.  All
// pointers 16-byte aligned.  split: attn_front_split's, the product's groups of k-slices, or 0 for what it does not take.
int attn_front_split(int64_t B, int64_t L, int64_t heads, int64_t h);
int launch_attn_front(int split, const void* x, bool normed, const void* ln_w, const void* ln_b, float eps, const void* Bt,
                      const void* bias, void* out, int64_t B, int64_t L, int64_t heads, float scale, hipStream_t st,
                      const Prefetch* ahead = nullptr);

// q, out: L rows per (batch, head); k, v: Lk rows.
int launch_flash_attn(const void* q, const void* k, const void* v, void* out,
                      int64_t B, int64_t N, int64_t L, int64_t Lk, int d, float scale,
                      Dropout drop, bool out_blnd, bool f16, hipStream_t st, const Prefetch* ahead = nullptr);


// The attention of an fp32 model on fp16 copies of q, k, v: the fp32 kernels round q, k and v to fp16
// as they read them, and the projection rounds its operand, so with the copies written by the product
// in front and the output rounded here the values are the same and half the bytes move.  fp32 softmax
// arithmetic as for fp32 storage; equal lengths; out [B][L][N][d] fp16.
int launch_flash_attn_operands(const void* q, const void* k, const void* v, void* out, int64_t B,
                               int64_t N, int64_t L, int d, float scale, Dropout drop, hipStream_t st,
                               const Prefetch* ahead = nullptr);

}  // namespace gptmi
