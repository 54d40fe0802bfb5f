// Bandwidth-bound row kernels: embedding gather, LayerNorm, row softmax and the
// operand packers of the GEMM.  One wavefront owns one row; a row is held in
// registers between its passes so HBM sees one read and one write per element.
#include <type_traits>

#include "common.h"
#include "layernorm.h"
#include "launch.h"

namespace gptmi {

template <typename T> struct Vec;
template <> struct Vec<_Float16> {
  static constexpr int N = 8;
  typedef h8 type;
};
template <> struct Vec<float> {
  static constexpr int N = 4;
  typedef f4 type;
};

// The row kernels write through (store_through): a line is on its way while the kernel still runs.  All stores
// of a thread come behind all its loads and arithmetic, kept there by `pin`, with one wait in front of them
// (`loads_done`): a wait for a load between two stores, which the compiler puts in front of every value that a
// branch may have left in flight, would be a wait for the first store's way to memory.  LayerNorm, us, plain
// stores / through with such waits / through without: halves 128 x 768 3.3 / 3.4 / 2.9, 128 x 1600 3.8 / 4.0 / 3.2,
// 4800 x 768 4.7 / 4.2 / 3.8, 4800 x 1600 8.2 / 7.0 / 6.2; captured forwards of 1 x 24 tokens, 1600-wide, 48 layers,
// 1820 / 1890 / 1770.
// What an embedding writes beyond half of the memory-side cache is non-temporal, as make_epi does it: a GEMM's
// epilogue reads it a block later (through / non-temporal: 65536 x 1024 halves 39 / 39, 65536 x 1600 79 / 61,
// 153600 x 768 75 / 67; with the LayerNorm, whose output counts too, 65536 x 768 51 / 44, 65536 x 1024 86 / 58).  A
// LayerNorm's output is the next kernel's operand and stays at any size (all non-temporal, the forward of 512 x
// 300 tokens takes 29.49 ms, 28.42).
constexpr int64_t kStreamBytes = 128 << 20;

template <typename V>
__device__ __forceinline__ void pin(V& v) {
  typedef std::conditional_t<sizeof(V) == 16, u4, u2> U;
  U u = __builtin_bit_cast(U, v);
  asm volatile("" : "+v"(u));
  v = __builtin_bit_cast(V, u);
}
__device__ __forceinline__ void loads_done() { __builtin_amdgcn_s_waitcnt(0x0f70); }  // vmcnt(0)

template <typename V>
__device__ __forceinline__ void store_row(bool stream, V* p, V v) {
  if (stream) __builtin_nontemporal_store(v, p);
  else store_through(p, v);
}

// ---------------------------------------------------------------------------
// Embedding gather: out[row,:] = wte[ids[row],:] + wpe[row % L,:]
// (reference: fused_embeddings_kernel, kernels.py:37-72).  The add is done in
// fp32 and rounded once, which equals one add in the storage dtype.  A token id
// outside [0, V) reads nothing: its wte row counts as zeros (the reference reads
// out of bounds there).
// ---------------------------------------------------------------------------
template <typename T, int LPR>
__global__ __launch_bounds__(256) void embed_vec_kernel(
    const int64_t* __restrict__ ids, const T* __restrict__ wte,
    const T* __restrict__ wpe, T* __restrict__ out, int64_t rows, int64_t L, int64_t V_, int H, int stream) {
  typedef typename Vec<T>::type V;
  constexpr int VN = Vec<T>::N;
  const int lane = threadIdx.x & (LPR - 1);  // LPR lanes per token, as in the LayerNorm kernel
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  if (row >= rows) return;
  const int64_t tok = ids[row];
  const bool known = (uint64_t)tok < (uint64_t)V_;
  const int64_t pos = row % L;
  const V* a = reinterpret_cast<const V*>(wte + (known ? tok : 0) * H);
  const V* b = reinterpret_cast<const V*>(wpe + pos * H);
  V* o = reinterpret_cast<V*>(out + row * H);
  const int nchunks = H / VN;
  for (int c0 = lane; c0 < nchunks; c0 += 4 * LPR) {
    V va[4], vb[4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c0 + i * LPR < nchunks) {
        va[i] = a[c0 + i * LPR];
        vb[i] = b[c0 + i * LPR];
      }
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c0 + i * LPR < nchunks) {
#pragma unroll
        for (int j = 0; j < VN; ++j) va[i][j] = (T)((known ? (float)va[i][j] : 0.f) + (float)vb[i][j]);
        pin(va[i]);
      }
    loads_done();
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (c0 + i * LPR < nchunks) store_row(stream, o + c0 + i * LPR, va[i]);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void embed_scalar_kernel(
    const int64_t* __restrict__ ids, const T* __restrict__ wte,
    const T* __restrict__ wpe, T* __restrict__ out, int64_t rows, int64_t L, int64_t V_, int H) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t tok = ids[row];
  const bool known = (uint64_t)tok < (uint64_t)V_;
  const int64_t pos = row % L;
  for (int c = lane; c < H; c += 64)
    out[row * H + c] = (T)((known ? (float)wte[tok * H + c] : 0.f) + (float)wpe[pos * H + c]);
}

// Embedding with dropout (kernels.py:65-70): the sum is rounded to the storage dtype first,
// the dropout works on that value in fp32 with the COLUMN as the generator's offset, so every
// token sees the same mask.  Rows of whole 16-byte chunks: a thread owns one chunk of columns, draws
// its mask once and walks the rows of its workgroup's share (4800 x 768 halves: 10.2 us, 16.1 with an evaluation
// per element).
template <typename T, bool STREAM>
__global__ __launch_bounds__(256) void embed_dropout_vec_kernel(
    const int64_t* __restrict__ ids, const T* __restrict__ wte,
    const T* __restrict__ wpe, T* __restrict__ out, int64_t rows, int64_t L, int64_t V_, int H,
    DropoutArgs drop) {
  typedef typename Vec<T>::type V;
  constexpr int VN = Vec<T>::N;
  const int nchunks = H / VN, rows_per = nchunks < 256 ? 256 / nchunks : 1;
  const int sub = nchunks < 256 ? (int)threadIdx.x / nchunks : 0;
  const int c = blockIdx.y * 256 + (int)threadIdx.x - sub * nchunks;
  if (sub >= rows_per || c >= nchunks) return;
  unsigned off[VN];
  float u[VN];
#pragma unroll
  for (int j = 0; j < VN; ++j) off[j] = (unsigned)(c * VN + j);
  philox_uniform<VN>(drop, off, u);
  const KeepScale scale(drop.p);
#pragma unroll 4
  for (int64_t row = (int64_t)blockIdx.x * rows_per + sub; row < rows; row += (int64_t)gridDim.x * rows_per) {
    const int64_t tok = ids[row];
    const bool known = (uint64_t)tok < (uint64_t)V_;
    const V va = reinterpret_cast<const V*>(wte + (known ? tok : 0) * H)[c];
    const V vb = reinterpret_cast<const V*>(wpe + row % L * H)[c];
    float sum[VN];
#pragma unroll
    for (int j = 0; j < VN; ++j) sum[j] = (float)(T)((known ? (float)va[j] : 0.f) + (float)vb[j]);
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int j = 0; j < VN; ++j) sum[j] = scale.of_half(sum[j]);
    } else {
      scale.apply(sum);
    }
    V vo;
#pragma unroll
    for (int j = 0; j < VN; ++j) vo[j] = (T)(u[j] > drop.p ? sum[j] : 0.f);
    store_row(STREAM, reinterpret_cast<V*>(out + row * H) + c, vo);
  }
}

// Any row length: one evaluation per element.
template <typename T>
__global__ __launch_bounds__(256) void embed_dropout_kernel(
    const int64_t* __restrict__ ids, const T* __restrict__ wte,
    const T* __restrict__ wpe, T* __restrict__ out, int64_t rows, int64_t L, int64_t V_, int H,
    DropoutArgs drop) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int64_t tok = ids[row];
  const bool known = (uint64_t)tok < (uint64_t)V_;
  const int64_t pos = row % L;
  for (int c = lane; c < H; c += 64) {
    const T sum = (T)((known ? (float)wte[tok * H + c] : 0.f) + (float)wpe[pos * H + c]);
    unsigned off[1] = {(unsigned)c};
    float z[1] = {(float)sum};
    dropout_apply<1>(drop, off, z);
    out[row * H + c] = (T)z[0];
  }
}


// ---------------------------------------------------------------------------
// LayerNorm (reference: fused_layer_norm_kernel, kernels.py:104-145): fp32
// mean, then fp32 centred biased variance, rstd = 1/sqrt(var + eps),
// z = (x - mean) * rstd * w + b.  CH = 16-byte chunks per lane.
//
// LPR = lanes per row, 64 or 32.  With 32 a wavefront works on two rows at once: for rows of
// 96 chunks (H = 768 in fp16) every lane then has work in every pass -- with 64 lanes a
// quarter of them idle in the second pass -- and twice the rows are in flight per wavefront
// (LayerNorm at the headline: 89 -> 74 us).  The launchers pick 32 when that wastes fewer lanes.
// ---------------------------------------------------------------------------
// OT: type of the output.  fp32 rows may be emitted as fp16, the rounding of a GEMM operand (the
// block functions of fp32 models: the operand is written at once instead of by a pack pass).
template <typename T, int CH, int LPR, typename OT>
__device__ __forceinline__ void layernorm_rows(
    const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ b,
    OT* __restrict__ out, int64_t M, int H, float eps, unsigned block) {
  typedef typename Vec<T>::type V;
  typedef OT OV __attribute__((ext_vector_type(Vec<T>::N)));
  constexpr int VN = Vec<T>::N;
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t row = (int64_t)block * (256 / LPR) + threadIdx.x / LPR;
  if (row >= M) return;
  const int nchunks = H / VN;
  const V* xr = reinterpret_cast<const V*>(x + row * H);
  const V* wv = reinterpret_cast<const V*>(w);
  const V* bv = reinterpret_cast<const V*>(b);
  V t[CH], tw[CH], tb[CH];  // weight and bias chunks, requested with the row: off the tail of the row
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = lane + i * LPR;
    if (c < nchunks) {
      t[i] = __builtin_nontemporal_load(xr + c);
      if (CH <= 4) {
        tw[i] = wv[c];
        tb[i] = bv[c];
      }
    } else {
#pragma unroll
      for (int j = 0; j < VN; ++j) t[i][j] = (T)0.f;
    }
  }
  float d[CH][VN], rstd;
  layernorm_stats<CH, VN, LPR, false>(t, lane, nchunks, H, eps, d, rstd);
  OV* o = reinterpret_cast<OV*>(out + row * H);
  // not a streaming store: the [T, H] output is what the following GEMM reads, two
  // or three times over; it fits the 256 MB memory-side cache, and a GEMM fed from there
  // instead of HBM ran 12 % faster (its operand loads are only one k-tile ahead)
  OV to[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = lane + i * LPR;
    if (c < nchunks) {
      if (CH > 4) {
        tw[i] = wv[c];
        tb[i] = bv[c];
      }
#pragma unroll
      for (int j = 0; j < VN; ++j)
        to[i][j] = (OT)layernorm_apply(d[i][j], rstd, (float)tw[i][j], (float)tb[i][j]);
      pin(to[i]);
    }
  }
  loads_done();
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (lane + i * LPR < nchunks) store_through(o + lane + i * LPR, to[i]);
}

template <typename T, int CH, int LPR, typename OT = T>
__global__ __launch_bounds__(256) void layernorm_vec_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ b,
    OT* __restrict__ out, int64_t M, int H, float eps) {
  layernorm_rows<T, CH, LPR, OT>(x, w, b, out, M, H, eps, blockIdx.x);
}

// Embedding gather and the first LayerNorm in one pass: emb[row,:] = wte[id,:] + wpe[pos,:]
// (rounded to the storage dtype, as embed_vec_kernel stores it) and ln[row,:] = LayerNorm of
// that ROUNDED row, so both outputs are bit-identical to embed_vec_kernel followed by
// layernorm_vec_kernel; the row never leaves the registers in between (fused_embeddings ->
// fused_layer_norm in the reference, gpt.py:166-170 and 40).
template <typename T, int CH, int LPR>
__global__ __launch_bounds__(256) void embed_layernorm_kernel(
    const int64_t* __restrict__ ids, const T* __restrict__ wte, const T* __restrict__ wpe,
    const T* __restrict__ w, const T* __restrict__ b, T* __restrict__ emb, T* __restrict__ out,
    int64_t rows, int64_t L, int64_t V_, int H, float eps, int stream) {
  typedef typename Vec<T>::type V;
  constexpr int VN = Vec<T>::N;
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  if (row >= rows) return;
  const int64_t tok = ids[row];
  const bool known = (uint64_t)tok < (uint64_t)V_;
  const int nchunks = H / VN;
  const V* ar = reinterpret_cast<const V*>(wte + (known ? tok : 0) * H);
  const V* pr = reinterpret_cast<const V*>(wpe + (row % L) * H);
  const V* wv = reinterpret_cast<const V*>(w);
  const V* bv = reinterpret_cast<const V*>(b);
  V* eo = reinterpret_cast<V*>(emb + row * H);
  V e[CH], tw[CH], tb[CH];
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = lane + i * LPR;
    if (c < nchunks) {
      const V va = ar[c], vb = pr[c];
      tw[i] = wv[c];
      tb[i] = bv[c];
#pragma unroll
      for (int j = 0; j < VN; ++j) e[i][j] = (T)((known ? (float)va[j] : 0.f) + (float)vb[j]);
      pin(e[i]);
    } else {
#pragma unroll
      for (int j = 0; j < VN; ++j) e[i][j] = (T)0.f;
    }
  }
  // (no loads_done: the parameters may still be on their way, and in front of the second stores it would be
  // a wait for these)
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (lane + i * LPR < nchunks) store_row(stream, eo + lane + i * LPR, e[i]);  // next read by a GEMM epilogue
  float d[CH][VN], rstd;
  layernorm_stats<CH, VN, LPR, false>(e, lane, nchunks, H, eps, d, rstd);
  V* o = reinterpret_cast<V*>(out + row * H);
#pragma unroll
  for (int i = 0; i < CH; ++i)
    if (lane + i * LPR < nchunks) {
#pragma unroll
      for (int j = 0; j < VN; ++j)
        e[i][j] = (T)layernorm_apply(d[i][j], rstd, (float)tw[i][j], (float)tb[i][j]);
      pin(e[i]);
    }
#pragma unroll
  for (int i = 0; i < CH; ++i)  // as in layernorm_rows: the following GEMM reads it
    if (lane + i * LPR < nchunks) store_through(o + lane + i * LPR, e[i]);
}

// Any H (no alignment requirement): the row is re-read from cache per pass.
template <typename T, typename OT = T>
__global__ __launch_bounds__(256) void layernorm_scalar_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ b,
    OT* __restrict__ out, int64_t M, int H, float eps) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const T* xr = x + row * H;
  float s = 0.f;
  for (int c = lane; c < H; c += 64) s += (float)xr[c];
  const float mean = wave_sum(s) / (float)H;
  float q = 0.f;
  for (int c = lane; c < H; c += 64) {
    const float d = (float)xr[c] - mean;
    q += d * d;
  }
  const float var = wave_sum(q) / (float)H;
  const float rstd = 1.0f / sqrtf(var + eps);
  for (int c = lane; c < H; c += 64) {
    if constexpr (sizeof(T) != sizeof(OT)) {
      // fp32 rows with an fp16 output stand for the fp32 LayerNorm and a conversion: two roundings
      out[row * H + c] = (OT)layernorm_apply((float)xr[c] - mean, rstd, (float)w[c], (float)b[c]);
    } else {
      const float z = ((float)xr[c] - mean) * rstd;
      out[row * H + c] = (OT)(z * (float)w[c] + (float)b[c]);
    }
  }
}

// ---------------------------------------------------------------------------
// Row softmax: fp32 max, exp(x - max), fp32 sum, divide.
// ---------------------------------------------------------------------------
template <typename T, int CH, int LPR>
__global__ __launch_bounds__(256) void softmax_vec_kernel(const T* __restrict__ x,
                                                          T* __restrict__ out,
                                                          int64_t M, int H) {
  typedef typename Vec<T>::type V;
  constexpr int VN = Vec<T>::N;
  const int lane = threadIdx.x & (LPR - 1);
  const int64_t row = (int64_t)blockIdx.x * (256 / LPR) + threadIdx.x / LPR;
  if (row >= M) return;
  const int nchunks = H / VN;
  const V* xr = reinterpret_cast<const V*>(x + row * H);
  float v[CH][VN];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = lane + i * LPR;
    if (c < nchunks) {
      V t = __builtin_nontemporal_load(xr + c);
#pragma unroll
      for (int j = 0; j < VN; ++j) {
        v[i][j] = (float)t[j];
        mx = fmaxf(mx, v[i][j]);
      }
    } else {
#pragma unroll
      for (int j = 0; j < VN; ++j) v[i][j] = -INFINITY;
    }
  }
  mx = group_max<LPR>(mx);
  float s = 0.f;
#pragma unroll
  for (int i = 0; i < CH; ++i) {
#pragma unroll
    for (int j = 0; j < VN; ++j) {
      v[i][j] = __expf(v[i][j] - mx);  // exp(-inf) = 0 for the padding lanes
      s += v[i][j];
    }
  }
  const float inv = 1.0f / group_sum<LPR>(s);
  V* o = reinterpret_cast<V*>(out + row * H);
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = lane + i * LPR;
    if (c < nchunks) {
      V to;
#pragma unroll
      for (int j = 0; j < VN; ++j) to[j] = (T)(v[i][j] * inv);
      __builtin_nontemporal_store(to, o + c);
    }
  }
}

template <typename T>
__global__ __launch_bounds__(256) void softmax_scalar_kernel(const T* __restrict__ x,
                                                             T* __restrict__ out,
                                                             int64_t M, int H) {
  const int lane = threadIdx.x & 63;
  const int64_t row = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= M) return;
  const T* xr = x + row * H;
  float mx = -INFINITY;
  for (int c = lane; c < H; c += 64) mx = fmaxf(mx, (float)xr[c]);
  mx = wave_max(mx);
  float s = 0.f;
  for (int c = lane; c < H; c += 64) s += __expf((float)xr[c] - mx);
  const float inv = 1.0f / wave_sum(s);
  for (int c = lane; c < H; c += 64)
    out[row * H + c] = (T)(__expf((float)xr[c] - mx) * inv);
}

// ---------------------------------------------------------------------------
// GEMM operand packers.  Both produce fp16 rows of Kp (a multiple of 64)
// elements, zero filled beyond K, which is the only operand form the MFMA
// kernel reads.
//   pack_rows:      src[R][K]  -> dst[R][Kp]   (x, or a weight given as [N][K])
//   pack_transpose: src[K][N]  -> dst[N][Kp]   (weight given as [K][N])
// ---------------------------------------------------------------------------
// Rows whose length is a multiple of 8 (so that a chunk of 8 never leaves its row) from a 16-byte
// aligned source: a thread converts 8 elements, 16 bytes out (32 x 300 x 768 floats: 61 us with an
// element and a 64-bit division per thread).
template <typename T>
__global__ __launch_bounds__(256) void pack_rows_vec_kernel(const T* __restrict__ src,
                                                            _Float16* __restrict__ dst,
                                                            int64_t R, unsigned K8, unsigned Kp8, int through) {
  typedef T V __attribute__((ext_vector_type(8)));
  const unsigned rows_per = 256 / Kp8 ? 256 / Kp8 : 1;  // rows a workgroup turn covers
  const unsigned lane_row = Kp8 <= 256 ? threadIdx.x / Kp8 : 0;
  const unsigned c0 = Kp8 <= 256 ? threadIdx.x - lane_row * Kp8 : threadIdx.x;
  if (lane_row >= rows_per) return;
  for (int64_t r = (int64_t)blockIdx.x * rows_per + lane_row; r < R; r += (int64_t)gridDim.x * rows_per)
    for (unsigned c = c0; c < Kp8; c += 256) {
      h8 o;
#pragma unroll
      for (int j = 0; j < 8; ++j) o[j] = (_Float16)0.f;
      if (c < K8) {
        const V v = *reinterpret_cast<const V*>(src + (r * K8 + c) * 8);
#pragma unroll
        for (int j = 0; j < 8; ++j) o[j] = (_Float16)(float)v[j];
      }
      h8* to = reinterpret_cast<h8*>(dst + (r * Kp8 + c) * 8);
      if (through) store_through(to, o);
      else *to = o;
    }
}

// Any row length: an element per thread.
template <typename T>
__global__ __launch_bounds__(256) void pack_rows_kernel(const T* __restrict__ src,
                                                        _Float16* __restrict__ dst,
                                                        int64_t R, int K, int Kp) {
  const int64_t total = R * (int64_t)Kp;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < total;
       i += (int64_t)gridDim.x * 256) {
    const int64_t r = i / Kp;
    const int k = (int)(i - r * Kp);
    dst[i] = k < K ? (_Float16)(float)src[r * K + k] : (_Float16)0.f;
  }
}

// N a multiple of 8 and a 16-byte aligned source: 16-byte accesses on both sides.  A 64 x 64 tile
// goes through LDS as halves; its rows are padded by 2 so that the 8 k-groups x 8 columns a wavefront
// gathers at once lie on different banks.  The launch is bound by one memory round trip each way:
// 768 x 3072 halves from HBM 8.7 -> 3.6 us, 1600 x 6400 18.5 -> 8.3.
//
// Up to two weights in one launch (a block's two, where they are packed on every call): the second
// one's tiles follow the first one's.  Half of a launch of this size is its start and its drain:
// the four weights of a 768-wide layer in two launches take 10.5 us, in four 18.8.
template <typename T>
struct PackArgs {
  const T* src;
  _Float16* dst;
  int K, N, Kp;
  unsigned tiles;  // (Kp / 64) * ceil(N / 64)
};
constexpr int PACK_PITCH = 66;
template <typename T>
__device__ __forceinline__ void pack_transpose_tile(const PackArgs<T>& first, const PackArgs<T>& second,
                                                    _Float16* tile, unsigned block) {
  typedef T V __attribute__((ext_vector_type(8)));
  constexpr int PITCH = PACK_PITCH;
  const bool is_second = block >= first.tiles;
  const unsigned id_ = block - (is_second ? first.tiles : 0);
  const T* __restrict__ src = is_second ? second.src : first.src;
  _Float16* __restrict__ dst = is_second ? second.dst : first.dst;
  const int K = is_second ? second.K : first.K, N = is_second ? second.N : first.N;
  const int Kp = is_second ? second.Kp : first.Kp;
  const unsigned kt = (unsigned)Kp / 64;
  const int k0 = (int)(id_ % kt) * 64, n0 = (int)(id_ / kt) * 64;
  V v[2];
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int id = it * 256 + threadIdx.x, k = k0 + (id >> 3), n = n0 + (id & 7) * 8;
    if (k < K && n < N) v[it] = *reinterpret_cast<const V*>(src + (int64_t)k * N + n);
    else {
#pragma unroll
      for (int j = 0; j < 8; ++j) v[it][j] = (T)0.f;
    }
  }
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int id = it * 256 + threadIdx.x;
    h2* row = reinterpret_cast<h2*>(tile + (id >> 3) * PITCH + (id & 7) * 8);
#pragma unroll
    for (int j = 0; j < 4; ++j) row[j] = h2{(_Float16)(float)v[it][2 * j], (_Float16)(float)v[it][2 * j + 1]};
  }
  __syncthreads();
#pragma unroll
  for (int it = 0; it < 2; ++it) {
    const int id = it * 256 + threadIdx.x, kg = id & 7, n = id >> 3;
    h8 o;
#pragma unroll
    for (int j = 0; j < 8; ++j) o[j] = tile[(kg * 8 + j) * PITCH + n];
    if (n0 + n < N) store_through(reinterpret_cast<h8*>(dst + (int64_t)(n0 + n) * Kp + k0 + kg * 8), o);
  }
}

template <typename T>
__global__ __launch_bounds__(256) void pack_transpose_vec_kernel(PackArgs<T> first, PackArgs<T> second) {
  __shared__ __attribute__((aligned(16))) _Float16 tile[64 * PACK_PITCH];
  pack_transpose_tile(first, second, tile, blockIdx.x);
}

// A block's LayerNorm and the images of its two weights in one launch, the weights' tiles first (they
// are the longer path).  Neither needs the other; together they are bound by HBM (4800 rows x 768 and the
// weights of an MLP: 34 MB in 8.0 us) and a launch's start and drain fall away: forward of 16 x 300 tokens
// in training mode, 124M, 1742 -> 1724 us.
template <typename T, int CH, int LPR>
__global__ __launch_bounds__(256) void layernorm_pack_kernel(
    const T* __restrict__ x, const T* __restrict__ w, const T* __restrict__ b,
    _Float16* __restrict__ out, int64_t M, int H, float eps, unsigned tiles, PackArgs<T> first,
    PackArgs<T> second) {
  __shared__ __attribute__((aligned(16))) _Float16 tile[64 * PACK_PITCH];
  if (blockIdx.x < tiles) pack_transpose_tile(first, second, tile, blockIdx.x);
  else layernorm_rows<T, CH, LPR, _Float16>(x, w, b, out, M, H, eps, blockIdx.x - tiles);
}

// Any shape: an element per thread and turn.
template <typename T>
__global__ __launch_bounds__(256) void pack_transpose_kernel(const T* __restrict__ src,
                                                             _Float16* __restrict__ dst,
                                                             int K, int N, int Kp) {
  __shared__ _Float16 tile[64][65];
  const int k0 = blockIdx.x * 64, n0 = blockIdx.y * 64;
  const int tx = threadIdx.x & 63, ty = threadIdx.x >> 6;
  for (int i = ty; i < 64; i += 4) {
    const int k = k0 + i, n = n0 + tx;
    tile[i][tx] = (k < K && n < N) ? (_Float16)(float)src[(int64_t)k * N + n]
                                   : (_Float16)0.f;
  }
  __syncthreads();
  for (int i = ty; i < 64; i += 4) {
    const int n = n0 + i, k = k0 + tx;
    if (n < N) dst[(int64_t)n * Kp + k] = tile[tx][i];
  }
}

// The dropout mask as bits, by the generator's offset: one word of 32 offsets per thread.  Every
// dropout of a training forward but the embedding's uses one seed and an offset that counts flat
// indices from 0, so one mask serves all its layers; what bounds the kernel is the generator:
// 14.7 M offsets (4800 x 3072) 24 us.
__global__ __launch_bounds__(256) void dropout_mask_kernel(unsigned* __restrict__ mask, int64_t words,
                                                           DropoutArgs drop) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= words) return;
  unsigned bits = 0;
#pragma unroll 1
  for (int b = 0; b < 32; b += 8) {
    unsigned off[8];
    float u[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) off[j] = (unsigned)(i * 32) + (unsigned)(b + j);
    philox_uniform<8>(drop, off, u);
#pragma unroll
    for (int j = 0; j < 8; ++j) bits |= (u[j] > drop.p ? 1u : 0u) << (b + j);
  }
  mask[i] = bits;
}

// ---------------------------------------------------------------------------
// Host launchers
// ---------------------------------------------------------------------------
void launch_dropout_mask(void* mask, int64_t words, Dropout drop, hipStream_t st) {
  const DropoutArgs d = {drop.p, (unsigned)drop.seed, (unsigned)(drop.seed >> 32)};
  hipLaunchKernelGGL(dropout_mask_kernel, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, st,
                     (unsigned*)mask, words, d);
}

template <typename T>
static int launch_embed_t(const int64_t* ids, const void* wte, const void* wpe,
                          void* out, int64_t rows, int64_t L, int64_t V, int H, Dropout drop,
                          hipStream_t st) {
  const bool aligned = (H % Vec<T>::N) == 0 && ((uintptr_t)wte % 16) == 0 &&
                       ((uintptr_t)wpe % 16) == 0 && ((uintptr_t)out % 16) == 0;
  const unsigned grid = (unsigned)((rows + 3) / 4);
  const int64_t bytes = rows * H * (int64_t)sizeof(T);
  const int stream = bytes > kStreamBytes;
  // The reference runs the dropout even at p = 0 (kernels.py:70), where it is the identity
  // unless a column's uniform is exactly 0; for the default seed no column below 2^20 has
  // that, so only other seeds or wider rows need the generator at p = 0.
  if (drop.p != 0.0f || drop.seed != 1337 || H > (1 << 20)) {
    const DropoutArgs d = {drop.p, (unsigned)drop.seed, (unsigned)(drop.seed >> 32)};
    if (aligned) {
      const int nchunks = H / Vec<T>::N, rows_per = nchunks < 256 ? 256 / nchunks : 1;
      const int64_t groups = (rows + rows_per - 1) / rows_per;
      const dim3 vgrid((unsigned)(groups < 768 ? groups : 768), (unsigned)((nchunks + 255) / 256));
      // a thread's rows follow one another, so stores written through hold up the loads of the next: only
      // where it has one or two (7 x 211 x 768 halves non-temporal 5.3, through 5.1 us; 16 x 300 7.2, 7.6; 512 x 300
      // 101, 128)
      if (bytes > (4 << 20))
        hipLaunchKernelGGL((embed_dropout_vec_kernel<T, true>), vgrid, dim3(256), 0, st, ids, (const T*)wte,
                           (const T*)wpe, (T*)out, rows, L, V, H, d);
      else
        hipLaunchKernelGGL((embed_dropout_vec_kernel<T, false>), vgrid, dim3(256), 0, st, ids, (const T*)wte,
                           (const T*)wpe, (T*)out, rows, L, V, H, d);
      return 0;
    }
    hipLaunchKernelGGL(embed_dropout_kernel<T>, dim3(grid), dim3(256), 0, st, ids,
                       (const T*)wte, (const T*)wpe, (T*)out, rows, L, V, H, d);
    return 0;
  }
  if (aligned)
    if (lanes_per_row(H / Vec<T>::N) == 32)
      hipLaunchKernelGGL((embed_vec_kernel<T, 32>), dim3((unsigned)((rows + 7) / 8)), dim3(256), 0,
                         st, ids, (const T*)wte, (const T*)wpe, (T*)out, rows, L, V, H, stream);
    else
      hipLaunchKernelGGL((embed_vec_kernel<T, 64>), dim3(grid), dim3(256), 0, st, ids,
                         (const T*)wte, (const T*)wpe, (T*)out, rows, L, V, H, stream);
  else
    hipLaunchKernelGGL(embed_scalar_kernel<T>, dim3(grid), dim3(256), 0, st, ids,
                       (const T*)wte, (const T*)wpe, (T*)out, rows, L, V, H);
  return 0;
}

int launch_embed(const int64_t* ids, const void* wte, const void* wpe, void* out,
                 int64_t rows, int64_t L, int64_t V, int H, Dropout drop, bool f16,
                 hipStream_t st) {
  return f16 ? launch_embed_t<_Float16>(ids, wte, wpe, out, rows, L, V, H, drop, st)
             : launch_embed_t<float>(ids, wte, wpe, out, rows, L, V, H, drop, st);
}

template <typename T, typename OT, int CH>
static void ln_go(const void* x, const void* w, const void* b, void* out, int64_t M,
                  int H, float eps, int lpr, hipStream_t st) {
  if (lpr == 32)
    hipLaunchKernelGGL((layernorm_vec_kernel<T, CH, 32, OT>), dim3((unsigned)((M + 7) / 8)),
                       dim3(256), 0, st, (const T*)x, (const T*)w, (const T*)b,
                       (OT*)out, M, H, eps);
  else
    hipLaunchKernelGGL((layernorm_vec_kernel<T, CH, 64, OT>), dim3((unsigned)((M + 3) / 4)),
                       dim3(256), 0, st, (const T*)x, (const T*)w, (const T*)b,
                       (OT*)out, M, H, eps);
}

template <typename T, typename OT>
static int launch_layernorm_t(const void* x, const void* w, const void* b, void* out,
                              int64_t M, int H, float eps, hipStream_t st) {
  constexpr int VN = Vec<T>::N;
  const bool aligned = (H % VN) == 0 && ((uintptr_t)x % 16) == 0 &&
                       ((uintptr_t)w % 16) == 0 && ((uintptr_t)b % 16) == 0 &&
                       ((uintptr_t)out % 16) == 0;
  const int lpr = lanes_per_row(H / VN);
  const int need = aligned ? (H / VN + lpr - 1) / lpr : 1 << 30;
  if (need <= 1) ln_go<T, OT, 1>(x, w, b, out, M, H, eps, lpr, st);
  else if (need <= 2) ln_go<T, OT, 2>(x, w, b, out, M, H, eps, lpr, st);
  else if (need <= 3) ln_go<T, OT, 3>(x, w, b, out, M, H, eps, lpr, st);
  else if (need <= 4) ln_go<T, OT, 4>(x, w, b, out, M, H, eps, lpr, st);
  else if (need <= 8) ln_go<T, OT, 8>(x, w, b, out, M, H, eps, lpr, st);
  else if (need <= 16) ln_go<T, OT, 16>(x, w, b, out, M, H, eps, lpr, st);
  else if (need <= 32) ln_go<T, OT, 32>(x, w, b, out, M, H, eps, lpr, st);
  else
    hipLaunchKernelGGL((layernorm_scalar_kernel<T, OT>), dim3((unsigned)((M + 3) / 4)),
                       dim3(256), 0, st, (const T*)x, (const T*)w, (const T*)b,
                       (OT*)out, M, H, eps);
  return 0;
}

int launch_layernorm(const void* x, const void* w, const void* b, void* out,
                     int64_t M, int H, float eps, bool f16, bool out_f16, hipStream_t st) {
  if (f16) return launch_layernorm_t<_Float16, _Float16>(x, w, b, out, M, H, eps, st);
  return out_f16 ? launch_layernorm_t<float, _Float16>(x, w, b, out, M, H, eps, st)
                 : launch_layernorm_t<float, float>(x, w, b, out, M, H, eps, st);
}

template <typename T, int CH>
static void sm_go(const void* x, void* out, int64_t M, int H, int lpr, hipStream_t st) {
  if (lpr == 32)
    hipLaunchKernelGGL((softmax_vec_kernel<T, CH, 32>), dim3((unsigned)((M + 7) / 8)),
                       dim3(256), 0, st, (const T*)x, (T*)out, M, H);
  else
    hipLaunchKernelGGL((softmax_vec_kernel<T, CH, 64>), dim3((unsigned)((M + 3) / 4)),
                       dim3(256), 0, st, (const T*)x, (T*)out, M, H);
}

template <typename T>
static int launch_softmax_t(const void* x, void* out, int64_t M, int H,
                            hipStream_t st) {
  constexpr int VN = Vec<T>::N;
  const bool aligned =
      (H % VN) == 0 && ((uintptr_t)x % 16) == 0 && ((uintptr_t)out % 16) == 0;
  const int lpr = lanes_per_row(H / VN);
  const int need = aligned ? (H / VN + lpr - 1) / lpr : 1 << 30;
  if (need <= 1) sm_go<T, 1>(x, out, M, H, lpr, st);
  else if (need <= 2) sm_go<T, 2>(x, out, M, H, lpr, st);
  else if (need <= 3) sm_go<T, 3>(x, out, M, H, lpr, st);
  else if (need <= 4) sm_go<T, 4>(x, out, M, H, lpr, st);
  else if (need <= 8) sm_go<T, 8>(x, out, M, H, lpr, st);
  else if (need <= 16) sm_go<T, 16>(x, out, M, H, lpr, st);
  else if (need <= 32) sm_go<T, 32>(x, out, M, H, lpr, st);
  else
    hipLaunchKernelGGL(softmax_scalar_kernel<T>, dim3((unsigned)((M + 3) / 4)),
                       dim3(256), 0, st, (const T*)x, (T*)out, M, H);
  return 0;
}

int launch_softmax(const void* x, void* out, int64_t M, int H, bool f16,
                   hipStream_t st) {
  return f16 ? launch_softmax_t<_Float16>(x, out, M, H, st)
             : launch_softmax_t<float>(x, out, M, H, st);
}

template <typename T, int CH>
static void eln_go(const int64_t* ids, const void* wte, const void* wpe, const void* w,
                   const void* b, void* emb, void* out, int64_t rows, int64_t L, int64_t V, int H,
                   float eps, int lpr, hipStream_t st) {
  const int stream = 2 * rows * H * (int64_t)sizeof(T) > kStreamBytes;  // both outputs
  if (lpr == 32)
    hipLaunchKernelGGL((embed_layernorm_kernel<T, CH, 32>), dim3((unsigned)((rows + 7) / 8)),
                       dim3(256), 0, st, ids, (const T*)wte, (const T*)wpe, (const T*)w,
                       (const T*)b, (T*)emb, (T*)out, rows, L, V, H, eps, stream);
  else
    hipLaunchKernelGGL((embed_layernorm_kernel<T, CH, 64>), dim3((unsigned)((rows + 3) / 4)),
                       dim3(256), 0, st, ids, (const T*)wte, (const T*)wpe, (const T*)w,
                       (const T*)b, (T*)emb, (T*)out, rows, L, V, H, eps, stream);
}

template <typename T>
static bool launch_embed_layernorm_t(const int64_t* ids, const void* wte, const void* wpe,
                                     const void* w, const void* b, void* emb, void* out,
                                     int64_t rows, int64_t L, int64_t V, int H, float eps,
                                     hipStream_t st) {
  constexpr int VN = Vec<T>::N;
  auto al = [](const void* p) { return ((uintptr_t)p % 16) == 0; };
  if ((H % VN) != 0 || !al(wte) || !al(wpe) || !al(w) || !al(b) || !al(emb) || !al(out))
    return false;
  const int lpr = lanes_per_row(H / VN);
  const int need = (H / VN + lpr - 1) / lpr;
  if (need <= 1) eln_go<T, 1>(ids, wte, wpe, w, b, emb, out, rows, L, V, H, eps, lpr, st);
  else if (need <= 2) eln_go<T, 2>(ids, wte, wpe, w, b, emb, out, rows, L, V, H, eps, lpr, st);
  else if (need <= 3) eln_go<T, 3>(ids, wte, wpe, w, b, emb, out, rows, L, V, H, eps, lpr, st);
  else if (need <= 4) eln_go<T, 4>(ids, wte, wpe, w, b, emb, out, rows, L, V, H, eps, lpr, st);
  else return false;
  return true;
}

// The fused embedding + LayerNorm launch for rows that fit the register-resident form (16-byte
// aligned, at most 4 chunks per lane: H <= 2048 halves / 1024 floats); otherwise false, and
// the caller launches the two kernels one after the other.
bool launch_embed_layernorm(const int64_t* ids, const void* wte, const void* wpe, const void* w,
                            const void* b, void* emb, void* out, int64_t rows, int64_t L,
                            int64_t V, int H, float eps, bool f16, hipStream_t st) {
  return f16 ? launch_embed_layernorm_t<_Float16>(ids, wte, wpe, w, b, emb, out, rows, L, V, H,
                                                  eps, st)
             : launch_embed_layernorm_t<float>(ids, wte, wpe, w, b, emb, out, rows, L, V, H, eps,
                                               st);
}

template <typename T>
static void launch_pack_rows_t(const T* src, _Float16* dst, int64_t R, int K, int Kp, hipStream_t st) {
  if (K % 8 == 0 && ((uintptr_t)src & 15) == 0) {
    const int64_t rows_per = 256 / (Kp / 8) ? 256 / (Kp / 8) : 1;
    int64_t blocks = (R + rows_per - 1) / rows_per;
    if (blocks > 16384) blocks = 16384;
    // written through while the rows are few; one store a thread and turn has nothing behind it to hide the
    // longer way when there are many (product and operand rows in fp32, plain / through: 300 x 768 x 768 6.3 / 6.0 us,
    // 1477 x 1024 x 1024 11.0 / 10.6, 2048 x 1280 x 1280 20.2 / 24.7, 9600 x 768 x 768 28.7 / 29.8)
    const int through = R * Kp * 2 <= (4 << 20);
    hipLaunchKernelGGL(pack_rows_vec_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, st, src, dst, R,
                       (unsigned)(K / 8), (unsigned)(Kp / 8), through);
    return;
  }
  int64_t blocks = (R * (int64_t)Kp + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(pack_rows_kernel<T>, dim3((unsigned)blocks), dim3(256), 0, st, src, dst, R, K, Kp);
}

void launch_pack_rows(const void* src, void* dst, int64_t R, int K, int Kp, bool f16,
                      hipStream_t st) {
  if (f16) launch_pack_rows_t((const _Float16*)src, (_Float16*)dst, R, K, Kp, st);
  else launch_pack_rows_t((const float*)src, (_Float16*)dst, R, K, Kp, st);
}

template <typename T>
static PackArgs<T> pack_args(const void* src, void* dst, int K, int N, int Kp) {
  return {(const T*)src, (_Float16*)dst, K, N, Kp, (unsigned)(Kp / 64) * (unsigned)((N + 63) / 64)};
}

// 16-byte accesses, and no more tiles than a grid has blocks
static bool pack_vec_ok(const void* src, const void* dst, int N, int Kp) {
  return N % 8 == 0 && (((uintptr_t)src | (uintptr_t)dst) & 15) == 0 &&
         (int64_t)(Kp / 64) * ((N + 63) / 64) < (1ll << 22);
}

template <typename T>
static void launch_pack_transpose_t(const T* src, _Float16* dst, int K, int N, int Kp, hipStream_t st) {
  if (pack_vec_ok(src, dst, N, Kp)) {
    const PackArgs<T> a = pack_args<T>(src, dst, K, N, Kp);
    hipLaunchKernelGGL(pack_transpose_vec_kernel<T>, dim3(a.tiles), dim3(256), 0, st, a, PackArgs<T>{});
  } else {
    const dim3 grid((unsigned)(Kp / 64), (unsigned)((N + 63) / 64));
    hipLaunchKernelGGL(pack_transpose_kernel<T>, grid, dim3(256), 0, st, src, dst, K, N, Kp);
  }
}

template <typename T>
static void launch_pack_pair_t(const void* s1, void* d1, int K1, int N1, const void* s2, void* d2, int K2,
                               int N2, hipStream_t st) {
  const PackArgs<T> a = pack_args<T>(s1, d1, K1, N1, K1), b = pack_args<T>(s2, d2, K2, N2, K2);
  hipLaunchKernelGGL(pack_transpose_vec_kernel<T>, dim3(a.tiles + b.tiles), dim3(256), 0, st, a, b);
}

void launch_pack_transpose_pair(const void* s1, void* d1, int K1, int N1, const void* s2, void* d2, int K2,
                                int N2, bool f16, hipStream_t st) {
  if (!pack_vec_ok(s1, d1, N1, K1) || !pack_vec_ok(s2, d2, N2, K2)) {
    if (N1 > 0) launch_pack_transpose(s1, d1, K1, N1, K1, f16, st);
    if (N2 > 0) launch_pack_transpose(s2, d2, K2, N2, K2, f16, st);
  } else if (f16) {
    launch_pack_pair_t<_Float16>(s1, d1, K1, N1, s2, d2, K2, N2, st);
  } else {
    launch_pack_pair_t<float>(s1, d1, K1, N1, s2, d2, K2, N2, st);
  }
}

template <typename T, int CH>
static void lnp_go(const void* x, const void* w, const void* b, void* out, int64_t M, int H, float eps,
                   int lpr, int64_t rows_blocks, const PackArgs<T>& p1, const PackArgs<T>& p2,
                   hipStream_t st) {
  const unsigned tiles = p1.tiles + p2.tiles;
  const dim3 grid((unsigned)(tiles + rows_blocks));
  if (lpr == 32)
    hipLaunchKernelGGL((layernorm_pack_kernel<T, CH, 32>), grid, dim3(256), 0, st, (const T*)x, (const T*)w,
                       (const T*)b, (_Float16*)out, M, H, eps, tiles, p1, p2);
  else
    hipLaunchKernelGGL((layernorm_pack_kernel<T, CH, 64>), grid, dim3(256), 0, st, (const T*)x, (const T*)w,
                       (const T*)b, (_Float16*)out, M, H, eps, tiles, p1, p2);
}

constexpr int kPackChunks = 4;  // of a lane: the registers of longer rows would leave the packing few wavefronts
bool layernorm_packs(int H) { return H <= kPackChunks * 64 * Vec<_Float16>::N; }

// False where the two do not go into one launch: unaligned rows, parameters or weights, long rows, too many blocks.
template <typename T>
static bool launch_layernorm_pack_t(const void* x, const void* w, const void* b, void* out, int64_t M, int H,
                                    float eps, const void* s1, void* d1, int K1, int N1, const void* s2,
                                    void* d2, int K2, int N2, hipStream_t st) {
  constexpr int VN = Vec<T>::N;
  if (H % VN != 0 || (((uintptr_t)x | (uintptr_t)w | (uintptr_t)b | (uintptr_t)out) & 15) != 0 ||
      !pack_vec_ok(s1, d1, N1, K1) || !pack_vec_ok(s2, d2, N2, K2))
    return false;
  const int lpr = lanes_per_row(H / VN), need = (H / VN + lpr - 1) / lpr;
  const int64_t blocks = lpr == 32 ? (M + 7) / 8 : (M + 3) / 4;
  if (need > kPackChunks || blocks >= (1ll << 30)) return false;
  const PackArgs<T> p1 = pack_args<T>(s1, d1, K1, N1, K1), p2 = pack_args<T>(s2, d2, K2, N2, K2);
  if (need <= 1) lnp_go<T, 1>(x, w, b, out, M, H, eps, lpr, blocks, p1, p2, st);
  else if (need <= 2) lnp_go<T, 2>(x, w, b, out, M, H, eps, lpr, blocks, p1, p2, st);
  else if (need <= 3) lnp_go<T, 3>(x, w, b, out, M, H, eps, lpr, blocks, p1, p2, st);
  else lnp_go<T, 4>(x, w, b, out, M, H, eps, lpr, blocks, p1, p2, st);
  return true;
}

void launch_layernorm_pack_pair(const void* x, const void* w, const void* b, void* out, int64_t M, int H,
                                float eps, const void* s1, void* d1, int K1, int N1, const void* s2, void* d2,
                                int K2, int N2, bool f16, hipStream_t st) {
  if (f16 ? launch_layernorm_pack_t<_Float16>(x, w, b, out, M, H, eps, s1, d1, K1, N1, s2, d2, K2, N2, st)
          : launch_layernorm_pack_t<float>(x, w, b, out, M, H, eps, s1, d1, K1, N1, s2, d2, K2, N2, st))
    return;
  launch_pack_transpose_pair(s1, d1, K1, N1, s2, d2, K2, N2, f16, st);
  launch_layernorm(x, w, b, out, M, H, eps, f16, true, st);
}

void launch_pack_transpose(const void* src, void* dst, int K, int N, int Kp, bool f16,
                           hipStream_t st) {
  if (f16) launch_pack_transpose_t((const _Float16*)src, (_Float16*)dst, K, N, Kp, st);
  else launch_pack_transpose_t((const float*)src, (_Float16*)dst, K, N, Kp, st);
}

}  // namespace gptmi
