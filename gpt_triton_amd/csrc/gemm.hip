// fp16 MFMA GEMM with a fused epilogue for gfx950.
//
//   C[M][N] = A[M][Kp] . Bt[N][Kp]^T      (both operands K-contiguous fp16)
//   out     = gelu?(C + bias) + residual  (fp32 math, one rounding at the store)
//
// Reference semantics: fused_ffn_kernel, kernels.py:169-257 (operands rounded to
// fp16, fp32 accumulation, epilogue order bias -> GELU -> residual -> cast) and
// the q/k/v relayout of matmul_and_split_qkv, kernels.py:347-367, which is done
// here by the store instead of by three copies.
//
// This file holds the persistent kernels for problems that fill the chip with 256 x 256 (or 192 x 256) tiles
// (gemm_stream_kernel without and gemm_stream_res_kernel with a residual): one workgroup per CU walks
// tiles and the pipeline runs across tile boundaries.  gemm_tile.hip holds the kernel with one
// workgroup per tile for everything else.  launch_shape (at the end) divides the rows between them.
//
// What they share: LDS rows of 64 halves (128 bytes) filled by direct global->LDS loads, whose
// 16-byte chunks are XOR-swizzled so that the 16 lanes the LDS serves per clock (64 banks x 4 B)
// never share a bank (chunk c of row r at c ^ ((r >> 1) & 7)); v_mfma_f32_16x16x32_f16 issued as
// D[n][m] (weight rows as the first operand), so a lane ends up with 4 consecutive n for one m; fp32
// accumulation over k in 32-wide steps; workgroup ids remapped so that each XCD (ids are dealt
// round-robin over the 8 XCDs) gets a contiguous range of tiles, and inside a group of column tiles
// whose weight panels fit the XCD's L2 the column runs fastest, so the tiles that share a row
// block of A run on the same L2 at the same time.
// Epilogues of the persistent kernels: bias/GELU in the accumulator layout, transposed through a
// wavefront-private LDS slab -- fp16 rounded first (store_wave_tile_h), with a residual the tile of
// it brought into the operand stages by direct loads as these fall free (store_wave_tile_rs), fp32
// output through fp32 slabs (store_wave_tile32).
#include <type_traits>

#include "gemm_common.h"
#include "layernorm.h"

namespace gptmi {

namespace {

// Bias of a wavefront's columns in the accumulator layout: of a 32 x 32 block a lane holds four
// quads, (mh, nh) -> row 16 mh + lane % 16, columns 16 nh + 4 (lane / 16) + 0..3, so two bias quads
// per block: [i][nh] -> columns nw0 + 32 i + 16 nh + 4 (lane / 16) + 0..3.  ONE branch stands around
// all the loads: with a test of ep.bias per load, every load got a basic block of its own and, behind
// it, a wait for everything in flight -- 8 memory round trips per tile, one after the other.
template <typename T, int NB>
__device__ __forceinline__ void load_bias16(const EpiDev& ep, int nw0, int lq,
                                            typename Pack4<T>::type (&raw)[NB][2]) {
  typedef typename Pack4<T>::type P4;
  if (ep.bias) {
    const T* bp = (const T*)ep.bias + (nw0 + lq * 4);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int nh = 0; nh < 2; ++nh) raw[i][nh] = *reinterpret_cast<const P4*>(bp + i * 32 + nh * 16);
  } else {
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int nh = 0; nh < 2; ++nh)
#pragma unroll
        for (int e = 0; e < 4; ++e) raw[i][nh][e] = 0;
  }
}
template <typename P4, int NB>
__device__ __forceinline__ void bias_to_f32_16(const P4 (&raw)[NB][2], f4 (&bias_r)[NB][2]) {
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int nh = 0; nh < 2; ++nh)
#pragma unroll
      for (int e = 0; e < 4; ++e) bias_r[i][nh][e] = (float)raw[i][nh][e];
}

// The dropout mask of a wavefront's 128 x 64 sub-tile: a lane takes the word of row 32 j + lane / 2 and the
// 32 columns from 32 (lane % 2) on.  N and nw0 are multiples of 64, so the words are aligned.
template <int MB>
__device__ __forceinline__ void load_keep(const EpiDev& ep, int64_t mw0, int nw0, int N, int lane,
                                          unsigned (&w)[MB]) {
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    const uint64_t at = (uint64_t)(mw0 + 32 * j + (lane >> 1)) * (uint64_t)N + (uint64_t)(nw0 + 32 * (lane & 1));
    w[j] = *reinterpret_cast<const unsigned*>(ep.keep + (at >> 3));
  }
}
// v where its bit of the low 8 of `bits` is set, +0 elsewhere
__device__ __forceinline__ h8 keep_halves(unsigned bits, h8 v) {
  u4 d = __builtin_bit_cast(u4, v);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    const unsigned lo = (unsigned)__builtin_amdgcn_sbfe((int)bits, 2 * e, 1);
    const unsigned hi = (unsigned)__builtin_amdgcn_sbfe((int)bits, 2 * e + 1, 1);
    d[e] &= (lo & 0xffffu) | (hi & 0xffff0000u);
  }
  return __builtin_bit_cast(h8, d);
}

// fp16 output without residual, whole tile, vector accesses allowed (and head size % 8 == 0 for
// the head-major scatter): bias (+GELU) and the rounding to fp16 happen in the accumulator
// layout, the transposition through the wavefront's slab moves halves (32 rows x 64 columns x
// 2 bytes per pass, 16-byte units XOR-swizzled with row & 7), and a lane gets 8 neighbouring
// columns back: 16-byte stores, 8 lanes per 128-byte line -- half the LDS traffic and half the
// store instructions of the fp32 staging above.  With a residual the sum must stay in fp32 until
// the one rounding, so those epilogues keep the fp32 slabs.
// (NB / 2) * MB * 4 stores per lane.  acc[2 NB][2 MB]: of the 32 x 32 block (i, j) a lane holds the
// quads (mh, nh) = acc[2 i + nh][2 j + mh]: row 16 mh + lane % 16, columns 16 nh + 4 (lane / 16) +
// 0..3, bias_r[i][nh] (see load_bias16).
//
// DROP: dropout behind the GELU, its mask at hand (ep.keep).  The division by 1 - p happens in fp32 in
// the accumulator layout; what is dropped is cleared in the halves on their way out, 8 columns = one byte
// of the mask.  keep_w[j]: the mask word of row 32 j + lane / 2, columns 32 (lane % 2).. (load_keep),
// which a lane takes from the lane that has it.  ffn1 of a training forward of 4800 rows x 768 on this
// kernel instead of 456 tiles of 128 x 256 with the mask (40.5 us a launch): the forward 1724 -> 1542 us.
template <int MB, int NB, bool QKV, bool GELU, bool DROP>
__device__ __forceinline__ void store_wave_tile_h(f4 (&acc)[2 * NB][2 * MB],
                                                  const f4 (&bias_r)[NB][2], const EpiDev& ep, int64_t mw0, int nw0, int N,
                                                  char* slab, int lane, const unsigned (&keep_w)[DROP ? MB : 1]) {
  static_assert(!DROP || NB == 2, "a mask word of 32 of the 64 columns per lane");
  static_assert(NB % 2 == 0, "wave tile must be a multiple of 64 columns");
  // key (row >> 1) & 7: the 32 rows x 2 lanes of one 8-byte write then cover 16 distinct
  // 16-byte slots of the 256-byte bank window twice -- the minimum for 512 bytes
  const int lq = lane >> 4;
  const int frow = lane & 15, fhalf = lq & 1;
  const int fkey = (frow >> 1) & 7;  // rows 16 apart share a key
  const int rrow = lane >> 3, runit = lane & 7;
  const int rkey = rrow >> 1;  // key of row 8 rr + rrow = rkey ^ 4 (rr & 1)
  _Float16* qkv_col[NB / 2];
  unsigned b0 = 0, l0 = 0;
  const unsigned Lu = (unsigned)ep.L;
  const bool step_rows = Lu >= 32u * MB;
  if (QKV) {
#pragma unroll
    for (int i2 = 0; i2 < NB / 2; ++i2)
      qkv_col[i2] = qkv_column_base<_Float16>(ep, nw0 + i2 * 64 + runit * 8);
    const unsigned m_first = (unsigned)mw0 + (unsigned)rrow;
    b0 = m_first / Lu;
    l0 = m_first - b0 * Lu;
  }
  const int64_t batch_stride = (int64_t)ep.heads * ep.L * ep.d;
  const KeepScale scale(DROP ? ep.drop.p : 0.f);
  const unsigned lane_byte_off = ((unsigned)rrow * (unsigned)N + runit * 8) * 2u;
#pragma unroll
  for (int j = 0; j < MB; ++j) {
#pragma unroll
    for (int i2 = 0; i2 < NB / 2; ++i2) {
#pragma unroll
      for (int ii = 0; ii < 2; ++ii)
#pragma unroll
        for (int mh = 0; mh < 2; ++mh) {
          const int i = i2 * 2 + ii;
          float z[8];  // both quads of the row
#pragma unroll
          for (int e = 0; e < 8; ++e) {
            z[e] = acc[2 * i + e / 4][2 * j + mh][e % 4] + bias_r[i][e / 4][e % 4];
            if (GELU) z[e] = gelu_new(z[e]);
          }
          if constexpr (DROP) scale.apply(z);
#pragma unroll
          for (int nh = 0; nh < 2; ++nh) {
            h4 o;
#pragma unroll
            for (int e = 0; e < 4; ++e) o[e] = (_Float16)z[4 * nh + e];
            const int row = 16 * mh + frow;
            const int grp = 2 * nh + (lq >> 1);  // 8-column group of the quad
            *reinterpret_cast<h4*>(slab + row * 128 + (((ii * 4 + grp) ^ fkey) << 4) + fhalf * 8) = o;
          }
        }
      // all four reads first: the stores are assembly with a memory clobber, which no LDS
      // read may cross, so reading inside the store loop would expose one LDS latency per store
      h8 vv[4];
#pragma unroll
      for (int rr = 0; rr < 4; ++rr)
        vv[rr] = *reinterpret_cast<const h8*>(slab + (rr * 8 + rrow) * 128 +
                                              ((runit ^ rkey ^ ((rr & 1) * 4)) << 4));
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        h8 v = vv[rr];
        if constexpr (DROP) {
          const unsigned word =
              __builtin_amdgcn_ds_bpermute((2 * (rr * 8 + rrow) + (runit >> 2)) * 4, (int)keep_w[j]);
          v = keep_halves(word >> ((runit & 3) * 8), v);
        }
        if constexpr (QKV) {
          unsigned b, l;
          if (step_rows) {
            b = b0;
            l = l0 + (unsigned)(j * 32 + rr * 8);
            if (l >= Lu) { l -= Lu; ++b; }
          } else {
            const unsigned m = (unsigned)mw0 + (unsigned)(j * 32 + rr * 8 + rrow);
            b = m / Lu;
            l = m - b * Lu;
          }
          _Float16* dst = qkv_col[i2] + ((int64_t)b * batch_stride + (int64_t)l * ep.d);
          store_at(ep.through, reinterpret_cast<h8*>(dst), v);
        } else {
          // wavefront-uniform 64-bit part in scalar registers + one 32-bit lane offset.  mw0 and
          // nw0 derive from a wavefront index the kernel made provably uniform, so this is
          // scalar arithmetic: a base produced by v_readfirstlane right in front of the store
          // would need five wait states the compiler does not insert for assembly, and the
          // store would now and then go out with the previous base.
          store_base(ep.through, reinterpret_cast<char*>(ep.out) +
                            ((mw0 + j * 32 + rr * 8) * (int64_t)N + nw0 + i2 * 64) * 2,
                        lane_byte_off, v);
        }
      }
    }
  }
}

// fp16 output WITH residual, whole tile, 16-byte accesses allowed: the wavefront's 128 x 64
// residual sub-tile was brought into LDS by direct loads (rows 0..63 at res_lo, rows 64..127 at
// res_hi; 128 bytes per row, 16-byte units XOR-swizzled with (row >> 1) & 7), so the epilogue reads it
// in the accumulator layout, adds it in fp32 behind bias (+GELU) -- the reference's order -- rounds
// once, and finishes like store_wave_tile_h.  No global load is waited for between the stores.
// The residual halves lie in the two operand stages; `mid` runs between row bands 1 and 2, when the stage that held the first half
// is free again (the kernel refills it there).  Younger than the first half's loads when band 0
// starts: the second half's 8 loads.  Younger than the second half's loads when band 2 starts: the
// 8 stores of bands 0 and 1 and, if `refilled`, the 8 operand loads `mid` issued.
// DROP (never with GELU): as in store_wave_tile_h, but cleared in the accumulator layout, in front of the residual.  Training
// forwards of 16800 rows x 768, projection and ffn2 on this kernel instead of one workgroup per tile: 4660 ->
// 4330 us.
template <int MB, int NB, bool GELU, bool DROP, typename Mid>
__device__ __forceinline__ void store_wave_tile_rs(f4 (&acc)[2 * NB][2 * MB], const f4 (&bias_r)[NB][2],
                                                   const EpiDev& ep, int64_t mw0, int nw0, int N,
                                                   const char* res_lo, const char* res_hi,
                                                   char* slab, int lane, bool refilled, Mid&& mid,
                                                   const unsigned (&keep_w)[DROP ? MB : 1]) {
  static_assert(MB == 4 && NB == 2, "128 x 64 sub-tile");
  // accumulators of v_mfma_f32_16x16x32: quad (mh, nh) of the 32 x 32 block (i, j), see
  // store_wave_tile_h<L16>
  const int frow = lane & 15, lq = lane >> 4, fhalf = lq & 1, fkey = (frow >> 1) & 7;
  const int rrow = lane >> 3, runit = lane & 7, rkey = rrow >> 1;
  const unsigned lane_byte_off = ((unsigned)rrow * (unsigned)N + runit * 8) * 2u;
  const KeepScale scale(DROP ? ep.drop.p : 0.f);
#pragma unroll
  for (int j = 0; j < MB; ++j) {
    if (j == 0) wait_vmcnt<8>();
    if (j == 2) {
      mid();
      if (refilled) wait_vmcnt<16>();
      else wait_vmcnt<8>();
    }
    const char* rb = (j < 2 ? res_lo : res_hi) + ((j & 1) * 32 + frow) * 128 + fhalf * 8;
    h4 r[NB][4];
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int mh = g >> 1, nh = g & 1;
        r[i][g] = *reinterpret_cast<const h4*>(rb + mh * 16 * 128 +
                                               (((i * 4 + 2 * nh + (lq >> 1)) ^ fkey) << 4));
      }
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int mh = 0; mh < 2; ++mh) {
        float z[8];  // both quads of the row
#pragma unroll
        for (int e = 0; e < 8; ++e) {
          z[e] = acc[2 * i + e / 4][2 * j + mh][e % 4] + bias_r[i][e / 4][e % 4];
          if (GELU) z[e] = gelu_new(z[e]);
        }
        if constexpr (DROP) {
          const unsigned word =
              (unsigned)__builtin_amdgcn_ds_bpermute((2 * (16 * mh + frow) + i) * 4, (int)keep_w[j]) >> (4 * lq);
          scale.apply(z);
#pragma unroll
          for (int e = 0; e < 8; ++e) z[e] = keep_if(word, 16 * (e / 4) + e % 4, z[e]);
        }
#pragma unroll
        for (int nh = 0; nh < 2; ++nh) {
          h4 o;
#pragma unroll
          for (int e = 0; e < 4; ++e) o[e] = (_Float16)(z[4 * nh + e] + (float)r[i][2 * mh + nh][e]);
          *reinterpret_cast<h4*>(slab + (16 * mh + frow) * 128 +
                                 (((i * 4 + 2 * nh + (lq >> 1)) ^ fkey) << 4) + fhalf * 8) = o;
        }
      }
    h8 vv[4];
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      vv[rr] = *reinterpret_cast<const h8*>(slab + (rr * 8 + rrow) * 128 +
                                            ((runit ^ rkey ^ ((rr & 1) * 4)) << 4));
#pragma unroll
    for (int rr = 0; rr < 4; ++rr)
      store_base(ep.through, reinterpret_cast<char*>(ep.out) +
                        ((mw0 + j * 32 + rr * 8) * (int64_t)N + nw0) * 2,
                    lane_byte_off, vv[rr]);
  }
}

// ---------------------------------------------------------------------------
// Streaming variant of the 256x256x64 kernel (BM = 192: 192x256x64): one workgroup per CU walks tiles
// blockIdx.x, blockIdx.x + gridDim.x, ...  The two operand stages keep alternating across tile
// boundaries, so the first two k-tiles of the NEXT output tile are requested while the current
// one finishes, and the epilogue runs with those loads in flight.  What this removes, per tile
// of ~28 us: the pipeline fill (3.5 k cycles) and the ~2.8 us a CU otherwise sits idle between
// two workgroups while the stores of the one that ended drain (measured: 231 of 256 CUs busy
// on average with one workgroup per tile, 251 when the kernel stores nothing).
//
// LDS: stages at [0, 128 KB), epilogue slabs behind them (8 wavefronts x 4 KB: 32 rows x 64
// halves for fp16 output, store_wave_tile_h; one 32 x 32 fp32 block for fp32 output, 16-byte
// units XOR-swizzled with (row >> 1) & 7), so the epilogue never touches a stage.
//
// Load/store counter.  Loads and stores of a wavefront retire in issue order on this ISA.  The
// loads of the next tile's k-tile 1 are issued BEFORE the epilogue's stores, so waiting for them
// with vmcnt(EPI_STORES) -- the epilogue issues exactly 16 (fp16) or 32 (fp32) stores per lane, 12 or 24 of 192 rows --
// does not wait for the stores' acknowledgements.  The bias is fetched, and waited for, before those loads are issued, so
// that no compiler-placed wait inside the epilogue falls behind them; so are the words of a dropout mask.  Only
// whole row tiles (the last one starts at row M - BM, see persistent_rows), no residual, dropout with its mask
// at hand and an fp16 output behind a GELU: the launcher sends everything else to gemm_tile.hip.
// ---------------------------------------------------------------------------
template <int MB, int NB, typename T, bool QKV, bool GELU>
__device__ __forceinline__ void store_wave_tile32(f4 (&acc)[2 * NB][2 * MB], const f4 (&bias_r)[NB][2],
                                                  const EpiDev& ep, int64_t mw0, int nw0, int N,
                                                  char* slab, int lane) {
  typedef typename Pack4<T>::type P4;
  // accumulators of v_mfma_f32_16x16x32: quad (mh, nh) of the 32 x 32 block (i, j) = row
  // 16 mh + lane % 16, columns 16 nh + 4 (lane / 16) + 0..3
  const int frow = lane & 15, lq = lane >> 4, fkey = (frow >> 1) & 7;
  const int rrow = lane >> 3, runit = lane & 7;
  T* qkv_col[NB];
  unsigned b0 = 0, l0 = 0;
  const unsigned Lu = (unsigned)ep.L;
  const bool step_rows = Lu >= 32u * MB;
  if (QKV) {
#pragma unroll
    for (int i = 0; i < NB; ++i) qkv_col[i] = qkv_column_base<T>(ep, nw0 + i * 32 + runit * 4);
    const unsigned m_first = (unsigned)mw0 + (unsigned)rrow;
    b0 = m_first / Lu;
    l0 = m_first - b0 * Lu;
  }
  const int64_t batch_stride = (int64_t)ep.heads * ep.L * ep.d;
  // byte offset of this lane's (row, 4 columns) inside a 32 x 32 pass of a row-major [.][N] matrix
  const unsigned lane_byte_off = ((unsigned)rrow * (unsigned)N + runit * 4) * (unsigned)sizeof(T);
#pragma unroll
  for (int j = 0; j < MB; ++j) {
#pragma unroll
    for (int i = 0; i < NB; ++i) {
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int mh = g >> 1, nh = g & 1;
        f4 z;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          z[e] = acc[2 * i + nh][2 * j + mh][e] + bias_r[i][nh][e];
          if (GELU) z[e] = gelu_new(z[e]);
        }
        *reinterpret_cast<f4*>(slab + (16 * mh + frow) * 128 + (((4 * nh + lq) ^ fkey) << 4)) = z;
      }
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int row = rr * 8 + rrow;
        const f4 z =
            *reinterpret_cast<const f4*>(slab + row * 128 + ((runit ^ ((row >> 1) & 7)) << 4));
        P4 o;
#pragma unroll
        for (int e = 0; e < 4; ++e) o[e] = (T)z[e];
        if constexpr (QKV) {
          unsigned b, l;
          if (step_rows) {
            b = b0;
            l = l0 + (unsigned)(j * 32 + rr * 8);
            if (l >= Lu) { l -= Lu; ++b; }
          } else {
            const unsigned m = (unsigned)mw0 + (unsigned)(j * 32 + row);
            b = m / Lu;
            l = m - b * Lu;
          }
          T* dst = qkv_col[i] + ((int64_t)b * batch_stride + (int64_t)l * ep.d);
          store_at(ep.through, reinterpret_cast<P4*>(dst), o);
        } else {
          // wavefront-uniform 64-bit part in scalar registers + one 32-bit lane offset
          store_base(ep.through, reinterpret_cast<char*>(ep.out) +
                            ((mw0 + j * 32 + rr * 8) * (int64_t)N + (nw0 + i * 32)) *
                                (int64_t)sizeof(T),
                        lane_byte_off, o);
        }
      }
    }
  }
}

// The weight half of a k-tile where the weight is read as the caller has it, W [K][N] in fp16 with N a multiple of
// 256, instead of from its packed image: 64 rows of k x 256 columns.  16-byte unit u of row r lies at u ^
// key(r), key = 2 (r & 3) + 8 (r >> 3 & 1), so that the 16 rows which a transposing load takes 32 bytes each of
// cover all banks twice, the least for its 512 bytes.  Load n of a thread: row 16 n + tid / 32, which has the
// key of row tid / 32.  A fragment is two transposing loads, k = 32 s + 8 (lane / 16) + 0..3 and 4..7 of columns
// 16 i + lane % 16 of the wavefront's 64: the k of a lane, and so the products' order and bits, are the image's.
// 4800 x 768 x 2304: transposed first 26.9 us, in place 21.7, packed once 20.9.  (In gemm_stream_res_kernel, which
// has no register left, the two loads of a fragment spill.)
struct KnTile {
  unsigned lane_off;
  int N, at;
  __device__ __forceinline__ KnTile(int tid, int lane, int wn, int n) : N(n) {
    auto key = [](int r) { return 2 * (r & 3) + (r & 8); };
    const int r = tid >> 5, lrow = lane & 15, kr = 8 * (lane >> 4) + (lrow >> 2);
    lane_off = (unsigned)r * (unsigned)n * 2u + (unsigned)(((tid & 31) ^ key(r)) << 4);
    at = kr * 512 + (((8 * wn + ((lrow & 3) >> 1)) ^ key(kr)) << 4) + (lrow & 1) * 8;
  }
  __device__ __forceinline__ const char* src(const _Float16* W, int n0, int k, int n) const {
    return (const char*)W + ((size_t)(64 * k + 16 * n) * N + n0) * 2;
  }
  __device__ __forceinline__ h8 fragment(const char* tile, int i, int s) const {
    const char* p = tile + (at ^ (i * 32)) + s * (32 * 512);  // bits 5 and 6 of `at` are the unit's
    const h4 lo = lds_read_tr16(p), hi = lds_read_tr16(p + 4 * 512);
    return h8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  }
};

// T: type of the bias.  OT: type of the output (fp16, or T).  DROP: fp16 output, plain, the mask at hand.
// KN: Bt is the weight [K][N] itself, N a multiple of 256 (see KnTile).
template <int BM, int WM, int WN, typename T, typename OT, bool QKV, bool DROP, bool KN>
__global__ __launch_bounds__(512, 2) void gemm_stream_kernel(
    const _Float16* __restrict__ A, const _Float16* __restrict__ Bt, int M, int N, int Kp,
    int tiles_m, int tiles_n, int group_w, EpiDev ep) {
  constexpr int BN = 256, ROWB = 128, T_ = 512;
  static_assert(WM * WN == 8, "8 wavefronts");
  static_assert(!DROP || (!QKV && sizeof(OT) == 2), "dropout with a plain fp16 output");
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int MB = TM / 32, NB = TN / 32;
  constexpr int A_IT = BM / 64, B_IT = 4, LPT = A_IT + B_IT;  // 16-byte loads per thread per k-tile
  constexpr int STAGE = (BM + BN) * ROWB;                     // 64 KB, 56 of 192 rows
  constexpr int SLABS = 2 * STAGE;                      // epilogue slabs start behind the stages
  constexpr bool HALF_SLABS = sizeof(OT) == 2;          // fp16 output: store_wave_tile_h
  constexpr int EPI_STORES = HALF_SLABS ? MB * NB * 2 : MB * NB * 4;  // stores per lane per epilogue

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  // provably wavefront-uniform, so that everything derived from the wavefront's sub-tile origin
  // (output and residual bases) lives in scalar registers
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int num_tiles = tiles_m * tiles_n;
  const int KT = Kp / 64;  // >= 2 (checked by the launcher)

  // Operand-tile slot s = it * 512 + tid: row it * 64 + tid / 8, 16-byte position tid % 8,
  // which holds source chunk (tid % 8) ^ ((row >> 1) & 7) -- the key does not depend on `it`.
  // M is BM or more, the last row tile starts at M - BM and N is a multiple of 64, so no
  // row is clamped: a load address is a per-tile scalar base (first row of the tile, k-tile
  // offset) plus one of four per-thread 32-bit offsets shared by A and B.
  const int r0 = tid >> 3;
  unsigned lane_off[B_IT];
#pragma unroll
  for (int it = 0; it < B_IT; ++it)
    lane_off[it] = (unsigned)(r0 + it * 64) * (unsigned)Kp * 2u +
                   (unsigned)(((tid & 7) ^ ((r0 >> 1) & 7)) * 16);
  const unsigned wave_off =
      __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem + (unsigned)wave * 1024u);
  auto tile_origin = [&](int vp, int& m0, int& n0) __attribute__((always_inline)) {
    const int tile = xcd_tile(vp, num_tiles);
    const int grp = tile / (tiles_m * group_w);
    const int in_grp = tile - grp * tiles_m * group_w;
    const int grp_w = min(group_w, tiles_n - grp * group_w);
    m0 = min((in_grp / grp_w) * BM, M - BM);
    n0 = (grp * group_w + in_grp % grp_w) * BN;
  };
  // A k-tile is eight 16-byte loads per lane: four for the A rows (three of 192), four for the B rows.  The
  // source of a half is a scalar (first row of the tile, first byte of the k-tile), computed once
  // and not per load: the scalar work of a load that goes between two MFMAs must fit under one.
  auto a_src = [&](int m0, int k) __attribute__((always_inline)) {
    return (const char*)A + ((size_t)m0 * Kp * 2 + (size_t)k * ROWB);
  };
  // Source of load n (64-row block n) of the B tile at n0.  N is a multiple of 64, not
  // necessarily of 256: in the last column tile a block that starts at or past row N loads
  // block 0 again (the shift goes into the scalar source, the lane offsets stay); its products
  // are never stored.
  const size_t blk_bytes = (size_t)64 * Kp * 2;
  const KnTile kn(tid, lane, wn, N);
  auto b_src = [&](int n0, int k, int n) __attribute__((always_inline)) {
    if constexpr (KN) return kn.src(Bt, n0, k, n);
    const int vb = (N - n0) >> 6;  // valid blocks of this tile (4 or more: all)
    const char* p = (const char*)Bt + ((size_t)n0 * Kp * 2 + (size_t)k * ROWB);
    return n < vb ? p : p - n * blk_bytes;
  };
  auto issue_a = [&](int stage, const char* src, int n) __attribute__((always_inline)) {
    lds_dma16_base(src, lane_off[n], wave_off + stage * STAGE + n * T_ * 16);
  };
  auto issue_b = [&](int stage, const char* src, int n) __attribute__((always_inline)) {
    lds_dma16_base(src, KN ? kn.lane_off : lane_off[n], wave_off + stage * STAGE + BM * ROWB + n * T_ * 16);
  };
  auto issue = [&](int stage, int m0, int n0, int k) __attribute__((always_inline)) {
    const char* a = a_src(m0, k);
#pragma unroll
    for (int n = 0; n < A_IT; ++n) issue_a(stage, a, n);
#pragma unroll
    for (int n = 0; n < B_IT; ++n) issue_b(stage, b_src(n0, k, n), n);
  };

  // Fragments of v_mfma_f32_16x16x32_f16: a lane supplies row lane % 16 of a block of 16 rows and
  // the 8 halves of 16-byte unit lane / 16 of a 32-wide k-step.  (Which k goes to which lane group
  // is free as long as both operands agree: k is summed over.)  16 consecutive lanes read 16
  // consecutive rows at one unit: no bank
  // conflicts.
  const int lrow = lane & 15, lq = lane >> 4, fkey = (lrow >> 1) & 7;
  const int a_row_off = (wm * TM + lrow) * ROWB;
  const int b_row_off = BM * ROWB + (wn * TN + lrow) * ROWB;
  // A slice = one 32-wide k-step s times one half h of the sub-tile's rows: MB A blocks (af; a
  // block's register takes the next slice's block as soon as its four MFMAs are issued) times 4 B
  // blocks (bf[s], good for both halves of step s).
  static_assert((TM == 128 || TM == 96) && TN == 64, "128 x 64 or 96 x 64 sub-tiles");
  h8 af[MB], bf[2][4];
  auto frag_a = [&](const char* st, int h, int jl, int s) __attribute__((always_inline)) {
    return *reinterpret_cast<const h8*>(st + a_row_off + (h * (TM / 2) + jl * 16) * ROWB +
                                        (((s * 4 + lq) ^ fkey) << 4));
  };
  auto frag_b = [&](const char* st, int i, int s) __attribute__((always_inline)) {
    if constexpr (KN) return kn.fragment(st + BM * ROWB, i, s);
    return *reinterpret_cast<const h8*>(st + b_row_off + i * 16 * ROWB +
                                        (((s * 4 + lq) ^ fkey) << 4));
  };
  // the fragments of a k-tile's first slice
  auto read_first = [&](int stage) __attribute__((always_inline)) {
    const char* st = smem + stage * STAGE;
#pragma unroll
    for (int jl = 0; jl < MB; ++jl) af[jl] = frag_a(st, 0, jl, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) bf[0][i] = frag_b(st, i, 0);
  };

  int vp = blockIdx.x;
  int m0, n0;
  tile_origin(vp, m0, n0);
  issue(0, m0, n0, 0);
  issue(1, m0, n0, 1);
  wait_vmcnt<LPT>();
  asm volatile("s_barrier" ::: "memory");
  read_first(0);
  int stage = 0;           // stage of the k-tile being multiplied
  bool prev_stored = false;  // this wavefront stored a tile right before the current one

  while (true) {
    const int vp_next = vp + (int)gridDim.x;
    const bool has_next = vp_next < num_tiles;
    int m0_n = 0, n0_n = 0;
    if (has_next) tile_origin(vp_next, m0_n, n0_n);
    const int64_t mw0 = (int64_t)m0 + wm * TM;
    const int nw0 = n0 + wn * TN;
    const bool wave_stores = nw0 < N;  // else this wavefront's 64 columns lie past the edge

    // acc[i][j] = the 16 x 16 block of columns 16 i.., rows 16 j.. of the sub-tile: a lane holds
    // row lane % 16 and the 4 columns 4 (lane / 16) + 0..3
    f4 acc[2 * NB][2 * MB];
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i)
#pragma unroll
      for (int j = 0; j < 2 * MB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

    // One slice, a quarter of a k-tile: 16 (12) MFMAs of 16 x 16 x 32 in eight (six) pairs (a pair takes the
    // matrix pipe as long as one 32 x 32 x 16, and this shape draws less power for the same
    // products: on random operands the chip holds a higher clock).  Behind the pairs, one each, go
    // the fragment reads for slice `rks` of `rstage`: a read issued in the shadow of an MFMA costs
    // no issue time, a burst of them in front of the MFMAs idles the pipe whenever both wavefronts
    // of a SIMD read at once (behind every barrier).  `extra(q)` runs behind pair q.
    auto slice = [&](int, bool fetch, int rstage, int rks, auto&& extra) __attribute__((always_inline)) {
      // this slice is t = rks - 1 (mod 4): k-step s = t / 2, row half h = t % 2
      const int t = (rks + 3) & 3, s = t >> 1, h = t & 1;
      const char* st = smem + rstage * STAGE;
#pragma unroll
      for (int q = 0; q < 2 * MB; ++q) {
        const int jl = q >> 1;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int ii = (q & 1) * 2 + p;
          const int i = (jl & 1) ? 3 - ii : ii;  // one operand changes per MFMA
          acc[i][MB * h + jl] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[s][i], af[jl],
                                                                      acc[i][MB * h + jl], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (fetch) {
          // behind an A block's second pair: the same block of the next slice.  Behind the first
          // pairs: the B blocks of k-step 1 (during slice 1) or of the published k-tile's k-step 0
          // (during slice 3); each B set is idle while it is written.
          if (q & 1) af[jl] = frag_a(st, rks & 1, jl, rks >> 1);
          else if (t == 1) bf[1][jl] = frag_b(st, jl, 1);
          else if (t == 3) bf[0][jl] = frag_b(st, jl, 0);
          if (MB == 3 && q == 1) {  // three pairs' first halves, four B blocks
            if (t == 1) bf[1][3] = frag_b(st, 3, 1);
            else if (t == 3) bf[0][3] = frag_b(st, 3, 0);
          }
        }
        extra(q);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto nothing = [](int) __attribute__((always_inline)) {};
    // A refill dealt one load behind every MFMA of one slice arrives at the texture unit faster
    // than it takes them (64 loads per CU in the time of 16 MFMAs): the wavefronts stall on
    // issue, the MFMAs behind the loads too.  So the A half goes behind every second MFMA of the
    // slice that frees the stage and the B half behind every second MFMA of the next slice.
    const char* b_half[B_IT] = {};  // B half still to be issued into the other stage
    auto with_b_half = [&](int q) __attribute__((always_inline)) {
      if (q & 1) issue_b(stage ^ 1, b_half[q / 2], q / 2);
      else if (MB == 3 && q == 4) issue_b(stage ^ 1, b_half[3], 3);
    };
    // k-slices 0..2 of the k-tile in `stage`; `extra0` goes with the first
    auto first_slices = [&](auto&& extra0) __attribute__((always_inline)) {
      slice(0, true, stage, 1, extra0);
      slice(1, true, stage, 2, nothing);
      slice(0, true, stage, 3, nothing);
    };
    // publish the k-tile in the other stage
    auto publish_next = [&](bool behind_epilogue) __attribute__((always_inline)) {
      // behind an epilogue exactly EPI_STORES stores are younger than the loads waited for
      if (behind_epilogue) wait_vmcnt<EPI_STORES>();
      else wait_vmcnt<0>();
      asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    };
    // The final slice of k-tile kt (not the last): it takes the first fragments of the published
    // k-tile and starts the refill of this stage with the k-tile two ahead -- of this tile, or
    // the first of the next one; behind the last tile it loads this tile's first k-tile again,
    // which nobody reads (no branch around the loads).
    auto final_slice = [&](int kt) __attribute__((always_inline)) {
      const bool own = kt + 2 < KT;
      // (values, not a choice between two captured variables: that would index the closure)
      const bool stay = own || !has_next;
      const int ra = stay ? +m0 : +m0_n, rb = stay ? +n0 : +n0_n;
      const int kk = own ? kt + 2 : 0;
      const char* src = a_src(ra, kk);
      __builtin_amdgcn_sched_barrier(0);
      slice(1, true, stage ^ 1, 0, [&](int q) __attribute__((always_inline)) {
        if (q & 1) issue_a(stage, src, q / 2);
      });
#pragma unroll
      for (int n = 0; n < B_IT; ++n) b_half[n] = b_src(rb, kk, n);
      stage ^= 1;
    };

    // all k-tiles but the last; the first has no half refill to carry
    first_slices(nothing);
    publish_next(prev_stored);
    final_slice(0);
    for (int kt = 1; kt + 1 < KT; ++kt) {
      first_slices(with_b_half);
      publish_next(false);
      final_slice(kt);
    }

    // last k-tile: before its final slice the next tile's first k-tile is published (this
    // stage is free for a refill then); the bias is requested in front of the k-tile and waited
    // for BEFORE the next tile's second k-tile is requested, so that no wait inside the epilogue
    // falls behind those loads.  The next tile's first fragments are read after the epilogue.
    // fp16: requested a whole k-tile before it is needed; fp32 (twice the registers) and with the words
    // of a dropout mask: in front of the last slice
    typename Pack4<T>::type bias_raw[NB][2];
    constexpr bool EARLY_BIAS = sizeof(T) == 2 && !DROP;
    if constexpr (EARLY_BIAS) {
      if (wave_stores) load_bias16<T, NB>(ep, nw0, lq, bias_raw);
    }
    __builtin_amdgcn_sched_barrier(0);
    first_slices(with_b_half);
    if (has_next) publish_next(false);
    unsigned keep_w[DROP ? MB : 1] = {};
    if constexpr (!EARLY_BIAS) {
      if (wave_stores) {
        load_bias16<T, NB>(ep, nw0, lq, bias_raw);
        if constexpr (DROP) {
          int lane_k = lane;  // as lane_e below
          asm volatile("" : "+v"(lane_k));
          load_keep(ep, mw0, nw0, N, lane_k, keep_w);
        }
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    slice(1, false, 0, 0, nothing);
    f4 bias_r[NB][2];
    bias_to_f32_16(bias_raw, bias_r);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g) asm volatile("" : "+v"(bias_r[i][g]));
    if constexpr (DROP) {
#pragma unroll
      for (int j = 0; j < MB; ++j) asm volatile("" : "+v"(keep_w[j]));
    }
    if (has_next) issue(stage, m0_n, n0_n, 1);
    stage ^= 1;

    // ---- epilogue: the next tile's first two k-tiles are landing meanwhile ----
    if (wave_stores) {
      char* slab = smem + SLABS + wave * 4096;
      // The lane id the epilogue derives its addresses from is re-made here from a value the
      // compiler cannot see through: otherwise it computes those addresses once, in front of the
      // tile loop, and they occupy registers through all the k-tiles.
      int lane_e = lane;
      asm volatile("" : "+v"(lane_e));
      if constexpr (HALF_SLABS) {
        if (DROP || ep.gelu)
          store_wave_tile_h<MB, NB, QKV, true, DROP>(acc, bias_r, ep, mw0, nw0, N, slab, lane_e, keep_w);
        else if constexpr (!DROP)
          store_wave_tile_h<MB, NB, QKV, false, false>(acc, bias_r, ep, mw0, nw0, N, slab, lane_e, keep_w);
      } else {
        if (ep.gelu) store_wave_tile32<MB, NB, OT, QKV, true>(acc, bias_r, ep, mw0, nw0, N, slab, lane_e);
        else store_wave_tile32<MB, NB, OT, QKV, false>(acc, bias_r, ep, mw0, nw0, N, slab, lane_e);
      }
    }
    if (!has_next) break;
    read_first(stage);
    prev_stored = wave_stores;
    vp = vp_next;
    m0 = m0_n;
    n0 = n0_n;
  }
  wait_vmcnt<0>();  // the last tile's unread refill
}

// ---------------------------------------------------------------------------
// Streaming kernel WITH a residual (fp16 row-major output, 256 rows or more): the
// persistent pipeline of gemm_stream_kernel, and the residual brought through LDS as in
// store_wave_tile_rs says.  The residual of a tile (128 KB) has no place of its own in LDS, so it
// takes the operand stages as they fall free at the end of the tile, and the next tile's first two
// k-tiles take them back as the epilogue lets go of them:
//
//   final slice of k-tile KT-2   its stage is refilled with residual rows 0..63 of every
//                                wavefront's 128 x 64 sub-tile (8 loads, dealt between the MFMAs)
//   behind k-tile KT-1           barrier, then residual rows 64..127 into that stage (8 loads)
//   epilogue, row bands 0, 1     read the first half, 8 stores
//   between bands 1 and 2        barrier, then the NEXT tile's k-tile 0 into the first stage
//   epilogue, row bands 2, 3     read the second half, 8 stores
//   behind the epilogue          barrier, then the next tile's k-tile 1 into the second stage
//   start of the next tile       k-tile 0 has landed when at most 16 operations are outstanding
//                                (8 stores and 8 loads are younger), barrier, first fragments
//
// A barrier stands in front of every refill because a wavefront's loads write stripes of every
// wavefront's part of a stage.  What this buys over one workgroup per tile: no pipeline fill per
// tile beyond what the epilogue's second half hides, and no idle CU between two workgroups while
// the stores of the one that ended drain.  The launcher sends row tiles that
// do not fill a round of the persistent workgroups to gemm_tile.hip.
// ---------------------------------------------------------------------------
template <int WM, int WN, bool DROP>
__global__ __launch_bounds__(512, 2) void gemm_stream_res_kernel(
    const _Float16* __restrict__ A, const _Float16* __restrict__ Bt, int M, int N, int Kp,
    int tiles_m, int tiles_n, int group_w, EpiDev ep) {
  constexpr int BM = 256, BN = 256, ROWB = 128, T_ = 512, KS = 4;
  static_assert(WM == 2 && WN == 4, "8 wavefronts, 128 x 64 sub-tiles");
  constexpr int TM = BM / WM, TN = BN / WN;
  constexpr int MB = TM / 32, NB = TN / 32;
  constexpr int A_IT = 4, B_IT = 4, LPT = A_IT + B_IT;
  constexpr int STAGE = (BM + BN) * ROWB;  // 64 KB
  constexpr int SLABS = 2 * STAGE;
  static_assert(MB * NB == LPT, "one load per MFMA of a k-slice");

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int num_tiles = tiles_m * tiles_n;
  const int KT = Kp / 64;  // >= 3 (checked by the launcher)

  const int r0 = tid >> 3;
  unsigned lane_off[A_IT];
#pragma unroll
  for (int it = 0; it < A_IT; ++it)
    lane_off[it] = (unsigned)(r0 + it * 64) * (unsigned)Kp * 2u +
                   (unsigned)(((tid & 7) ^ ((r0 >> 1) & 7)) * 16);
  const unsigned smem_base = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem);
  const unsigned wave_off = smem_base + (unsigned)wave * 1024u;
  auto tile_origin = [&](int vp, int& m0, int& n0) __attribute__((always_inline)) {
    const int tile = xcd_tile(vp, num_tiles);
    const int grp = tile / (tiles_m * group_w);
    const int in_grp = tile - grp * tiles_m * group_w;
    const int grp_w = min(group_w, tiles_n - grp * group_w);
    m0 = min((in_grp / grp_w) * BM, M - BM);
    n0 = (grp * group_w + in_grp % grp_w) * BN;
  };
  // the halves of a k-tile (four loads per lane each) and their scalar sources, as in
  // gemm_stream_kernel
  auto a_src = [&](int m0, int k) __attribute__((always_inline)) {
    return (const char*)A + ((size_t)m0 * Kp * 2 + (size_t)k * ROWB);
  };
  // Source of load n (64-row block n) of the B tile at n0.  N is a multiple of 64, not
  // necessarily of 256: in the last column tile a block that starts at or past row N loads
  // block 0 again (the shift goes into the scalar source, the lane offsets stay); its products
  // are never stored.
  const size_t blk_bytes = (size_t)64 * Kp * 2;
  auto b_src = [&](int n0, int k, int n) __attribute__((always_inline)) {
    const int vb = (N - n0) >> 6;  // valid blocks of this tile (4 or more: all)
    const char* p = (const char*)Bt + ((size_t)n0 * Kp * 2 + (size_t)k * ROWB);
    return n < vb ? p : p - n * blk_bytes;
  };
  auto issue_a = [&](int stage, const char* src, int n) __attribute__((always_inline)) {
    lds_dma16_base(src, lane_off[n], wave_off + stage * STAGE + n * T_ * 16);
  };
  auto issue_b = [&](int stage, const char* src, int n) __attribute__((always_inline)) {
    lds_dma16_base(src, lane_off[n], wave_off + stage * STAGE + BM * ROWB + n * T_ * 16);
  };
  auto issue = [&](int stage, int m0, int n0, int k) __attribute__((always_inline)) {
    const char* a = a_src(m0, k);
#pragma unroll
    for (int n = 0; n < A_IT; ++n) issue_a(stage, a, n);
#pragma unroll
    for (int n = 0; n < B_IT; ++n) issue_b(stage, b_src(n0, k, n), n);
  };
  // Residual half h (rows 64 h .. 64 h + 63 of this wavefront's sub-tile) goes to the
  // wavefront's own 8 KB of `stage`: load q fetches 8 rows, lane l the 16-byte unit
  // (l % 8) ^ key of row 8 q + l / 8, key = (row >> 1) & 7 = (l / 16) ^ 4 (q & 1).
  unsigned res_lane_off[2];
#pragma unroll
  for (int odd = 0; odd < 2; ++odd)
    res_lane_off[odd] = ((unsigned)(lane >> 3) * (unsigned)N +
                         (unsigned)(((lane & 7) ^ (lane >> 4) ^ (odd * 4)) * 8)) * 2u;
  auto res_src = [&](int m0, int n0, int h) __attribute__((always_inline)) {
    return (const char*)ep.residual +
           (((int64_t)m0 + wm * TM + h * 64) * N + (n0 + wn * TN)) * 2;
  };
  const int64_t res_step = (int64_t)N * 16;  // 8 rows
  auto issue_res_one = [&](int stage, const char* src, int q) __attribute__((always_inline)) {
    lds_dma16_base(src + q * res_step, res_lane_off[q & 1],
                   smem_base + (unsigned)stage * STAGE + (unsigned)wave * 8192u + q * 1024);
  };

  // Fragments of v_mfma_f32_16x16x32_f16: a lane supplies row lane % 16 of a block of 16 rows and
  // the 8 halves of 16-byte unit lane / 16 of a 32-wide k-step.  (Which k goes to which lane group
  // is free as long as both operands agree: k is summed over.)  16 consecutive lanes read 16
  // consecutive rows at one unit: no bank
  // conflicts.
  const int lrow = lane & 15, lq = lane >> 4, fkey = (lrow >> 1) & 7;
  const int a_row_off = (wm * TM + lrow) * ROWB;
  const int b_row_off = BM * ROWB + (wn * TN + lrow) * ROWB;
  // A slice = one 32-wide k-step s times one half h of the sub-tile's rows: 4 A blocks (af; a
  // block's register takes the next slice's block as soon as its four MFMAs are issued) times 4 B
  // blocks (bf[s], good for both halves of step s).
  static_assert(TM == 128 && TN == 64, "128 x 64 sub-tiles");
  h8 af[4], bf[2][4];
  auto frag_a = [&](const char* st, int h, int jl, int s) __attribute__((always_inline)) {
    return *reinterpret_cast<const h8*>(st + a_row_off + (h * 64 + jl * 16) * ROWB +
                                        (((s * 4 + lq) ^ fkey) << 4));
  };
  auto frag_b = [&](const char* st, int i, int s) __attribute__((always_inline)) {
    return *reinterpret_cast<const h8*>(st + b_row_off + i * 16 * ROWB +
                                        (((s * 4 + lq) ^ fkey) << 4));
  };
  // the fragments of a k-tile's first slice
  auto read_first = [&](int stage) __attribute__((always_inline)) {
    const char* st = smem + stage * STAGE;
#pragma unroll
    for (int jl = 0; jl < 4; ++jl) af[jl] = frag_a(st, 0, jl, 0);
#pragma unroll
    for (int i = 0; i < 4; ++i) bf[0][i] = frag_b(st, i, 0);
  };
  auto barrier_lds = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };

  int vp = blockIdx.x;
  int m0, n0;
  tile_origin(vp, m0, n0);
  issue(0, m0, n0, 0);
  issue(1, m0, n0, 1);
  wait_vmcnt<LPT>();
  asm volatile("s_barrier" ::: "memory");
  read_first(0);
  int stage = 0;  // stage of the k-tile being multiplied

  while (true) {
    const int vp_next = vp + (int)gridDim.x;
    const bool has_next = vp_next < num_tiles;
    int m0_n = 0, n0_n = 0;
    if (has_next) tile_origin(vp_next, m0_n, n0_n);
    const int64_t mw0 = (int64_t)m0 + wm * TM;
    const int nw0 = n0 + wn * TN;
    // false: this wavefront's 64 columns lie past the edge -- it loads operands and keeps the
    // barriers, and has no residual, bias or output of its own
    const bool wave_stores = nw0 < N;

    // acc[i][j] = the 16 x 16 block of columns 16 i.., rows 16 j.. of the sub-tile: a lane holds
    // row lane % 16 and the 4 columns 4 (lane / 16) + 0..3
    f4 acc[2 * NB][2 * MB];
#pragma unroll
    for (int i = 0; i < 2 * NB; ++i)
#pragma unroll
      for (int j = 0; j < 2 * MB; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

    // One slice, as in gemm_stream_kernel: eight pairs of MFMAs, the fragment reads for slice
    // `rks` of `rstage` behind them, `extra(q)` behind pair q.
    auto slice = [&](int, bool fetch, int rstage, int rks, auto&& extra) __attribute__((always_inline)) {
      // this slice is t = rks - 1 (mod 4): k-step s = t / 2, row half h = t % 2
      const int t = (rks + 3) & 3, s = t >> 1, h = t & 1;
      const char* st = smem + rstage * STAGE;
#pragma unroll
      for (int q = 0; q < 8; ++q) {
        const int jl = q >> 1;
#pragma unroll
        for (int p = 0; p < 2; ++p) {
          const int ii = (q & 1) * 2 + p;
          const int i = (jl & 1) ? 3 - ii : ii;  // one operand changes per MFMA
          acc[i][4 * h + jl] = __builtin_amdgcn_mfma_f32_16x16x32_f16(bf[s][i], af[jl],
                                                                      acc[i][4 * h + jl], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (fetch) {
          // behind an A block's second pair: the same block of the next slice.  Behind the first
          // pairs: the B blocks of k-step 1 (during slice 1) or of the published k-tile's k-step 0
          // (during slice 3); each B set is idle while it is written.
          if (q & 1) af[jl] = frag_a(st, rks & 1, jl, rks >> 1);
          else if (t == 1) bf[1][jl] = frag_b(st, jl, 1);
          else if (t == 3) bf[0][jl] = frag_b(st, jl, 0);
        }
        extra(q);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    auto nothing = [](int) __attribute__((always_inline)) {};
    // The three slices in front of a k-tile's last.  `extra0` deals the second half of the
    // refill that the slice before started: four loads there, four here, because eight behind
    // the MFMAs of one slice arrive faster than the texture unit takes them.
    auto first_slices = [&](auto&& extra0) __attribute__((always_inline)) {
      slice(0, true, stage, 1, extra0);
      slice(1, true, stage, 2, nothing);
      slice(0, true, stage, 3, nothing);
    };
    auto publish_next = [&]() __attribute__((always_inline)) {
      wait_vmcnt<0>();
      barrier_lds();
    };
    const char* b_half[B_IT] = {};  // B half still to be issued into the other stage
    auto with_b_half = [&](int q) __attribute__((always_inline)) {
      if (q & 1) issue_b(stage ^ 1, b_half[q / 2], q / 2);
    };
    // the final slice of a k-tile in front of the last but one: it takes the first fragments of
    // the published k-tile and starts the refill of this stage with the k-tile two ahead
    auto final_slice = [&](int kt) __attribute__((always_inline)) {
      const char* src = a_src(m0, kt + 2);
      __builtin_amdgcn_sched_barrier(0);
      slice(1, true, stage ^ 1, 0, [&](int q) __attribute__((always_inline)) {
        if (q & 1) issue_a(stage, src, q / 2);
      });
#pragma unroll
      for (int n = 0; n < B_IT; ++n) b_half[n] = b_src(n0, kt + 2, n);
      stage ^= 1;
    };

    // All k-tiles but the last two (KT >= 3, checked by the launcher): publish the next one (its
    // loads are the only ones in flight), refill this stage.  The first has no half refill to
    // carry.
    first_slices(nothing);
    publish_next();
    final_slice(0);
    for (int kt = 1; kt + 2 < KT; ++kt) {
      first_slices(with_b_half);
      publish_next();
      final_slice(kt);
    }
    // k-tile KT-2: its stage takes the first half of the residual
    const char* res0 = res_src(m0, n0, 0);
    first_slices(with_b_half);
    publish_next();
    slice(1, true, stage ^ 1, 0, [&](int q) __attribute__((always_inline)) {
      if ((q & 1) && wave_stores) issue_res_one(stage, res0, q / 2);
    });
    stage ^= 1;

    // last k-tile; its first slice carries the rest of the residual's first half, and behind its
    // fragment reads the stage is free for the second half.  The bias is requested in front of
    // the last slice and waited for behind it, before those loads are issued, so that no wait
    // the compiler places falls behind them.
    first_slices([&](int q) __attribute__((always_inline)) {
      if ((q & 1) && wave_stores) issue_res_one(stage ^ 1, res0, 4 + q / 2);
    });
    h4 bias_raw[NB][2];
    // all 4 loads in flight under the last slice
    if (wave_stores) load_bias16<_Float16, NB>(ep, nw0, lq, bias_raw);
    unsigned keep_w[DROP ? MB : 1] = {};
    if constexpr (DROP) {
      int lane_k = lane;  // addresses made here, not kept through the tile loop
      asm volatile("" : "+v"(lane_k));
      if (wave_stores) load_keep(ep, mw0, nw0, N, lane_k, keep_w);
    }
    __builtin_amdgcn_sched_barrier(0);
    slice(1, false, 0, 0, nothing);
    f4 bias_r[NB][2];
    bias_to_f32_16(bias_raw, bias_r);
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int g = 0; g < 2; ++g) asm volatile("" : "+v"(bias_r[i][g]));
    if constexpr (DROP) {
#pragma unroll
      for (int j = 0; j < MB; ++j) asm volatile("" : "+v"(keep_w[j]));
    }
    barrier_lds();  // every wavefront has read the last k-tile's fragments
    if (wave_stores) {
      const char* res1 = res_src(m0, n0, 1);
#pragma unroll
      for (int q = 0; q < 8; ++q) issue_res_one(stage, res1, q);
    }
    stage ^= 1;  // now the stage of k-tile KT-2: the residual's first half, then the next tile's k-tile 0

    // ---- epilogue ----
    if (wave_stores) {
      const char* res_lo = smem + stage * STAGE + wave * 8192;
      const char* res_hi = smem + (stage ^ 1) * STAGE + wave * 8192;
      char* slab = smem + SLABS + wave * 4096;
      auto mid = [&]() __attribute__((always_inline)) {
        if (has_next) {
          barrier_lds();  // nobody reads the first half any more
          issue(stage, m0_n, n0_n, 0);
        }
      };
      if (DROP || !ep.gelu)
        store_wave_tile_rs<MB, NB, false, DROP>(acc, bias_r, ep, mw0, nw0, N, res_lo, res_hi, slab, lane,
                                                has_next, mid, keep_w);
      else if constexpr (!DROP)
        store_wave_tile_rs<MB, NB, true, false>(acc, bias_r, ep, mw0, nw0, N, res_lo, res_hi, slab, lane,
                                                has_next, mid, keep_w);
    } else if (has_next) {
      barrier_lds();  // the barrier and the refill of `mid`
      issue(stage, m0_n, n0_n, 0);
    }
    if (!has_next) break;
    barrier_lds();  // nobody reads the second half any more
    issue(stage ^ 1, m0_n, n0_n, 1);
    // the next tile's k-tile 0: younger are the 8 stores of row bands 2 and 3 (of a wavefront
    // that stores) and the 8 loads above
    if (wave_stores) wait_vmcnt<16>();
    else wait_vmcnt<8>();
    asm volatile("s_barrier" ::: "memory");
    read_first(stage);
    vp = vp_next;
    m0 = m0_n;
    n0 = n0_n;
  }
}

template <int BM, typename T, typename OT, bool QKV, bool DROP = false, bool KN = false>
int launch_stream(const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                  hipStream_t st) {
  auto kern = gemm_stream_kernel<BM, 2, 4, T, OT, QKV, DROP, KN>;
  constexpr int smem = 2 * (BM + 256) * 128 + 8 * 4096;  // two stages + the epilogue slabs: 160 KB, or 144
  static bool attr_done = false;  // idempotent; a race only repeats the call
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) {
      set_error("hipFuncSetAttribute(%d bytes LDS): %s", smem, hipGetErrorString(e));
      return -4;
    }
    attr_done = true;
  }
  const int num_cus = cu_count();
  if (num_cus < 0) return num_cus;
  const int tiles_m = (int)((M + BM - 1) / BM), tiles_n = (N + 255) / 256;
  const int num_tiles = tiles_m * tiles_n;
  const int group_w = column_group(M, N, Kp, QKV, BM, 256, num_cus);
  const int grid = num_tiles < num_cus ? num_tiles : num_cus;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(512), smem, st, (const _Float16*)A,
                     (const _Float16*)Bt, (int)M, N, Kp, tiles_m, tiles_n, group_w, ep);
  return 0;
}

template <bool DROP>
int launch_stream_res(const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                      hipStream_t st) {
  auto kern = gemm_stream_res_kernel<2, 4, DROP>;
  constexpr int smem = 2 * 512 * 128 + 8 * 4096;  // 160 KB: two stages + the epilogue slabs
  static bool attr_done = false;  // idempotent; a race only repeats the call
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, smem);
    if (e != hipSuccess) {
      set_error("hipFuncSetAttribute(%d bytes LDS): %s", smem, hipGetErrorString(e));
      return -4;
    }
    attr_done = true;
  }
  const int num_cus = cu_count();
  if (num_cus < 0) return num_cus;
  const int tiles_m = (int)((M + 255) / 256), tiles_n = (N + 255) / 256;
  const int num_tiles = tiles_m * tiles_n;
  const int group_w = column_group(M, N, Kp, false, 256, 256, num_cus);
  const int grid = num_tiles < num_cus ? num_tiles : num_cus;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(512), smem, st, (const _Float16*)A,
                     (const _Float16*)Bt, (int)M, N, Kp, tiles_m, tiles_n, group_w, ep);
  return 0;
}

// Cost in microseconds of a persistent launch over `tiles` tiles of 256 or 192 rows x 256, in the terms of the
// cost model of gemm_tile.hip: every workgroup walks ceil(tiles / CUs) of them, and tile and k-slice take
// longer the more of the chip works (L2 and clock).  Fitted to the same products from 256 rows on; the tiles of 192
// rows relative to those of 256, at 181 sizes from 256 to 26000 rows (2 % off; of the two the one that the
// model takes is the faster one, 6 % faster on average than 256 rows always).
inline float stream_cost(int64_t tiles, int Kp, bool res, int cus, int bm) {
  const float rounds = (float)((tiles + cus - 1) / cus), fill = (float)tiles / (float)cus, k = (float)(Kp / 64);
  if (bm == 192) return 1.67f + rounds * 2.82f + fill * 0.98f + k * (0.853f * rounds + 0.488f * fill);
  return res ? rounds * 7.42f + k * (0.787f * rounds + 0.780f * fill)
             : 1.67f + rounds * 4.70f + fill * 1.63f + k * (0.917f * rounds + 0.659f * fill);
}

// Whether the two matrices of M x N elements share an address.
inline bool overlap(const void* a, const void* b, int64_t M, int N, size_t elem) {
  const uintptr_t p = (uintptr_t)a, q = (uintptr_t)b;
  return (p < q ? q - p : p - q) < (uintptr_t)M * (uintptr_t)N * elem;
}

// Whether the persistent kernel, without a residual, takes the weight [K][N] as it stands (see gemm_reads_kn).
inline bool stream_reads_kn(int64_t M, int N) { return N % 256 == 0 && M <= 32768; }

// Divides the rows between the persistent kernel and the tile kernel.  The persistent kernel takes
// 256-row tiles: all rows, as many tiles as fill whole rounds of the CUs (every workgroup walks
// ceil(tiles / CUs) tiles, so a few tiles beyond a whole number of rounds cost a full round: the
// headline's ffn1 has 7200 tiles = 28 rounds + 32, 597 of its 600 row tiles stay), or none, whichever
// the cost model says is the fastest; the rows that are left follow in a launch of the tile kernel.
// All rows also where they are no multiple of 256: the last row tile starts at row M - 256, and the rows
// that it shares with the tile in front of it are formed twice, from the same operands in the same order,
// so both store the same bits (4800 x 3072 x 768 with GELU: 25.2 us by itself and 29.7 within a forward, 35.1 on
// the tile kernel; 3885 x 1024 x 4096 35.2, 43.6; a second launch for the rows beyond a multiple costs 6 us and more).  Not with an output
// over its own residual, which the second pass would read changed: whole row tiles and a launch behind them.
// It needs N a multiple of 64 (the wavefronts of the last column tile whose 64 columns lie past the
// edge store nothing), two k-tiles (three with a residual), vector epilogues, and dropout only with its
// mask at hand and an fp16 output, behind a GELU or in front of a residual (the two products of a block that
// have one).
// Tiles of 192 rows move 17 % more bytes a product and lose 5 % of the rate, but leave fewer CUs without a tile where
// those of 256 fill the rounds badly (fp16, 256 / 192 rows, us: 4800 x 2304 x 768, 171 / 225 tiles, 23.3 / 21.7; 3885 x
// 3072 x 1024, 192 / 252, 32.3 / 29.8; 4000 x 3072 x 768 25.7 / 22.7; 9600 x 2304 x 768, 342 / 450, 44.0 / 38.7, and 43.5
// with the rows beyond one round on the tile kernel; 12000 x 3072 x 768, 564 / 756, 73.3 / 64.9; 4800 x 3072 x 768, 228 /
// 300, 27.8 / 37.8).  Without a residual and without dropout, up to 6 rounds, beyond which there is nothing to gain.
// Nor where the rows that those of 256 leave to the tile kernel get a tile that divides K: the sums of its two or four groups
// are the more exact ones (K 3072 and more, relative to 64 bits 2.5e-7 against 3.5e-7), and no row is to lose them
// (7200 x 1088 x 4352, the last rows of 11384 x 3072 x 768; one in 55 of the sizes of 192 rows, which then take 2 % longer).
// kn: whether the weight can be read in place is asked (gemm_reads_kn), or it is: where the persistent kernel cannot, what
// tiles of 192 rows save is less than the image costs.  The image of such a weight takes them only with whole sums everywhere,
// which are those of the plan without them: a weight and its image give the same bits.
// Sets *head to the number of rows for the persistent kernel and *bm to its tiles' rows.
template <typename T, typename OT, bool QKV>
int persistent_rows(int64_t M, int N, int Kp, const EpiDev& ep, int64_t* head, int* bm, bool kn = false) {
  const bool res = !QKV && ep.residual != nullptr;
  const bool drop = ep.drop.p > 0.f;
  const bool drop_ok = !QKV && sizeof(OT) == 2 && ep.keep != nullptr && ((uintptr_t)ep.keep & 3) == 0 &&
                       (ep.gelu != 0) != res;
  const bool persistent =
      M >= 256 && N >= 256 && N % 64 == 0 && Kp >= (res ? 192 : 128) && Kp <= (1 << 21) && ep.vec_ok &&
      (sizeof(OT) == 4 || ep.vec8_ok) && (!drop || drop_ok) &&
      (!res || (sizeof(T) == 2 && (((uintptr_t)ep.residual) & 15) == 0));
  *head = 0;
  *bm = 256;
  if (!persistent) return 0;
  const int cus = cu_count();
  if (cus < 0) return cus;
  const int64_t tiles_n = (N + 255) / 256;
  const int64_t all = res && overlap(ep.out, ep.residual, M, N, sizeof(OT)) ? M / 256 * 256 : M;
  if (drop && all != M) return 0;  // all or none: the mask counts from row 0
  const int64_t tiles = (all + 255) / 256 * tiles_n;
  // Two whole rounds and more: always persistent.  Under a load that long the chip's clock falls, and
  // with it the tile kernel, which moves more bytes per product (65536 x 1600 x 1600 with a residual:
  // 336 against 419 us, and 2.4 rounds of 20480 x 1600 x 6400 430 against 445; one round and a bit,
  // 20480 x 1024 x 4096, is the other way round, 196 against 183).
  float least = tiles >= 2 * (int64_t)cus ? INFINITY : gemm_tile_cost(M, N, Kp, cus);
  auto one_sum = [&](int64_t rows) { return rows == M || gemm_tile_split(M - rows, N, Kp, cus) == 1; };
  for (const int tm : {256, 192}) {
    if (tm == 192 && (res || drop || tiles > 6 * (int64_t)cus || (kn && !stream_reads_kn(M, N)))) break;
    if (tm == 192 && !one_sum(*head)) break;
    // rows of the row tiles that fill whole rounds
    const int64_t whole = drop ? all : (all + tm - 1) / tm * tiles_n / cus * cus / tiles_n * tm;
    for (const int64_t rows : {all, whole < all ? whole : all}) {
      if (rows == 0) continue;
      float c = stream_cost((rows + tm - 1) / tm * tiles_n, Kp, res, cus, tm);
      if (rows < M) c += 1.0f + gemm_tile_cost(M - rows, N, Kp, cus);
      if (c < least && (tm == 256 || stream_reads_kn(M, N) || one_sum(rows))) least = c, *head = rows, *bm = tm;
    }
  }
  return 0;
}

// The epilogue of the rows from `head` on.
template <typename T, typename OT, bool QKV>
EpiDev tail_epi(const EpiDev& ep, int64_t head, int N) {
  EpiDev tail = ep;
  if (QKV) {
    tail.m_off = ep.m_off + (int)head;
  } else {
    tail.out = (OT*)ep.out + head * N;
    if (ep.residual) tail.residual = (const T*)ep.residual + head * N;
  }
  return tail;
}

template <typename T, typename OT, bool QKV, bool KN = false>
int launch_shape(const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                 hipStream_t st) {
  const bool res = !QKV && ep.residual != nullptr;
  int64_t m_head;
  int bm;
  if (const int rc = persistent_rows<T, OT, QKV>(M, N, Kp, ep, &m_head, &bm, KN)) return rc;
  if (m_head > 0) {
    int rc;
    if constexpr (sizeof(OT) == 2 && !QKV) {
      if (ep.drop.p > 0.f) {  // m_head == M
        if constexpr (sizeof(T) == 2)
          if (res) return launch_stream_res<true>(A, Bt, M, N, Kp, ep, st);
        return launch_stream<256, T, OT, QKV, true, KN>(A, Bt, M, N, Kp, ep, st);
      }
    }
    if (bm == 192) {
      rc = launch_stream<192, T, OT, QKV, false, KN>(A, Bt, m_head, N, Kp, ep, st);
    } else {
      if constexpr (sizeof(T) == 2 && !QKV)
        rc = res ? launch_stream_res<false>(A, Bt, m_head, N, Kp, ep, st)
                 : launch_stream<256, T, OT, QKV, false, KN>(A, Bt, m_head, N, Kp, ep, st);
      else
        rc = launch_stream<256, T, OT, QKV, false, KN>(A, Bt, m_head, N, Kp, ep, st);
    }
    if (rc != 0 || m_head == M) return rc;
  }
  if constexpr (KN)
    return launch_gemm_tile_kn((const _Float16*)A + m_head * Kp, Bt, M - m_head, N, Kp,
                               tail_epi<T, OT, QKV>(ep, m_head, N), QKV, st);
  return launch_gemm_tile((const _Float16*)A + m_head * Kp, Bt, M - m_head, N, Kp,
                          tail_epi<T, OT, QKV>(ep, m_head, N), sizeof(T) == 2, sizeof(OT) == 2, QKV, st);
}

// The rows divided as the plain launch divides them, so that every row's sum is formed in the same
// order: those of the persistent kernel by the form that does not split K.
template <typename T, bool QKV>
int launch_shape_layernorm(const void* x, const void* Bt, int64_t M, int N, int H, const EpiDev& ep,
                           const LnArgs& ln, hipStream_t st) {
  int64_t m_head;
  int bm;
  if (const int rc = persistent_rows<T, _Float16, QKV>(M, N, H, ep, &m_head, &bm)) return rc;
  if (m_head > 0) {
    const int rc = launch_gemm_layernorm_tile(x, Bt, m_head, N, H, ep, ln, sizeof(T) == 2, QKV, false, st);
    if (rc != 0 || m_head == M) return rc;
  }
  return launch_gemm_layernorm_tile((const T*)x + m_head * H, Bt, M - m_head, N, H,
                                    tail_epi<T, _Float16, QKV>(ep, m_head, N), ln, sizeof(T) == 2, QKV, true, st);
}

}  // namespace

// The device-side epilogue description of a launch, or a negative error code.
static int make_epi(const GemmEpilogue& e, int64_t M, int N, EpiDev& ep) {
  if (M >= (1ll << 31) - 512) {
    set_error("gemm: M=%lld does not fit the kernel's 32-bit row index", (long long)M);
    return -2;
  }
  if (e.qkv && (e.d % 4) != 0) {
    set_error("gemm qkv epilogue: head size %d must be a multiple of 4", e.d);
    return -2;
  }
  ep = EpiDev{};
  ep.bias = e.bias;
  ep.residual = e.residual;
  ep.out = e.out;
  ep.q = e.q;
  ep.k = e.k;
  ep.v = e.v;
  ep.L = e.L;
  ep.heads = e.heads;
  ep.d = e.d;
  ep.gelu = e.gelu;
  ep.drop = DropoutArgs{e.qkv ? 0.f : e.drop.p, (unsigned)e.drop.seed,
                        (unsigned)(e.drop.seed >> 32)};
  ep.keep = (const unsigned char*)e.drop.keep;
  const uintptr_t amask = e.f16 ? 7 : 15;
  auto aligned = [&](const void* p) { return p == nullptr || ((uintptr_t)p & amask) == 0; };
  const bool vec = (N % 4) == 0 && aligned(e.bias) && aligned(e.residual) && aligned(e.out) &&
                   aligned(e.q) && aligned(e.k) && aligned(e.v);
  ep.vec_ok = vec ? 1 : 0;
  auto aligned16 = [&](const void* p) { return ((uintptr_t)p & 15) == 0; };
  const bool half_out = e.f16 || e.out_f16;
  // What the next kernel finds in the 256 MB memory-side cache it need not fetch from HBM; beyond a good third
  // of that, non-temporal stores, which leave the cache to the operands (forwards, all non-temporal / all through:
  // medium 5 x 777 3686 / 3461 us, 16 x 300 with logits 1720 / 1697 (1686 with the line), 512 x 300
  // 28.57 / 30.16 ms; lines from 40 to 160 MB are equal.  Products with a residual, which takes as much of the
  // cache again: 10000 x 6400 x 1600, 122 MB, 181 / 192 us, 8192 x 8192 x 1024, 128 MB, 134 / 145, 12000 x 4096 x 1024,
  // 93 MB, 96.6 / 95.7).
  ep.through = M * (int64_t)N * (half_out ? 2 : 4) <= (96ll << 20);
  const int cw = half_out ? 8 : 4;
  ep.tile_vec = N % cw == 0 && (!e.qkv || e.d % cw == 0) && aligned16(e.bias) && aligned16(e.residual) &&
                aligned16(e.out) && aligned16(e.q) && aligned16(e.k) && aligned16(e.v);
  ep.vec8_ok = vec && half_out && (N % 8) == 0 && aligned16(e.out) && aligned16(e.q) &&
               aligned16(e.k) && aligned16(e.v) && (!e.qkv || (e.d % 8) == 0);
  return 0;
}

int launch_gemm(const void* A, const void* Bt, int64_t M, int N, int Kp, const GemmEpilogue& e,
                hipStream_t st) {
  EpiDev ep;
  if (const int rc = make_epi(e, M, N, ep)) return rc;
  if (e.f16)
    return e.qkv ? launch_shape<_Float16, _Float16, true>(A, Bt, M, N, Kp, ep, st)
                 : launch_shape<_Float16, _Float16, false>(A, Bt, M, N, Kp, ep, st);
  if (e.out_f16)
    return e.qkv ? launch_shape<float, _Float16, true>(A, Bt, M, N, Kp, ep, st)
                 : launch_shape<float, _Float16, false>(A, Bt, M, N, Kp, ep, st);
  return e.qkv ? launch_shape<float, float, true>(A, Bt, M, N, Kp, ep, st)
               : launch_shape<float, float, false>(A, Bt, M, N, Kp, ep, st);
}

static bool disjoint(const void* a, size_t a_bytes, const void* b, size_t b_bytes) {
  return (uintptr_t)a + a_bytes <= (uintptr_t)b || (uintptr_t)b + b_bytes <= (uintptr_t)a;
}

// Wherever the tile kernel takes all rows: every size gains (microseconds, weights from HBM, transposed first /
// in place / packed once: 16 x 768 x 2304 6.7 / 3.9 / 3.4, 16 x 3072 x 768 8.9 / 7.8 / 4.8, 128 x 768 x 3072 10.4 / 5.7
// / 5.1, 128 x 3072 x 768 12.8 / 8.8 / 6.2, 600 x 768 x 768 8.2 / 5.4 / 5.1, 1477 x 768 x 3072 19.3 / 13.4 / 12.7, 4800 x
// 3072 x 768 32.5 / 28.2 / 29.2).  Tiles of 16 columns lose most against the image, a line of a row of W
// being 32 bytes of theirs.  In the persistent kernel without a residual, whole column tiles, up to the rows at which
// the 1 to 2 % that it takes longer are what the transposition takes (4800 x 768 x 3072 31.4 / 26.2 / 24.8, 9600 x 768 x
// 3072 54.7 / 49.2 / 48.5, 40000 x 768 x 3072 203 / 202 / 198).
// Not where an output lies over the weight, whose image is complete before the first output is stored.
bool gemm_reads_kn(const void* W, int64_t M, int N, int K, const GemmEpilogue& e) {
  EpiDev ep;
  int64_t head;
  int bm;
  const size_t w_bytes = (size_t)K * N * 2, out_bytes = (size_t)M * N * 2, part = out_bytes / 3;
  if (e.qkv ? !disjoint(W, w_bytes, e.q, part) || !disjoint(W, w_bytes, e.k, part) || !disjoint(W, w_bytes, e.v, part)
            : !disjoint(W, w_bytes, e.out, out_bytes))
    return false;
  if (!e.f16 || K % 64 != 0 || ((uintptr_t)W & 15) != 0 || !gemm_tile_reads_kn(N, K) || make_epi(e, M, N, ep) != 0)
    return false;
  if ((e.qkv ? persistent_rows<_Float16, _Float16, true>(M, N, K, ep, &head, &bm, true)
             : persistent_rows<_Float16, _Float16, false>(M, N, K, ep, &head, &bm, true)) != 0)
    return false;
  return head == 0 || (e.residual == nullptr && stream_reads_kn(M, N));
}

int launch_gemm_kn(const void* A, const void* W, int64_t M, int N, int K, const GemmEpilogue& e, hipStream_t st) {
  EpiDev ep;
  if (const int rc = make_epi(e, M, N, ep)) return rc;
  return e.qkv ? launch_shape<_Float16, _Float16, true, true>(A, W, M, N, K, ep, st)
               : launch_shape<_Float16, _Float16, false, true>(A, W, M, N, K, ep, st);
}

int gemm_qkv_split(int64_t M, int N, int K, int64_t L, int heads, int d) {
  const int cus = cu_count();
  if (cus < 0) return cus;
  GemmEpilogue e = {};
  e.L = L, e.heads = heads, e.d = d;
  e.qkv = e.f16 = true;
  EpiDev ep;
  int64_t head;
  int bm;
  if (const int rc = make_epi(e, M, N, ep)) return rc;
  if (const int rc = persistent_rows<_Float16, _Float16, true>(M, N, K, ep, &head, &bm)) return rc;
  if (head > 0) return head == M ? 1 : 0;
  return gemm_tile_split(M, N, K, cus);
}

int launch_gemm_layernorm(const void* x, const void* ln_w, const void* ln_b, float eps,
                          const void* Bt, int64_t M, int N, int H, const GemmEpilogue& e,
                          hipStream_t st) {
  if (!(e.f16 || e.out_f16) || e.residual != nullptr || e.drop.p > 0.f || !gemm_layernorm_supported(M, H, e.f16)) {
    set_error("gemm with LayerNorm prologue: fp16 output, no residual, no dropout, H=%d a multiple of "
              "64 whose 32-row panel fits the LDS", H);
    return -2;
  }
  if ((((uintptr_t)x | (uintptr_t)ln_w | (uintptr_t)ln_b | (uintptr_t)Bt) & 15) != 0) {
    set_error("gemm with LayerNorm prologue: x, the LayerNorm parameters and W must be 16-byte aligned");
    return -2;
  }
  EpiDev ep;
  if (const int rc = make_epi(e, M, N, ep)) return rc;
  const LnArgs ln = {ln_w, ln_b, eps, lanes_per_row(H / (e.f16 ? 8 : 4))};
  if (e.f16)
    return e.qkv ? launch_shape_layernorm<_Float16, true>(x, Bt, M, N, H, ep, ln, st)
                 : launch_shape_layernorm<_Float16, false>(x, Bt, M, N, H, ep, ln, st);
  return e.qkv ? launch_shape_layernorm<float, true>(x, Bt, M, N, H, ep, ln, st)
               : launch_shape_layernorm<float, false>(x, Bt, M, N, H, ep, ln, st);
}

}  // namespace gptmi
