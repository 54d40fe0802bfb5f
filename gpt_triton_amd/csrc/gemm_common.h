// What the GEMM translation units share: the epilogue description, the direct global->LDS loads
// with their hand-counted waits, the tile order, and the CU count of the persistent launches.
#pragma once
#include <math.h>
#include <stdlib.h>

#include "common.h"
#include "launch.h"

namespace gptmi {

struct EpiDev {
  const void* bias;
  const void* residual;
  void* out;
  void* q;
  void* k;
  void* v;
  int64_t L;
  int heads;
  int d;
  int gelu;
  int vec_ok;  // pointers and N allow 4-element vector accesses
  int tile_vec; // gemm_tile_kernel: N, head size and every pointer allow 16-byte accesses
  int vec8_ok; // fp16 output: N, head size and the output pointers also allow 16-byte stores
  int through; // outputs written through (store_through), not non-temporal: make_epi
  int m_off;   // head-major scatter: row 0 of this launch is row m_off of the [B*L] token rows
  DropoutArgs drop;  // p > 0: dropout between GELU and residual
  const unsigned char* keep;  // its mask by flat index, or nullptr: generated in the epilogue (gemm_tile_kernel)
};

// LayerNorm in the operand prologue (gemm_tile_kernel<..., LNA = true>): weight, bias, epsilon and
// the lanes per row the LayerNorm kernel would use for rows of this width (the sums are then
// formed in the same order and the normalised operand has the same bits as that kernel's output).
struct LnArgs {
  const void* w;
  const void* b;
  float eps;
  int lpr;
};

// Direct global->LDS load of 16 bytes per lane: lane l's bytes land at LDS
// byte offset lds_off + 16*l (lds_off is wavefront-uniform and travels in M0).
// Issued as inline assembly so that the compiler's wait-count tracking does not
// see an LDS-writing memory instruction in flight: with the builtin, every LDS
// wait inside the pipelined loop degrades to "wait for everything".  Completion
// is tracked by hand with vmcnt (wait_vmcnt) ahead of the workgroup barrier.
__device__ __forceinline__ void lds_dma16(const void* gsrc, unsigned lds_off) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off"
               :
               : "s"(lds_off), "v"(gsrc)
               : "memory", "m0");
}

// The same with a wavefront-uniform 64-bit base in scalar registers and a 32-bit per-lane
// byte offset: one VGPR per load instead of an address pair, and the k-step is a scalar add.
__device__ __forceinline__ void lds_dma16_base(const void* base, unsigned lane_off,
                                               unsigned lds_off) {
  // s_mov + s_nop 3 = 5 wait states between a VALU write of `base` (v_readfirstlane, should
  // the compiler ever have to move it out of a vector register) and the load that reads it
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 3\n\tglobal_load_lds_dwordx4 %1, %2"
               :
               : "s"(lds_off), "v"(lane_off), "s"(base)
               : "memory", "m0");
}

// Store of 4 or 8 output elements at (wavefront-uniform 64-bit base) + (32-bit lane
// offset), written through (see store_through) or non-temporal as ep.through says (make_epi).
// Written as assembly because the compiler otherwise materialises one 64-bit address
// pair per store of an unrolled epilogue and spills.  Two hazards the compiler handles for its
// own instructions and cannot see inside assembly:
//   * a scalar register written by a VALU instruction (v_readfirstlane) must not be read by a
//     memory instruction within the next 5 wait states -- the leading s_nop 4 covers a base
//     that the compiler had to move out of a vector register;
//   * a store of more than 64 bits reads its data registers a little after issue -- the
//     trailing s_nop 1 keeps the next VALU instruction from overwriting them.
template <typename V>
__device__ __forceinline__ void store_base(int through, void* base, unsigned lane_off, V v) {
  static_assert(sizeof(V) == 8 || sizeof(V) == 16, "8 or 16 bytes");
  if constexpr (sizeof(V) == 8) {
    if (through)
      asm volatile("s_nop 4\n\tglobal_store_dwordx2 %0, %1, %2 sc0 sc1"
                   : : "v"(lane_off), "v"(v), "s"(base) : "memory");
    else
      asm volatile("s_nop 4\n\tglobal_store_dwordx2 %0, %1, %2 nt"
                   : : "v"(lane_off), "v"(v), "s"(base) : "memory");
  } else {
    if (through)
      asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 sc0 sc1\n\ts_nop 1"
                   : : "v"(lane_off), "v"(v), "s"(base) : "memory");
    else
      asm volatile("s_nop 4\n\tglobal_store_dwordx4 %0, %1, %2 nt\n\ts_nop 1"
                   : : "v"(lane_off), "v"(v), "s"(base) : "memory");
  }
}
// The same at a pointer of each lane's own.
template <typename V>
__device__ __forceinline__ void store_at(int through, V* p, V v) {
  if (through) store_through(p, v);
  else __builtin_nontemporal_store(v, p);
}

// Workgroup barrier that does not drain the vector-memory counter: the
// compiler's own barrier waits for vmcnt(0), which would serialise the
// global->LDS prefetch of the younger pipeline stages behind it.
__device__ __forceinline__ void block_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  static_assert(N >= 0 && N <= 63, "vmcnt is a 6-bit counter");
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

template <typename T> struct Pack4;
template <> struct Pack4<_Float16> { typedef h4 type; };
template <> struct Pack4<float> { typedef f4 type; };

// Address of out[m][n] (plain) or of the q/k/v element that column n of row m
// scatters to (qkv mode; n is a multiple of 4 and head sizes are too, so 4
// consecutive columns stay inside one head).
template <typename T, bool QKV>
__device__ __forceinline__ T* out_ptr(const EpiDev& ep, int64_t m, int n, int N) {
  if constexpr (!QKV) {
    return (T*)ep.out + (m * (int64_t)N + n);
  } else {
    // m < 2^31 (checked by the launcher) and L <= m's range: 32-bit divisions
    const unsigned hd = (unsigned)(ep.heads * ep.d);
    const unsigned which = (unsigned)n / hd;
    const unsigned within = (unsigned)n - which * hd;
    const unsigned head = within / (unsigned)ep.d;
    const unsigned dd = within - head * (unsigned)ep.d;
    const unsigned L = (unsigned)ep.L;
    const unsigned b = (unsigned)m / L;
    const unsigned l = (unsigned)m - b * L;
    T* base = (T*)(which == 0 ? ep.q : (which == 1 ? ep.k : ep.v));
    return base + ((((int64_t)b * ep.heads + head) * ep.L + l) * ep.d + dd);
  }
}

// Head-major destination of column n, row 0 of batch 0: q/k/v base + (head * L + 0) * d + dd.
template <typename T>
__device__ __forceinline__ T* qkv_column_base(const EpiDev& ep, int n) {
  const unsigned hd = (unsigned)(ep.heads * ep.d);
  const unsigned which = (unsigned)n / hd;
  const unsigned within = (unsigned)n - which * hd;
  const unsigned head = within / (unsigned)ep.d;
  const unsigned dd = within - head * (unsigned)ep.d;
  T* base = (T*)(which == 0 ? ep.q : (which == 1 ? ep.k : ep.v));
  return base + ((int64_t)head * ep.L * ep.d + dd);
}

// XCD-aware tile id: workgroup ids are dealt round-robin over the 8 XCDs, so id
// p runs on XCD p % 8.  The remap hands every XCD a contiguous range of tiles.
__device__ __forceinline__ int xcd_tile(int pid, int num_tiles) {
  const int per = (num_tiles + 7) >> 3;
  int tall = num_tiles & 7;
  if (tall == 0) tall = 8;
  const int xcd = pid & 7, loc = pid >> 3;
  return xcd < tall ? xcd * per + loc : tall * per + (xcd - tall) * (per - 1) + loc;
}

// Width, in column tiles, of the groups the tile order walks through.
//
// A launch whose tiles all run at once (no more than CUs): an XCD has one contiguous range of R tiles, and reads the
// weight panels of its columns and the activation panels of its rows into its L2 once each, so the fewest bytes are
// those of a patch of as nearly the same bytes either way: w = sqrt(R BM / BN) columns.  Groups of one column, all
// its rows one after the other, where the rows of w columns are no more than the range, or hardly (then a column is
// read by one XCD alone).  Weights from HBM, the activations in the L2s, us, column fastest throughout / so: 128 x 2304 x
// 768 4.66 / 4.22, 300 x 768 x 768 4.12 / 3.68, 128 x 768 x 3072 7.2 / 7.0, 3885 x 1024 x 4096 38.3 / 35.8.
// In a forward the row order has something for it too: an XCD then finds rows in its L2 that it has just written.  So
// the patches are for few rows, for products whose weight does not fit beside that in an L2 of 4 MB, and for
// those that are no deeper than wide, without the scatter.  Forwards replayed, column fastest / patches in the q, k, v
// product / projection / ffn1 / ffn2: 2 x 64 tokens of 124M 357 / 352 / 356 / 349 / 358, 8 x 40 420 / 424 / 420 / 422 / 427,
// 2 x 300 525 / 529 / 523 / 525 / 529, 1 x 800 670 / 674 / 669 / 667 / 670; 1024 wide 3 x 300 1502 / 1493 / 1494 / 1505 /
// 1479, 5 x 777 3490 / 3493 / 3488 / 3488 / 3459; 1600 wide 1 x 300 3140 / 3130 / 3125 / 3120 / 3120, 3 x 300 4983 / 4986 /
// 4984 / 4955 / 4931.
//
// More tiles than that: the weight panels of one group (group_w * BN rows of Kp halves) should stay in a 4 MB L2
// beside the activation panels in flight, so they get about 2.4 MB; every group re-reads the activations once, so
// the groups are as few and as even as that allows.  Panels too long for two of them to fit
// (large K) keep the plain column-fastest order.
inline int column_group(int64_t M, int N, int Kp, bool scatter, int bm, int bn, int cus) {
  const int64_t tiles_m = (M + bm - 1) / bm;
  const int tiles_n = (N + bn - 1) / bn;
  if (tiles_m * tiles_n <= cus && (M <= 128 || (int64_t)N * Kp > 5 << 19 || (!scatter && Kp <= N))) {
    const float range = (float)((tiles_m * tiles_n + 7) / 8), w = sqrtf(range * (float)bm / (float)bn);
    if (w * (float)tiles_m <= 1.25f * range) return 1;
    const int groups = (int)((float)tiles_n / w + 0.5f);
    return groups <= 1 ? tiles_n : (tiles_n + groups - 1) / groups;
  }
  const int64_t panel = (int64_t)bn * Kp * 2;
  const int fit = (int)((2400 << 10) / panel);
  if (fit < 2 || tiles_n <= fit) return tiles_n;
  const int groups = (tiles_n + fit - 1) / fit;
  return (tiles_n + groups - 1) / groups;
}

// CUs of the current device rounded down to a multiple of 8 (workgroup id % 8 = XCD for every
// tile of a persistent launch), or a negative error code.  The environment variable
// GPTMI_MAX_WORKGROUPS (read once) caps the number: a measurement knob -- with fewer persistent
// workgroups than CUs the chip's power management holds a higher clock, which is how one tells a
// kernel that is bound by the power budget from one that is bound by its own schedule.
inline int cu_count() {
  static int num_cus = 0;  // idempotent one-time setup; a race only repeats it
  if (num_cus == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus < 8) {
      set_error("gemm: cannot query the CU count");
      return -4;
    }
    if (const char* cap = getenv("GPTMI_MAX_WORKGROUPS")) {
      const int c = atoi(cap);
      if (c >= 8 && c < cus) cus = c;
    }
    num_cus = cus - cus % 8;
  }
  return num_cus;
}

// One workgroup per output tile (gemm_tile.hip), every size, type and epilogue; the LayerNorm
// prologue form of it (split: K over as many groups as the cost model takes for these rows, otherwise
// one); and what the cost model says a launch takes, in microseconds.
int launch_gemm_tile(const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                     bool f16, bool out_f16, bool qkv, hipStream_t st);
// The same on fp16 operands and the weight [K][N] as it stands, 16-byte aligned, where gemm_tile_reads_kn.
bool gemm_tile_reads_kn(int N, int Kp);
int launch_gemm_tile_kn(const void* A, const void* W, int64_t M, int N, int K, const EpiDev& ep, bool qkv,
                        hipStream_t st);
int launch_gemm_layernorm_tile(const void* x, const void* Bt, int64_t M, int N, int H, const EpiDev& ep,
                               const LnArgs& ln, bool f16, bool qkv, bool split, hipStream_t st);
float gemm_tile_cost(int64_t M, int N, int Kp, int cus);
// Over how many groups launch_gemm divides K for M rows of a q, k, v product in fp16, the order of its sums; 0: not
// the same for all rows; negative: an error.
int gemm_qkv_split(int64_t M, int N, int K, int64_t L, int heads, int d);
int gemm_tile_split(int64_t M, int N, int Kp, int cus);

}  // namespace gptmi
