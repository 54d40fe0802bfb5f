// GEMM on one workgroup per output tile, for problems that do not fill the persistent 256 x 256
// kernels of gemm.hip: a few rows up to a few thousand.
//
//   C[M][N] = A[M][Kp] . Bt[N][Kp]^T,  out = dropout(gelu?(C + bias)) + residual
//
// (reference: fused_ffn_kernel, kernels.py:169-257, and the q/k/v relayout of
// matmul_and_split_qkv, kernels.py:347-367.)  With A = LayerNorm(x) where asked for (LNA).
//
// What bounds it.  At these sizes a workgroup's own path through its k-tiles does: a barrier, an
// LDS round trip and a memory round trip per k-tile that no other workgroup of the CU hides.  So
//   * WK groups of wavefronts split K inside the workgroup: group g multiplies the 64-wide
//     k-slices g, g + WK, ..., so a "k-step" of the workgroup is WK slices wide and the number of
//     barriers and round trips falls by WK.  The groups' partial sums meet in LDS at the end and are
//     added in group order: deterministic, but the order depends on the tile that the row count picks,
//     so a row's last bit may differ between batches (four sums of K / 4 terms are nearer to the exact
//     one: 128 x 768 x 3072 in fp32 1.8e-7 rms against 3.5e-7 for one running sum);
//   * the fragments of the whole next k-step are read from LDS (into a second register set) while the
//     current one is multiplied, one read behind every MFMA or two, so an LDS round trip has the time
//     of a k-step, not of one slice;
//   * NST k-steps are in LDS or on their way; a stage is refilled as soon as its fragments are in
//     registers.
//   * The epilogue goes through a row-major fp32 tile in LDS: every thread owns 16 bytes of the
//     output at a time (8 halves or 4 floats), so loads and stores are whole lines whatever the
//     tile's shape, a ragged last row costs one comparison, and residual, GELU, dropout and the
//     head-major scatter are the same few lines for every configuration.
#include <type_traits>

#include "gemm_common.h"
#include "layernorm_panel.h"

namespace gptmi {

namespace {

// One shape of workgroup: BM x BN output tile on WM x WN wavefronts times WK groups that split K,
// NST k-steps of LDS stages.
template <int BM_, int BN_, int WM_, int WN_, int WK_, int NST_>
struct Tile {
  static constexpr int BM = BM_, BN = BN_, WM = WM_, WN = WN_, WK = WK_, NST = NST_;
  static constexpr int THREADS = 64 * WM_ * WN_ * WK_;
};

// T: storage type of bias and residual, and with LNA of the rows and the LayerNorm's parameters.  OT: type of the output: T, or fp16 for
// fp32 storage where the output is the next product's operand (no residual then).
// WIDE: rows of 2^22 elements and more (64-bit lane addresses).
//
// KN: the weight as the caller has it, Bt = W [K][N] in fp16, instead of its packed image: no launch that
// transposes it first (3.5 us and more, on every call with a weight that is not packed once).  A slice is then
// 64 rows of BN columns, and a fragment is two transposing LDS loads (ds_read_b64_tr_b16: 4 rows of k x 16
// columns each) where the image takes one load of 16 bytes; the products, their order and the sums are the
// same, and so are the bits.
template <class C, typename T, typename OT, bool QKV, bool LNA, bool DROP, bool WIDE, bool KN>
__global__ __launch_bounds__(C::THREADS, 2) void gemm_tile_kernel(
    const void* __restrict__ Av, const _Float16* __restrict__ Bt, int M, int N, int Kp,
    int tiles_m, int tiles_n, int group_w, EpiDev ep, LnArgs ln) {
  constexpr int BM = C::BM, BN = C::BN, WM = C::WM, WN = C::WN, WK = C::WK, NST = C::NST;
  constexpr int TG = 64 * WM * WN, NT = TG * WK;  // threads per k-group, per workgroup
  constexpr int TM = BM / WM, TN = BN / WN, MB = TM / 16, NB = TN / 16;
  constexpr int A_IT = LNA ? 0 : BM * 8 / TG, B_IT = BN * 8 / TG, LPT = A_IT + B_IT;
  constexpr int A_N = A_IT ? A_IT : 1;
  constexpr int B_AT = LNA ? 0 : BM * 128;     // byte offset of the weight rows inside a slice
  constexpr int SLICE = B_AT + BN * 128;       // one group's 64-wide k-slice
  constexpr int STAGE = SLICE * WK;
  static_assert((LNA || (BM * 8) % TG == 0) && (BN * 8) % TG == 0, "tile/threads mismatch");
  static_assert(TM % 16 == 0 && TN % 16 == 0, "16 x 16 MFMA blocks");
  static_assert(NST >= 2 && (NST - 2) * LPT <= 63, "vmcnt range");

  extern __shared__ __attribute__((aligned(1024))) char smem[];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int g = wave / (WM * WN), w = wave % (WM * WN);
  const int wm = w % WM, wn = w / WM;
  const int tg = tid % TG;

  const int tile = xcd_tile(blockIdx.x, tiles_m * tiles_n);
  const int grp = tile / (tiles_m * group_w);
  const int in_grp = tile - grp * tiles_m * group_w;
  const int grp_w = min(group_w, tiles_n - grp * group_w);
  const int m0 = (in_grp / grp_w) * BM, n0 = (grp * group_w + in_grp % grp_w) * BN;

  // ---- direct global->LDS loads ------------------------------------------------------------
  // Load `it` of a thread: 16-byte slot it * TG + tg of its group's slice: row slot / 8, position
  // slot % 8, which holds source unit (slot % 8) ^ ((row >> 1) & 7).  Rows past the matrix edge
  // re-read the last row (their products are never stored).
  typedef typename std::conditional<WIDE, size_t, unsigned>::type Off;
  auto row_off = [&](int r0, int rows, int s) __attribute__((always_inline)) {
    const int r = s >> 3;
    return (Off)(min(r0 + r, rows - 1) - r0) * (Off)Kp * 2u + (Off)(((s & 7) ^ ((r >> 1) & 7)) * 16);
  };
  // KN: slot s is row s / UPB of k, position s % UPB, which holds source unit (s % UPB) ^ kn_key(row), 8
  // columns; columns past the edge re-read the last 8.
  constexpr int UPB = BN / 8;
  auto kn_key = [](int r) __attribute__((always_inline)) {
    return UPB >= 16 ? 2 * ((r & 3) | (r >> 1 & 4)) : UPB == 8 ? 2 * ((r >> 1 & 1) | (r >> 2 & 2))
                                                   : UPB == 4 ? 2 * (r >> 3 & 1) : 0;
  };
  auto kn_off = [&](int s) __attribute__((always_inline)) {
    const int r = s / UPB, u = (s % UPB) ^ kn_key(r);
    return ((Off)r * (Off)N + (Off)(min(n0 + 8 * u, N - 8) - n0)) * 2u;
  };
  Off a_off[A_N], b_off[B_IT];
#pragma unroll
  for (int it = 0; it < A_IT; ++it) a_off[it] = row_off(m0, M, it * TG + tg);
#pragma unroll
  for (int it = 0; it < B_IT; ++it) b_off[it] = KN ? kn_off(it * TG + tg) : row_off(n0, N, it * TG + tg);
  const int KT = Kp / 64, ST = (KT + WK - 1) / WK;  // k-slices, k-steps
  const char* a_base = (const char*)Av + (size_t)m0 * Kp * 2;
  const char* b_base = (const char*)(Bt + (KN ? (size_t)n0 : (size_t)n0 * Kp));
  const unsigned wave_off = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem) +
                            (unsigned)g * SLICE + (unsigned)w * 1024u;
  // a group without a slice in the last k-step loads the last slice again and multiplies nothing
  auto issue_one = [&](int t, int stage, int n) __attribute__((always_inline)) {
    const size_t slice = (size_t)min(t * WK + g, KT - 1);
    const unsigned at = wave_off + (unsigned)stage * STAGE;
    const char* base = n < A_IT ? a_base + slice * 128 : b_base + slice * (KN ? (size_t)N * 128 : 128);
    const Off off = n < A_IT ? a_off[n < A_IT ? n : 0] : b_off[n < A_IT ? 0 : n - A_IT];
    const unsigned lds = at + (n < A_IT ? n * (TG * 16) : B_AT + (n - A_IT) * (TG * 16));
    if constexpr (WIDE) lds_dma16(base + off, lds);
    else lds_dma16_base(base, off, lds);
  };
  // The loads of a k-step are dealt over the second half of one k-step (the first L1 of them) and
  // the first half of the next: a burst arrives faster than the texture unit takes it (16 cycles a
  // load and CU), and the wavefronts then stall on issue with their MFMAs behind it.
  constexpr int L1 = LPT / 2;
#pragma unroll
  for (int s = 0; s < NST; ++s)
    if (s < ST) {
#pragma unroll
      for (int n = 0; n < (s + 1 < NST ? LPT : L1); ++n) issue_one(s, s, n);
    }

  // acc[i][j]: columns 16 i.., rows 16 j.. of the wavefront's sub-tile; a lane holds the 4
  // columns 4 (lane / 16) + 0..3 of row lane % 16
  f4 acc[NB][MB];
#pragma unroll
  for (int i = 0; i < NB; ++i)
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[i][j][r] = 0.f;

  // Fragments of v_mfma_f32_16x16x32_f16: row lane % 16 of a block, 16-byte unit lane / 16 of a
  // 32-wide half slice.  16 consecutive lanes read 16 rows at one unit: no bank conflicts.
  const int lrow = lane & 15, lq = lane >> 4, fkey = (lrow >> 1) & 7;
  const int a_row = (wm * TM + lrow) * 128, b_row = B_AT + (wn * TN + lrow) * 128;
  const char* panel = smem + NST * STAGE;
  // KN: of block i, lane s = lane % 16 points at the 4 columns 4 (s % 4).. of row 8 lq + s / 4 of a half slice and
  // of the row 4 below, and gets column s of the 4 rows each
  int kn_at[NB];
  if constexpr (KN) {
    const int r = 8 * lq + (lrow >> 2);
#pragma unroll
    for (int i = 0; i < NB; ++i)
      kn_at[i] = B_AT + r * (BN * 2) + ((((wn * TN + i * 16) / 8 + ((lrow & 3) >> 1)) ^ kn_key(r)) << 4) + (lrow & 1) * 8;
  }
  h8 fa[2][MB], fb[2][NB];  // [half slice][block]
  constexpr int NR = MB + NB, NM = MB * NB;  // fragment reads, MFMAs per half slice
  constexpr int RPM = (NR + (NM + 1) / 2 - 1) / ((NM + 1) / 2);  // reads behind an MFMA: all behind the first half of them
  auto read_one = [&](int t, int stage, int half, int n) __attribute__((always_inline)) {
    const char* st = smem + stage * STAGE + g * SLICE;
    const int un = ((half * 4 + lq) ^ fkey) << 4;
    if (n < MB) {
      const char* sa = LNA ? panel + (size_t)min(t * WK + g, KT - 1) * (BM * 128) : st;
      fa[half][n < MB ? n : 0] = *reinterpret_cast<const h8*>(sa + a_row + n * 2048 + un);
    } else if constexpr (KN) {
      const char* at = st + kn_at[n < MB ? 0 : n - MB] + half * (32 * BN * 2);
      const h4 lo = lds_read_tr16(at), hi = lds_read_tr16(at + 4 * (BN * 2));
      fb[half][n < MB ? 0 : n - MB] = h8{lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    } else {
      fb[half][n < MB ? 0 : n - MB] = *reinterpret_cast<const h8*>(st + b_row + (n - MB) * 2048 + un);
    }
  };
  auto mfma_one = [&](int half, int n) __attribute__((always_inline)) {
    const int j = n / NB, ii = n % NB;
    const int i = (j & 1) ? NB - 1 - ii : ii;  // one operand changes per MFMA
    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[half][i], fa[half][j], acc[i][j], 0, 0, 0);
  };
  // the k-steps younger than the one that must have landed: `younger` of them, LPT loads each
  auto wait_landed = [&](int younger) __attribute__((always_inline)) {
    if (younger <= 0) wait_vmcnt<0>();
    else if (younger == 1 || NST < 3) wait_vmcnt<LPT>();
    else if (younger == 2 || NST < 4) wait_vmcnt<2 * LPT>();
    else if (younger == 3 || NST < 5) wait_vmcnt<3 * LPT>();
    else wait_vmcnt<4 * LPT>();
  };
  // a group of one wavefront reads only what it loaded itself
  auto meet = [&]() __attribute__((always_inline)) {
    if constexpr (WM * WN > 1) asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  };

  if constexpr (LNA) {
    normalise_panel<BM, NT>((const T*)Av, M, Kp, m0, ln, smem + NST * STAGE, tid);
    wait_vmcnt<0>();
    __syncthreads();
  } else {
    // k-step 0; behind it min(NST, ST) - 1 more, the last of them in part if it is the NST-th
    if (ST >= NST) wait_vmcnt<(NST - 2) * LPT + L1>();
    else wait_landed(ST - 1);
    meet();
  }
#pragma unroll
  for (int n = 0; n < NR; ++n) read_one(0, 0, 0, n);

  // ---- bias and residual of the chunks this thread will store, requested behind the first k-steps
  // (the counted waits of the loop then wait for these too, once, and otherwise for no more than
  // they name; at the end of the loop they would cost a memory round trip of their own)
  constexpr int CW = 16 / (int)sizeof(OT);  // output columns per 16 bytes
  constexpr int CPR = BN / CW, CHUNKS = BM * CPR, IT = (CHUNKS + NT - 1) / NT;
  static_assert(NT % CPR == 0, "a thread keeps its columns");
  typedef T TV __attribute__((ext_vector_type(CW)));
  typedef OT OV __attribute__((ext_vector_type(CW)));
  const int cc = tid % CPR, n = n0 + cc * CW, r_first = tid / CPR;
  constexpr int RSTEP = NT / CPR;
  const bool col_ok = n < N && (CHUNKS >= NT || tid < CHUNKS);
  // `vec`: N, head size and pointers allow 16-byte accesses; otherwise element by element
  const bool vec = ep.tile_vec;
  auto load_chunk = [&](const T* p) __attribute__((always_inline)) {
    TV v;
    if (vec) v = *reinterpret_cast<const TV*>(p);
    else {
#pragma unroll
      for (int e = 0; e < CW; ++e) v[e] = n + e < N ? p[e] : (T)0.f;
    }
    return v;
  };
  TV bias_v, res_v[IT];
#pragma unroll
  for (int e = 0; e < CW; ++e) bias_v[e] = (T)0.f;
  if (ep.bias && col_ok) bias_v = load_chunk((const T*)ep.bias + n);
  const bool res = !QKV && sizeof(T) == sizeof(OT) && ep.residual != nullptr;
  if (res && col_ok) {
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      const int m = m0 + r_first + it * RSTEP;
      if (m < M) res_v[it] = load_chunk((const T*)ep.residual + ((int64_t)m * N + n));
    }
  }

  // the dropout mask of those chunks, where the caller has it: CW bits of one byte (N and n are
  // multiples of CW then).  Generated in the epilogue, 17 wide products per element, it more than
  // doubled the time of the launch (4800 x 768 x 3072: 85 us; 43 with the bits, 36 without dropout).
  unsigned keep_v[DROP ? IT : 1];
  if constexpr (DROP) {
    if (ep.keep != nullptr && col_ok) {
#pragma unroll
      for (int it = 0; it < IT; ++it) {
        const int m = m0 + r_first + it * RSTEP;
        const uint64_t at = (uint64_t)m * (uint64_t)N + (uint64_t)n;
        keep_v[it] = m < M ? (unsigned)ep.keep[at >> 3] >> (at & 7) : 0u;
      }
    }
  }

  // One k-step: the MFMAs of its first half with the fragment reads of its second half dealt
  // between them; the barrier that publishes k-step t + 1 and frees this stage; the MFMAs of the
  // second half with the reads of the next k-step's first half and the refill of this stage
  // with k-step t + NST.
  int stage = 0, st_prev = NST - 1;
  auto step = [&](auto load0, auto load1, int t) __attribute__((always_inline)) {
    constexpr bool LOAD0 = decltype(load0)::value, LOAD1 = decltype(load1)::value;
    const int st_next = stage + 1 == NST ? 0 : stage + 1;
#pragma unroll
    for (int q = 0; q < NM; ++q) {
      mfma_one(0, q);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = q * RPM; n < (q + 1) * RPM && n < NR; ++n) read_one(t, stage, 1, n);
      if constexpr (LOAD0) {
#pragma unroll
        for (int n = q * (LPT - L1) / NM; n < (q + 1) * (LPT - L1) / NM; ++n)
          issue_one(t + NST - 1, st_prev, L1 + n);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    if constexpr (LOAD0) wait_vmcnt<(NST - 2) * LPT>();
    else wait_landed(ST - 2 - t);
    meet();
#pragma unroll
    for (int q = 0; q < NM; ++q) {
      mfma_one(1, q);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int n = q * RPM; n < (q + 1) * RPM && n < NR; ++n) read_one(t + 1, st_next, 0, n);
      if constexpr (LOAD1) {
#pragma unroll
        for (int n = q * L1 / NM; n < (q + 1) * L1 / NM; ++n) issue_one(t + NST, stage, n);
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    st_prev = stage;
    stage = st_next;
  };
  std::true_type yes;
  std::false_type no;
  int t = 0;
  for (; t + NST < ST; ++t) step(yes, yes, t);
  if (t + 1 < ST && t + NST == ST) step(yes, no, t++);
  for (; t + 1 < ST; ++t) step(no, no, t);

  // ---- last k-step
  if (KT % WK == 0 || t * WK + g < KT) {
#pragma unroll
    for (int n = 0; n < NR; ++n) read_one(t, stage, 1, n);
#pragma unroll
    for (int q = 0; q < 2 * NM; ++q) mfma_one(q / NM, q % NM);
  }

  // ---- the groups' sums into LDS, row-major fp32: 16-byte unit u of row r at u ^ key(r), the key
  // such that the 16 rows a quarter wavefront writes fall on 16 different 16-byte slots
  __syncthreads();
  constexpr int UPR = BN / 4;  // 16-byte units per row
  auto unit_at = [&](int r, int u) __attribute__((always_inline)) {
    return UPR >= 16 ? u ^ (r & 15) : u ^ ((r >> 1) & (UPR - 1));
  };
  {
    char* mine = smem + g * (BM * BN * 4);
#pragma unroll
    for (int j = 0; j < MB; ++j)
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        const int r = wm * TM + j * 16 + lrow, u = (wn * TN + i * 16) / 4 + lq;
        *reinterpret_cast<f4*>(mine + r * (BN * 4) + (unit_at(r, u) << 4)) = acc[i][j];
      }
  }
  __syncthreads();
  if (!col_ok) return;

  OT* col = nullptr;  // head-major scatter: row 0 of batch 0 at this thread's columns
  if constexpr (QKV) col = qkv_column_base<OT>(ep, n);
  const int64_t batch_stride = (int64_t)ep.heads * ep.L * ep.d;
#pragma unroll
  for (int it = 0; it < IT; ++it) {
    const int r = r_first + it * RSTEP, m = m0 + r;
    if (m >= M || (CHUNKS % NT != 0 && r >= BM)) break;  // the last turn may be one of some threads only
    float z[CW];
#pragma unroll
    for (int u = 0; u < CW / 4; ++u) {
      const int at = r * (BN * 4) + (unit_at(r, cc * (CW / 4) + u) << 4);
      f4 s = *reinterpret_cast<const f4*>(smem + at);
#pragma unroll
      for (int k = 1; k < WK; ++k) s += *reinterpret_cast<const f4*>(smem + k * (BM * BN * 4) + at);
#pragma unroll
      for (int e = 0; e < 4; ++e) z[u * 4 + e] = s[e];
    }
#pragma unroll
    for (int e = 0; e < CW; ++e) {
      z[e] += (float)bias_v[e];
      if (ep.gelu) z[e] = gelu_new(z[e]);
    }
    if constexpr (DROP) {
      if (ep.keep != nullptr) {
        KeepScale(ep.drop.p).apply(z);
#pragma unroll
        for (int e = 0; e < CW; ++e) z[e] = keep_if(keep_v[it], e, z[e]);
      } else {
        unsigned off[CW];
#pragma unroll
        for (int e = 0; e < CW; ++e) off[e] = (unsigned)((uint64_t)m * (uint64_t)N + (uint64_t)(n + e));
        dropout_apply<CW>(ep.drop, off, z);
      }
    }
    OV o;
#pragma unroll
    for (int e = 0; e < CW; ++e) o[e] = (OT)(res ? z[e] + (float)res_v[it][e] : z[e]);
    OT* dst;
    if constexpr (QKV) {
      const unsigned mt = (unsigned)(m + ep.m_off), b = mt / (unsigned)ep.L, l = mt - b * (unsigned)ep.L;
      dst = col + ((int64_t)b * batch_stride + (int64_t)l * ep.d);
    } else {
      dst = (OT*)ep.out + ((int64_t)m * N + n);
    }
    if (vec) store_at(ep.through, reinterpret_cast<OV*>(dst), o);
    else {
#pragma unroll
      for (int e = 0; e < CW; ++e)
        if (n + e < N) dst[e] = o[e];
    }
  }
}

template <class C, typename T, typename OT, bool QKV, bool LNA, bool DROP, bool WIDE = false, bool KN = false>
int launch_tile_cfg(const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                    const LnArgs& ln, hipStream_t st) {
  auto kern = gemm_tile_kernel<C, T, OT, QKV, LNA, DROP, WIDE, KN>;
  constexpr int stages = C::NST * ((LNA ? 0 : C::BM) + C::BN) * 128 * C::WK, sums = C::BM * C::BN * 4 * C::WK;
  static_assert(stages <= 160 * 1024 && sums <= 160 * 1024, "LDS");
  const size_t panel = LNA ? (size_t)C::BM * Kp * 2 : 0;
  const size_t smem = stages + panel > (size_t)sums ? stages + panel : (size_t)sums;
  static bool attr_done = false;  // idempotent; a race only repeats the call
  if (!attr_done) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, 160 * 1024);
    if (e != hipSuccess) {
      set_error("hipFuncSetAttribute(160 KB LDS): %s", hipGetErrorString(e));
      return -4;
    }
    attr_done = true;
  }
  const int64_t tiles_m = (M + C::BM - 1) / C::BM, tiles_n = ((int64_t)N + C::BN - 1) / C::BN;
  if (tiles_m * tiles_n > 0x7fffffffll) {
    set_error("gemm: %lld x %lld output tiles exceed the grid", (long long)tiles_m, (long long)tiles_n);
    return -2;
  }
  const int cus = cu_count();
  if (cus < 0) return cus;
  const int group_w = column_group(M, N, Kp, QKV, C::BM, C::BN, cus);
  hipLaunchKernelGGL(kern, dim3((unsigned)(tiles_m * tiles_n)), dim3(C::THREADS), smem, st, A,
                     (const _Float16*)Bt, (int)M, N, Kp, (int)tiles_m, (int)tiles_n, group_w, ep, ln);
  return 0;
}

// The menu, with the numbers of the cost model: a launch of ceil(tiles / CUs) = R rounds takes about
// launch + R (fixed + k_slices * slice) microseconds.  Fitted to the products of a layer of the four GPT-2
// widths (GELU and residual epilogues, weights from HBM, outputs written through) at 23 row counts from 8 to
// 20000: 8 % off on average, and the model's choice among these tiles and the persistent kernels is 0.9 %
// slower than the fastest of 17 shapes.  What the numbers say: a workgroup takes in 36 to 48 bytes per
// clock whatever its shape (4800 x 3072 x 768: the loads alone take 18 of the 22 us of the k-loop, 14.5 of
// them if every line is in the L2), so a tile costs its operand bytes -- small tiles win while they
// fill the 256 CUs once, large ones as soon as they do.
//                    BM   BN  WM WN WK NST
typedef Tile< 32,  16, 1, 1, 4, 4> T32x16;
typedef Tile< 32,  32, 1, 1, 4, 4> T32x32;
typedef Tile< 64,  32, 2, 1, 4, 3> T64x32;
typedef Tile< 64,  64, 2, 2, 2, 4> T64x64;
typedef Tile< 64, 128, 2, 2, 2, 3> T64x128;
typedef Tile<128, 128, 2, 4, 1, 4> T128x128;
typedef Tile<192, 128, 4, 2, 1, 3> T192x128;
typedef Tile<128, 256, 2, 4, 1, 3> T128x256;
struct TileCost {
  int bm, bn, wk;
  float launch, fixed, slice;
};
constexpr TileCost kTiles[] = {
    {32, 16, 4, 0.92f, 2.50f, 0.049f},  {32, 32, 4, 1.26f, 1.76f, 0.086f},
    {64, 32, 4, 1.09f, 2.17f, 0.129f},  {64, 64, 2, 1.00f, 1.65f, 0.180f},
    {64, 128, 2, 0.85f, 3.23f, 0.283f}, {128, 128, 1, 0.f, 4.21f, 0.476f},
    {192, 128, 1, 0.f, 5.35f, 0.664f},  {128, 256, 1, 0.f, 6.91f, 0.740f},
};
// Shapes between those: for row and column counts that leave the ones above a last round with few tiles
// (products at 24 to 4800 rows, before -> after: 48 x 1280 x 5120 8.4 -> 7.0 us, 1477 x 768 x 3072 15.7 -> 14.0,
// 3072 x 768 x 3072 24.1 -> 22.0, 4800 x 1600 x 6400 111 -> 91; 1.6 % over all of them).
typedef Tile< 16,  16, 1, 1, 4, 4> T16x16;
typedef Tile< 48,  32, 1, 1, 4, 3> T48x32;
typedef Tile< 96,  64, 2, 2, 2, 3> T96x64;
typedef Tile<192,  64, 4, 2, 1, 4> T192x64;
typedef Tile<256, 128, 4, 2, 1, 3> T256x128;
constexpr TileCost kTilesBetween[] = {
    {16, 16, 4, 2.70f, 0.72f, 0.033f},  {48, 32, 4, 1.28f, 1.91f, 0.108f},
    {96, 64, 2, 1.04f, 2.58f, 0.236f},  {192, 64, 1, 0.28f, 3.52f, 0.403f},
    {256, 128, 1, 0.f, 6.84f, 0.753f},
};
constexpr int kNumFirst = sizeof(kTiles) / sizeof(kTiles[0]);
constexpr int kNumTiles = kNumFirst + sizeof(kTilesBetween) / sizeof(kTilesBetween[0]);

constexpr const TileCost& tile_cost(int i) { return i < kNumFirst ? kTiles[i] : kTilesBetween[i - kNumFirst]; }

// Unrolled, with the table's numbers as constants: a forward of few tokens asks four times a layer, and
// the host sets its pace.
template <int I>
inline void pick_from(int64_t M, int N, float k, int cus, int& best, float& least) {
  if constexpr (I < kNumTiles) {
    constexpr TileCost c = tile_cost(I);
    const int64_t tiles = ((M + c.bm - 1) / c.bm) * ((N + (c.bn - 1)) / c.bn);
    const int64_t rounds = tiles <= cus ? 1 : (tiles + cus - 1) / cus;
    const float cost = c.launch + (float)rounds * (c.fixed + k * c.slice);
    if (cost < least) least = cost, best = I;
    pick_from<I + 1>(M, N, k, cus, best, least);
  }
}

inline int pick_tile(int64_t M, int N, int Kp, int cus, float* cost) {
  int best = 0;
  float least = INFINITY;
  pick_from<0>(M, N, (float)(Kp / 64), cus, best, least);
  if (cost) *cost = least;
  return best;
}

template <typename T, typename OT, bool QKV, bool DROP, bool KN>
int launch_pick(int i, const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                hipStream_t st) {
  const LnArgs ln = {};
  switch (i) {
    case 0: return launch_tile_cfg<T32x16, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 1: return launch_tile_cfg<T32x32, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 2: return launch_tile_cfg<T64x32, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 3: return launch_tile_cfg<T64x64, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 4: return launch_tile_cfg<T64x128, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 5: return launch_tile_cfg<T128x128, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 6: return launch_tile_cfg<T192x128, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 7: return launch_tile_cfg<T128x256, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 8: return launch_tile_cfg<T16x16, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 9: return launch_tile_cfg<T48x32, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 10: return launch_tile_cfg<T96x64, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    case 11: return launch_tile_cfg<T192x64, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
    default: return launch_tile_cfg<T256x128, T, OT, QKV, false, DROP, false, KN>(A, Bt, M, N, Kp, ep, ln, st);
  }
}

// rows of 2^22 elements and more: 64-bit addresses, one tile shape
constexpr int kWideK = 1 << 22;

}  // namespace

int gemm_tile_split(int64_t M, int N, int Kp, int cus) {
  return tile_cost(pick_tile(M, N, Kp, cus, nullptr)).wk;
}

float gemm_tile_cost(int64_t M, int N, int Kp, int cus) {
  float cost;
  pick_tile(M, N, Kp, cus, &cost);
  return cost;
}

template <typename T, typename OT, bool QKV, bool KN = false>
static int launch_tile_t(const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                         hipStream_t st) {
  const int cus = cu_count();
  if (cus < 0) return cus;
  if constexpr (!QKV) {
    if (ep.drop.p > 0.f) {
      if constexpr (!KN)
        if (Kp >= kWideK)
          return launch_tile_cfg<T32x32, T, OT, false, false, true, true>(A, Bt, M, N, Kp, ep, LnArgs{}, st);
      return launch_pick<T, OT, false, true, KN>(pick_tile(M, N, Kp, cus, nullptr), A, Bt, M, N, Kp, ep, st);
    }
  }
  if constexpr (!KN)
    if (Kp >= kWideK)
      return launch_tile_cfg<T32x32, T, OT, QKV, false, false, true>(A, Bt, M, N, Kp, ep, LnArgs{}, st);
  return launch_pick<T, OT, QKV, false, KN>(pick_tile(M, N, Kp, cus, nullptr), A, Bt, M, N, Kp, ep, st);
}

bool gemm_tile_reads_kn(int N, int Kp) { return N % 8 == 0 && N <= 1 << 22 && Kp < kWideK; }

int launch_gemm_tile_kn(const void* A, const void* W, int64_t M, int N, int K, const EpiDev& ep, bool qkv,
                        hipStream_t st) {
  return qkv ? launch_tile_t<_Float16, _Float16, true, true>(A, W, M, N, K, ep, st)
             : launch_tile_t<_Float16, _Float16, false, true>(A, W, M, N, K, ep, st);
}

int launch_gemm_tile(const void* A, const void* Bt, int64_t M, int N, int Kp, const EpiDev& ep,
                     bool f16, bool out_f16, bool qkv, hipStream_t st) {
  if (f16)
    return qkv ? launch_tile_t<_Float16, _Float16, true>(A, Bt, M, N, Kp, ep, st)
               : launch_tile_t<_Float16, _Float16, false>(A, Bt, M, N, Kp, ep, st);
  if (out_f16)
    return qkv ? launch_tile_t<float, _Float16, true>(A, Bt, M, N, Kp, ep, st)
               : launch_tile_t<float, _Float16, false>(A, Bt, M, N, Kp, ep, st);
  return qkv ? launch_tile_t<float, float, true>(A, Bt, M, N, Kp, ep, st)
             : launch_tile_t<float, float, false>(A, Bt, M, N, Kp, ep, st);
}

// ---- LayerNorm prologue ----------------------------------------------------------------------
// Tiles of 16 or 32 rows on 8 wavefronts: the LDS panel of 32 normalised rows takes 64 * K bytes (100 KB at
// GPT-2 XL's 1600), three stages of weight rows 48 KB beside it -- up to K = 1024 also 96 KB, and then
// the four-way split has a 64-wide tile.  K is split over as many groups as the plain launch splits
// it (split = false: not at all, the rows that launch gives to the persistent kernel), so that the
// sums, too, are formed in the same order.  One workgroup fills a CU's
// LDS, so more workgroups than CUs take a second round: one launch of 128 rows x 768 x 3072 as 384
// tiles of 32 x 32 took 13.4 us against 9.3 for the LayerNorm launch and the plain one, as 192 of
// 32 x 64 8.3 (7.3 with the arithmetic of layernorm.h as it stands).  Normalising is a third of the
// launch, so while tiles of 16 rows still run at once, they do (24 rows x 768 x 2304: 5.6 us as 72 tiles
// of 32 x 32, 5.0 as 144 of 16 x 32), and beyond that those of 16 x 64 (us, 32 rows / so: 64 x 768 x 3072 6.4 / 6.1, 80 x
// 768 x 3072 6.9 / 6.1, 64 x 768 x 2304 5.5 / 5.0, 112 x 768 x 2304 5.9 / 5.0).
namespace {
typedef Tile<16,  32, 1, 2, 4, 3> Ln16x32;
typedef Tile<16,  64, 1, 2, 4, 3> Ln16x64;
typedef Tile<32,  32, 1, 2, 4, 3> Ln32x32;
typedef Tile<32,  64, 1, 2, 4, 3> Ln32x64w;
typedef Tile<32,  64, 1, 4, 2, 3> Ln32x64;
typedef Tile<32, 128, 1, 8, 1, 3> Ln32x128;
constexpr int kLnStages = 3 * 128 * 128;

// Index of the form that serves these sizes.
inline int pick_ln(int64_t M, int N, int K, bool split, int cus) {
  const int wk = split ? tile_cost(pick_tile(M, N, K, cus, nullptr)).wk : 1;
  if (wk < 4) return wk == 1 ? 3 : 2;
  const int64_t cols = (N + 31) / 32;
  if ((M + 15) / 16 * cols <= cus) return 4;
  if ((M + 15) / 16 * ((N + 63) / 64) <= cus) return 5;
  return K <= 1024 && (M + 31) / 32 * cols > cus ? 1 : 0;
}

template <typename T, bool QKV>
int launch_ln(const void* x, const void* Bt, int64_t M, int N, int K, const EpiDev& ep, const LnArgs& ln,
              bool split, hipStream_t st) {
  const int cus = cu_count();
  if (cus < 0) return cus;
  switch (pick_ln(M, N, K, split, cus)) {
    case 0: return launch_tile_cfg<Ln32x32, T, _Float16, QKV, true, false>(x, Bt, M, N, K, ep, ln, st);
    case 1: return launch_tile_cfg<Ln32x64w, T, _Float16, QKV, true, false>(x, Bt, M, N, K, ep, ln, st);
    case 2: return launch_tile_cfg<Ln32x64, T, _Float16, QKV, true, false>(x, Bt, M, N, K, ep, ln, st);
    case 4: return launch_tile_cfg<Ln16x32, T, _Float16, QKV, true, false>(x, Bt, M, N, K, ep, ln, st);
    case 5: return launch_tile_cfg<Ln16x64, T, _Float16, QKV, true, false>(x, Bt, M, N, K, ep, ln, st);
    default: return launch_tile_cfg<Ln32x128, T, _Float16, QKV, true, false>(x, Bt, M, N, K, ep, ln, st);
  }
}
}  // namespace

bool gemm_layernorm_supported(int64_t M, int H, bool f16) {
  if (H <= 0 || H % 64 != 0 || M <= 0) return false;
  const int nchunks = H / (f16 ? 8 : 4), lpr = lanes_per_row(nchunks);
  return (nchunks + lpr - 1) / lpr <= 4 && (size_t)kLnStages + 64 * (size_t)H <= 160 * 1024;
}

int launch_gemm_layernorm_tile(const void* x, const void* Bt, int64_t M, int N, int H, const EpiDev& ep,
                               const LnArgs& ln, bool f16, bool qkv, bool split, hipStream_t st) {
  if (f16)
    return qkv ? launch_ln<_Float16, true>(x, Bt, M, N, H, ep, ln, split, st)
               : launch_ln<_Float16, false>(x, Bt, M, N, H, ep, ln, split, st);
  return qkv ? launch_ln<float, true>(x, Bt, M, N, H, ep, ln, split, st)
             : launch_ln<float, false>(x, Bt, M, N, H, ep, ln, split, st);
}

}  // namespace gptmi
