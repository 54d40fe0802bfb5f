// LayerNorm, the q, k, v product and causal attention of short sequences in one launch: fp16, head size 64, up to
// 32 rows a sequence, rows of up to 768 (reference: gpt.py:40-51, the operators of kernels.py:104-164, 347-367 and
// 375-525).  One workgroup = one (sequence, head).
//
// What bounds the three launches it replaces (two where the LayerNorm is the product's prologue) is their own
// latency: a launch, the first loads of rows and weights, a store and a load of q, k and v of a few KB.  Here the
// rows are normalised into an LDS panel while the head's 192 weight rows are on their way, q, k and v go from the
// accumulators to LDS, and one wavefront attends.  A head's panel of weights (295 KB at 768) passes through
// one CU, and takes what the launch lasts beside the LayerNorm, so: one round of workgroups, and rows of up to 768
// (forwards of 1 x 32, 4 x 32 and 16 x 32 tokens 1024 wide 795, 860 and 1143 us, 672, 823 and 1200 in the launches
// it would replace).  At 768, replayed, in the launches / so: 1 x 24 tokens 285 / 298 us, 2 x 24 301 / 311, 3 x 30 335 /
// 331, 4 x 32 348 / 336, 8 x 24 403 / 363, 21 x 32 553 / 525: with few pairs, 12 workgroups pulling 295 KB of weights each,
// it is the longer way for the GPU, and pays where the host sets the pace (front_pays).
//
// Bits: those of the launches it stands for.  The LayerNorm is theirs (normalise_panel); the product's
// k-slices of 64 are summed in WK groups (slice t in group t % WK) that are added in order, as the tile that the
// row count picks does it, here in as many accumulator sets; scores, softmax and P.V are the ring kernel's.
//
// LDS: NST k-slices of 192 weight rows, then the panel of all k of 32 rows, both as in gemm_tile.hip.  Behind the
// product q, k and v lie where the slices were, 32 rows of 128 bytes each, in the ring kernel's swizzles.
//
// Up to 32 rows.  With 64 the panel leaves room for 60 KB of weights and the LayerNorm is twice as long: 2 x 64 tokens 381 us
// against 343 in the launches it would replace, 16 x 64 520 against 543.
#include "layernorm_panel.h"
#include "softmax.h"

namespace gptmi {

namespace {

constexpr int ROWS = 32, NST = 4, kSliceBytes = 192 * 128;

// NORMED: x is LayerNorm's output already.
template <int WK, bool NORMED>
__global__ __launch_bounds__(512, 2) void attn_front_kernel(
    const _Float16* __restrict__ x, const _Float16* __restrict__ Bt, const _Float16* __restrict__ bias,
    _Float16* __restrict__ out, int B, int heads, int L, int H, float scale, LnArgs ln, PrefetchArgs ahead) {
  constexpr int NB = 3, LPT = 3;  // a wavefront: 16 rows x 48 columns; its loads of a slice
  extern __shared__ __attribute__((aligned(1024))) char smem[];
  char* panel = smem + NST * kSliceBytes;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;
  const int lrow = lane & 15, lq = lane >> 4;

  if ((int)blockIdx.x >= B * heads) {
    prefetch_lines<512>(ahead, B * heads);
    return;
  }
  // the sequences of a head on one XCD, whose L2 holds the head's weights
  const int item = xcd_tile(blockIdx.x, B * heads);
  const int head = item / B, b = item - head * B;

  // ---- weights: slot s of a slice is row s / 8, position s % 8, which holds source unit (s % 8) ^ ((row >> 1) & 7)
  const int KT = H / 64;
  unsigned w_off[LPT];
#pragma unroll
  for (int it = 0; it < LPT; ++it) {
    const int r = it * 64 + (tid >> 3);
    w_off[it] = ((unsigned)((r >> 6) * H + head * 64 + (r & 63)) * (unsigned)H +
                 (unsigned)(((tid & 7) ^ (r >> 1 & 7)) * 8)) * 2u;
  }
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(uintptr_t)smem) + (unsigned)wave * 1024u;
  auto issue = [&](int t, int stage) __attribute__((always_inline)) {
    const char* src = (const char*)Bt + (size_t)t * 128;
#pragma unroll
    for (int it = 0; it < LPT; ++it)
      lds_dma16_base(src, w_off[it], lds0 + (unsigned)(stage * kSliceBytes) + (unsigned)(it * 8192));
  };
#pragma unroll
  for (int t = 0; t < NST; ++t)
    if (t < KT) issue(t, t);

  // ---- rows of the sequence; places past its end repeat the last one
  const _Float16* rows = x + (size_t)b * L * H;
  if constexpr (NORMED) {
    const int cpr = H / 8;
    for (int i = tid; i < ROWS * cpr; i += 512) {
      const int r = i / cpr, c = i - r * cpr;
      const h8 v = *reinterpret_cast<const h8*>(rows + (size_t)min(r, L - 1) * H + c * 8);
      *reinterpret_cast<h8*>(panel + (c >> 3) * (ROWS * 128) + r * 128 + (((c & 7) ^ (r >> 1 & 7)) << 4)) = v;
    }
  } else {
    normalise_panel<ROWS, 512>(rows, L, H, 0, ln, panel, tid);
  }
  // bias of this lane's columns 16 i + 4 lq.. of the wavefront's 48
  h4 bias_v[NB];
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int c = wn * 48 + i * 16 + lq * 4;
#pragma unroll
    for (int e = 0; e < 4; ++e) bias_v[i][e] = (_Float16)0.f;
    if (bias) bias_v[i] = *reinterpret_cast<const h4*>(bias + (c >> 6) * H + head * 64 + (c & 63));
  }
  wait_vmcnt<0>();
  __syncthreads();

  // ---- product; a slice's fragments are read while the one in front of it is multiplied
  f4 acc[WK][NB];
#pragma unroll
  for (int w = 0; w < WK; ++w)
#pragma unroll
    for (int i = 0; i < NB; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r) acc[w][i][r] = 0.f;
  const int key = lrow >> 1 & 7, a_at = (wm * 16 + lrow) * 128, b_at = (wn * 48 + lrow) * 128;
  h8 fa[2][2], fb[2][2][NB];  // [slice's parity][half slice]
  auto read = [&](int t, int stage, int to) __attribute__((always_inline)) {
    const char *pa = panel + t * (ROWS * 128) + a_at, *pb = smem + stage * kSliceBytes + b_at;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const int un = ((half * 4 + lq) ^ key) << 4;
      fa[to][half] = *reinterpret_cast<const h8*>(pa + un);
#pragma unroll
      for (int i = 0; i < NB; ++i) fb[to][half][i] = *reinterpret_cast<const h8*>(pb + i * 2048 + un);
    }
  };
  read(0, 0, 0);
  int stage = 0;
  constexpr int UN = WK > 2 ? WK : 2;
  for (int t0 = 0; t0 < KT; t0 += UN) {
#pragma unroll
    for (int u = 0; u < UN; ++u) {
      const int t = t0 + u;
      if (t < KT) {
        if (t + 1 < KT) {
          const int next = stage + 1 == NST ? 0 : stage + 1;
          // slice t + 1 has landed: NST - 2 younger ones are on their way, at the end fewer
          if (t - 1 + NST < KT) wait_vmcnt<LPT * (NST - 2)>();
          else wait_vmcnt<0>();
          block_barrier();  // for every wavefront, and everyone has slice t's fragments
          if (t + NST < KT) issue(t + NST, stage);
          read(t + 1, next, (u + 1) & 1);
          stage = next;
        }
#pragma unroll
        for (int half = 0; half < 2; ++half)
#pragma unroll
          for (int i = 0; i < NB; ++i)
            acc[u % WK][i] = __builtin_amdgcn_mfma_f32_16x16x32_f16(fb[u & 1][half][i], fa[u & 1][half], acc[u % WK][i], 0, 0, 0);
      }
    }
  }

  // ---- q, k, v in fp16 to LDS
  __syncthreads();
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int c = wn * 48 + i * 16 + lq * 4, which = c >> 6, r = wm * 16 + lrow;
    h4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      float z = acc[0][i][e];
#pragma unroll
      for (int w = 1; w < WK; ++w) z += acc[w][i][e];
      o[e] = (_Float16)(z + (float)bias_v[i][e]);
    }
    const int unit = ((c & 63) >> 3) ^ (which == 2 ? 2 * (r & 3) : r >> 1 & 7);
    *reinterpret_cast<h4*>(smem + which * 4096 + r * 128 + (unit << 4) + (c & 4) * 2) = o;
  }
  __syncthreads();

  // ---- attention of one key block that the diagonal cuts; layouts and arithmetic are the ring kernel's
  // (flash_attn.hip)
  if (wave != 0) return;
  const int ql = lane & 31, g = lane >> 5, tri_q = ql - 4 * g;
  const char *qs = smem, *ks_ = smem + 4096, *vs = smem + 8192;
  const Softmax<false> sm(scale);
  f16v s;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
  for (int ks = 0; ks < 4; ++ks) {
    const int at = ql * 128 + (((ks * 2 + g) ^ (ql >> 1 & 7)) << 4);
    s = __builtin_amdgcn_mfma_f32_32x32x16_f16(*reinterpret_cast<const h8*>(ks_ + at),
                                               *reinterpret_cast<const h8*>(qs + at), s, 0, 0, 0);
  }
  float m = -INFINITY;
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    s[r] = 8 * (r >> 2) + (r & 3) <= tri_q ? sm.score(s[r]) : -INFINITY;
    m = fmaxf(m, s[r]);
  }
  m = half_max(m);
  const float mb = sm.base(m);
  float psum = 0.f;
  h8 pf[2];
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float p = sm.weight(s[8 * tt + j], mb);
      psum += p;
      pf[tt][j] = (_Float16)p;
    }
  const NormaliseHalf<false> norm(half_sum(psum));
  f16v o[2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[i][r] = 0.f;
  const int sl = lane & 15, vrow = 4 * g + (sl >> 2);
#pragma unroll
  for (int tt = 0; tt < 2; ++tt)
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int unit = 4 * i + 2 * (lane >> 4 & 1) + ((sl & 3) >> 1);
      const char* vt = vs + (tt * 16 + vrow) * 128 + ((unit ^ (2 * (vrow & 3))) << 4) + (sl & 1) * 8;
      const h4 lo = lds_read_tr16(vt), hi = lds_read_tr16(vt + 8 * 128);
      const h8 vf = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      o[i] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, pf[tt], o[i], 0, 0, 0);
    }
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int pr = 0; pr < 2; ++pr) {
      h4 lo, hi;  // d = 32 i + 16 pr + 4 g + 0..3 and the same + 8
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        lo[j] = (_Float16)norm(o[i][8 * pr + j]);
        hi[j] = (_Float16)norm(o[i][8 * pr + 4 + j]);
      }
      const u2 xd = __builtin_bit_cast(u2, lo), yd = __builtin_bit_cast(u2, hi);
      const auto r0 = __builtin_amdgcn_permlane32_swap(xd[0], yd[0], false, false);
      const auto r1 = __builtin_amdgcn_permlane32_swap(xd[1], yd[1], false, false);
      if (ql < L)
        store_through(reinterpret_cast<u4*>(out + (((size_t)b * L + ql) * heads + head) * 64 + i * 32 + 16 * pr + 8 * g),
                      u4{r0[0], r1[0], r0[1], r1[1]});
    }
}

template <int WK, bool NORMED>
int launch_front(const void* x, const void* Bt, const void* bias, void* out, int64_t B, int heads, int L, int H,
                 float scale, const LnArgs& ln, hipStream_t st, const Prefetch* ahead) {
  auto kern = attn_front_kernel<WK, NORMED>;
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
  const size_t lds = (size_t)NST * kSliceBytes + (size_t)ROWS * H * 2;
  const int workers = (int)(B * heads), cus = cu_count();
  hipLaunchKernelGGL(kern, dim3((unsigned)(workers + front_ahead_workgroups(ahead, workers, cus))), dim3(512), lds, st,
                     (const _Float16*)x, (const _Float16*)Bt, (const _Float16*)bias, (_Float16*)out, (int)B, heads, L, H, scale,
                     ln, prefetch_args(ahead));
  return 0;
}

}  // namespace

int attn_front_split(int64_t B, int64_t L, int64_t heads, int64_t h) {
  if (L > ROWS || h > 768 || heads * 64 != h) return 0;
  const int cus = cu_count();
  const int wk = cus > 0 && B * heads <= cus ? gemm_qkv_split(B * L, (int)(3 * h), (int)h, L, (int)heads, 64) : 0;
  return wk > 0 ? wk : 0;
}

int launch_attn_front(int split, const void* x, bool normed, const void* ln_w, const void* ln_b, float eps, const void* Bt,
                      const void* bias, void* out, int64_t B, int64_t L, int64_t heads, float scale, hipStream_t st,
                      const Prefetch* ahead) {
  const int H = (int)heads * 64;
  const LnArgs ln = {ln_w, ln_b, eps, lanes_per_row(H / 8)};
  const auto go = [&](auto kernel) { return kernel(x, Bt, bias, out, B, (int)heads, (int)L, H, scale, ln, st, ahead); };
  switch (split) {
    case 4: return normed ? go(launch_front<4, true>) : go(launch_front<4, false>);
    case 2: return normed ? go(launch_front<2, true>) : go(launch_front<2, false>);
    default: return normed ? go(launch_front<1, true>) : go(launch_front<1, false>);
  }
}

}  // namespace gptmi
