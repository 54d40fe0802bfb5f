// The C ABI of libgptmi (declared in include/gptmi.h): argument validation,
// operand packing for the GEMM, and dispatch to the kernel launchers.
#include "../../include/gptmi.h"

#include <math.h>
#include <stdarg.h>
#include <stdio.h>

#include <mutex>

#include "common.h"
#include "gemm_common.h"
#include "launch.h"

namespace gptmi {

static thread_local char g_err[512] = "";

void set_error(const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
}

static int check_launch(const char* what) {
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) {
    set_error("%s: launch failed: %s", what, hipGetErrorString(e));
    return GPTMI_ERR_LAUNCH;
  }
  return GPTMI_OK;
}

static bool dtype_ok(int dtype) { return dtype == GPTMI_F32 || dtype == GPTMI_F16; }
static bool dropout_ok(float p) { return p >= 0.0f && p < 1.0f; }  // false for NaN too

static inline int64_t round_up(int64_t v, int64_t a) { return (v + a - 1) / a * a; }

// Widest output row the GEMM epilogues address: their per-lane offsets cover up to 8 rows of N
// elements of 4 bytes in an unsigned 32-bit register (8 * 2^26 * 4 = 2^31).
constexpr int kMaxN = 1 << 26;

// Workspace plan of one GEMM: where the packed weight and (if needed) the
// packed activations live.
struct LinearPlan {
  int Kp;
  bool pack_x;     // x must be converted / zero padded into the workspace
  size_t w_off, w_bytes, x_off, x_bytes, total;
};

static LinearPlan plan_linear(int64_t M, int64_t N, int64_t K, int dtype, int wlayout) {
  LinearPlan p;
  p.Kp = (int)round_up(K, 64);
  p.pack_x = !(dtype == GPTMI_F16 && p.Kp == K);
  const bool pack_w = !(wlayout == GPTMI_W_PACKED ||
                        (wlayout == GPTMI_W_NK && dtype == GPTMI_F16 && p.Kp == K));
  p.w_off = 0;
  p.w_bytes = pack_w ? (size_t)round_up(N * (int64_t)p.Kp * 2, 256) : 0;
  p.x_off = p.w_bytes;
  p.x_bytes = p.pack_x ? (size_t)round_up(M * (int64_t)p.Kp * 2, 256) : 0;
  p.total = p.w_bytes + p.x_bytes;
  return p;
}

// Packs operands as the plan says, but for a weight that the product reads in place; returns the A and Bt
// pointers the GEMM reads.
static int prepare_operands(const void* x, const void* W, int64_t M, int64_t N, int64_t K,
                            int dtype, int wlayout, bool in_place, void* workspace, size_t workspace_bytes,
                            hipStream_t st, const void** A, const void** Bt, int* Kp) {
  const LinearPlan p = plan_linear(M, N, K, dtype, wlayout);
  if (p.total > 0) {
    if (workspace == nullptr || workspace_bytes < p.total) {
      set_error("linear: workspace of %zu bytes needed, %zu given", p.total,
                workspace ? workspace_bytes : (size_t)0);
      return GPTMI_ERR_WORKSPACE;
    }
    if (((uintptr_t)workspace & 255) != 0) {
      set_error("linear: workspace must be 256-byte aligned");
      return GPTMI_ERR_WORKSPACE;
    }
  }
  const bool f16 = dtype == GPTMI_F16;
  char* ws = (char*)workspace;
  if (p.w_bytes && !in_place) {
    if (wlayout == GPTMI_W_KN)
      launch_pack_transpose(W, ws + p.w_off, (int)K, (int)N, p.Kp, f16, st);
    else
      launch_pack_rows(W, ws + p.w_off, N, (int)K, p.Kp, f16, st);
    *Bt = ws + p.w_off;
  } else {
    *Bt = W;
  }
  if (p.pack_x) {
    launch_pack_rows(x, ws + p.x_off, M, (int)K, p.Kp, f16, st);
    *A = ws + p.x_off;
  } else {
    *A = x;
  }
  *Kp = p.Kp;
  return GPTMI_OK;
}

// Scratch of gptmi_linear_static: the packed operand images that gptmi_linear puts into the
// caller's workspace.  Every GPU the library runs on holds its own copy of the array (at its own
// address) until the process ends.  In host code the array's name is only a handle for
// hipGetSymbolAddress -- never a device address -- so all uses go through static_scratch().
static __device__ __align__(256) __attribute__((used)) unsigned char scratch[GPTMI_STATIC_SCRATCH_BYTES];

constexpr int kMaxDevices = 64;

// Device address of `scratch` on the current device, resolved once per device; nullptr (and
// the error text set) on failure.
static void* static_scratch() {
  static std::mutex mu;
  static void* ptrs[kMaxDevices] = {};
  int dev = -1;
  hipError_t e = hipGetDevice(&dev);
  if (e != hipSuccess || dev < 0 || dev >= kMaxDevices) {
    set_error("linear_static: cannot identify the current device (%s, device %d)",
              hipGetErrorString(e), dev);
    return nullptr;
  }
  std::lock_guard<std::mutex> lock(mu);
  if (ptrs[dev] == nullptr) {
    void* p = nullptr;
    e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess || p == nullptr) {
      set_error("linear_static: hipGetSymbolAddress(scratch) on device %d: %s", dev,
                hipGetErrorString(e));
      return nullptr;
    }
    ptrs[dev] = p;
  }
  return ptrs[dev];
}

// The operands as the plan says, packed into `workspace` or as they are, then the GEMM.
static int product(const char* what, const void* x, const void* W, int64_t M, int64_t N, int64_t K,
                   const GemmEpilogue& ep, int wlayout, void* workspace, size_t workspace_bytes, int dtype,
                   hipStream_t st) {
  const void *A, *Bt;
  int Kp;
  const bool in_place = wlayout == GPTMI_W_KN && gemm_reads_kn(W, M, (int)N, (int)K, ep);
  int rc = prepare_operands(x, W, M, N, K, dtype, wlayout, in_place, workspace, workspace_bytes, st, &A, &Bt, &Kp);
  if (rc) return rc;
  if (((uintptr_t)A & 15) || ((uintptr_t)Bt & 15)) {
    set_error("%s: x and W must be 16-byte aligned", what);
    return GPTMI_ERR_INVALID;
  }
  rc = in_place ? launch_gemm_kn(A, Bt, M, (int)N, Kp, ep, st) : launch_gemm(A, Bt, M, (int)N, Kp, ep, st);
  if (rc) return rc;
  return check_launch(what);
}

// gptmi_linear and gptmi_linear_static behind their argument checks.
static int linear_impl(const void* x, const void* W, const void* bias, const void* residual,
                       void* out, int64_t M, int64_t N, int64_t K, int gelu, float p,
                       uint64_t seed, int wlayout, void* workspace, size_t workspace_bytes,
                       int dtype, hipStream_t st) {
  GemmEpilogue ep = {};
  ep.bias = bias;
  ep.residual = residual;
  ep.out = out;
  ep.gelu = gelu ? 1 : 0;
  ep.drop = Dropout{p, seed};
  ep.qkv = false;
  ep.f16 = dtype == GPTMI_F16;
  return product("linear", x, W, M, N, K, ep, wlayout, workspace, workspace_bytes, dtype, st);
}

static int check_linear_args(const void* x, const void* W, const void* out, int64_t M, int64_t N,
                             int64_t K, float p, int wlayout, int dtype) {
  if (!x || !W || !out || M <= 0 || N <= 0 || K <= 0 || !dtype_ok(dtype) ||
      (wlayout != GPTMI_W_KN && wlayout != GPTMI_W_NK && wlayout != GPTMI_W_PACKED)) {
    set_error("linear: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  // the epilogues form per-lane byte offsets of up to 8 rows (8 * N * 4 bytes in fp32) in 32 bits
  if (N > kMaxN || K > (1 << 30)) {
    set_error("linear: N=%lld beyond %d or K=%lld beyond 2^30", (long long)N, kMaxN, (long long)K);
    return GPTMI_ERR_UNSUPPORTED;
  }
  if (!dropout_ok(p)) {
    set_error("linear: dropout probability %g outside [0, 1)", (double)p);
    return GPTMI_ERR_INVALID;
  }
  return GPTMI_OK;
}

// ---- whole blocks ------------------------------------------------------------------------------
// A transformer block's launches behind one call.  Intermediate matrices live in the caller's
// workspace, all of them fp16: for fp16 storage that is the storage type, for fp32 storage it is the
// rounding that the next product (or the attention) applies to its operands anyway -- LayerNorm, q, k,
// v, the attention's output and the GELU's output are each written once in fp16 instead of in fp32 and
// again by a pack pass.

// Carves 256-byte aligned pieces out of a workspace.
struct Carver {
  char* base;
  size_t used;
  void* take(size_t bytes) {
    void* p = base ? base + used : nullptr;
    used += (size_t)round_up((int64_t)bytes, 256);
    return p;
  }
};

// The weight images that a block's two products read: the caller's (packed), or built into its workspace.
// K1 and K2 are multiples of 64.  in_place: the first product reads the caller's [K][N] weight as it is.
//
// The first is read as the caller has it, [K][N], wherever it can be: its rows of 3 h or 4 h hold whole lines for a
// tile, and the 0.1 to 2 us more that the product lasts are less than its share of the packing.  The second one's rows are
// short where its K is long (K = 4 h): read in place it lasts 1 to 8 us more, at widths that are a power of 2 up to 15,
// while its image is built in the LayerNorm's own launch, which has room, and stays in the memory-side cache.  Where
// there is no such launch (normalised rows handed in, layernorm_packs) it is read in place too.  With more than some 6
// rows for a column the products gain from the images what packing both costs (few_rows).  Blocks with plain
// weights from HBM, us a layer, both packed / first in place / both in place: width 512, 50 rows 27.8 / 25.6 / 25.3;
// 768: 24 34.3 / 31.4 / 33.2, 512 48.8 / 42.5 / 49.9, 2048 66.8 / 67.2 / 73.6; 896: 186 45.6 / 39.0 / 41.6;
// 1024: 24 40.2 / 37.2 / 40.8, 512 51.5 / 51.0 / 58.9, 4800 164.9 / 163.5 / 168.5; 1280: 300 63.0 / 59.1 / 65.0, 777
// 88.4 / 83.0 / 79.5; 1600: 100 60.9 / 54.6 / 54.6, 777 113.1 / 109.5 / 103.6, 1500 158.4 / 153.2 / 157.5; 2048: 300
// 105.3 / 96.6 / 103.2, 8192 808.8 / 817.2 / 808.6.  No launch to pack in: attention blocks of 768 with 300 rows handed
// in 21.4 / 18.4 / 15.5, of 1600 31.8 / 30.0 / 23.8; both blocks of 3200, 300 rows 262 / 211 / 180.  Both packed / first in
// place with dropout, many rows: 768: 3000 102.2 / 100.6, 4800 119.9 / 121.7, 8192 204.9 / 209.1; 1024: 4800 196.7 /
// 194.3, 12000 380 / 381; 1280: 6000 292.0 / 290.4, 16384 791 / 792; 1600: 8192 591.5 / 590.6, 16384 1120 / 1129.
static bool few_rows(int64_t M, int64_t h) { return M <= 6 * h; }
struct BlockWeights {
  const void *W1, *W2;
  void *ws1, *ws2;
  int K1, N1, K2, N2;
  bool packed, f16;
  bool first_in_place = false, second_in_place = false;
  const void* first() const { return packed || first_in_place ? W1 : ws1; }
  const void* second() const { return packed || second_in_place ? W2 : ws2; }
  int multiply_first(const void* A, int64_t M, const GemmEpilogue& ep, hipStream_t st) const {
    return first_in_place ? launch_gemm_kn(A, W1, M, N1, K1, ep, st) : launch_gemm(A, first(), M, N1, K1, ep, st);
  }
  int multiply_second(const void* A, int64_t M, const GemmEpilogue& ep, hipStream_t st) const {
    return second_in_place ? launch_gemm_kn(A, W2, M, N2, K2, ep, st) : launch_gemm(A, second(), M, N2, K2, ep, st);
  }
  // columns to be packed
  int n1() const { return packed || first_in_place ? 0 : N1; }
  int n2() const { return packed || second_in_place ? 0 : N2; }
  void build(hipStream_t st) const {
    if (n1() + n2() > 0) launch_pack_transpose_pair(W1, ws1, K1, n1(), W2, ws2, K2, n2(), f16, st);
  }
  // together with the block's LayerNorm, to fp16
  void build_and_normalise(const void* x, const void* ln_w, const void* ln_b, void* normed, int64_t M, int h,
                           float eps, hipStream_t st) const {
    if (n1() + n2() == 0) launch_layernorm(x, ln_w, ln_b, normed, M, h, eps, f16, true, st);
    else
      launch_layernorm_pack_pair(x, ln_w, ln_b, normed, M, h, eps, W1, ws1, K1, n1(), W2, ws2, K2, n2(), f16, st);
  }
};
// The one launch in front of a short sequences' projection: of few pairs it takes longer than the two it stands
// for, but an eager forward that small waits for the host, which then has a launch less a block.  A graph's replay
// does not.  124M, weights from HBM, us, in two launches / in one: eager 1 x 24 tokens 333 / 293, 2 x 24 333 / 305 (a pass
// that is waited for 433 / 430, 450 / 443; on a host that takes 1.5 us a launch instead of 2.5 all equal), 4 x 32 344 /
// 331; replayed 1 x 24 285 / 298, 2 x 24 301 / 311, 3 x 30 335 / 331, 4 x 32 348 / 336, 8 x 24 403 / 363, all with requests
// ahead from every idle CU.  With 64 workgroups for them (front_ahead_workgroups) the two are close: replayed in two
// launches / eager in one behind other work 1 x 8 286 / 283, 1 x 24 289 / 290, 1 x 32 290 / 290, 2 x 24 298 / 292.
static bool front_pays(int64_t pairs, hipStream_t st) {
  if (pairs > 32) return true;
  hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
  if (hipStreamIsCapturing(st, &status) != hipSuccess) (void)hipGetLastError();
  return status == hipStreamCaptureStatusNone;
}
// The split of that launch (attn_front_split), 0 where it is not taken.
static int front_split(int64_t B, int64_t L, int64_t heads, int64_t d, bool f16, hipStream_t st) {
  const int split = f16 && d == 64 ? attn_front_split(B, L, heads, heads * d) : 0;
  return split > 0 && gemm_layernorm_supported(B * L, (int)(heads * d)) && front_pays(B * heads, st) ? split : 0;
}
static size_t image_bytes(int64_t N, int64_t K, int wlayout) {
  return wlayout == GPTMI_W_PACKED ? 0 : (size_t)(N * round_up(K, 64) * 2);
}

struct AttentionPlan {
  void *normed, *q, *k, *v, *merged, *w_qkv, *w_proj;
  size_t total;
};
static AttentionPlan plan_attention(void* ws, int64_t M, int64_t h, int wlayout) {
  Carver c = {(char*)ws, 0};
  AttentionPlan p;
  const size_t mat = (size_t)(M * h * 2);
  p.normed = c.take(mat);
  p.q = c.take(mat);
  p.k = c.take(mat);
  p.v = c.take(mat);
  p.merged = c.take(mat);
  p.w_qkv = c.take(image_bytes(3 * h, h, wlayout));
  p.w_proj = c.take(image_bytes(h, h, wlayout));
  p.total = c.used;
  return p;
}

struct MlpPlan {
  void *normed, *inner, *w1, *w2;
  size_t total;
};
static MlpPlan plan_mlp(void* ws, int64_t M, int64_t h, int64_t inner, int wlayout) {
  Carver c = {(char*)ws, 0};
  MlpPlan p;
  p.normed = c.take((size_t)(M * h * 2));
  p.inner = c.take((size_t)(M * inner * 2));
  p.w1 = c.take(image_bytes(inner, h, wlayout));
  p.w2 = c.take(image_bytes(h, inner, wlayout));
  p.total = c.used;
  return p;
}

// The generator's offsets are 32-bit numbers: a mask longer than that would repeat itself.
constexpr int64_t kMaxMaskBits = 1ll << 32;

// What the block functions take: row widths that are multiples of 64 (every operand is then read in
// place), up to the LayerNorm kernel's 8192.
static int check_block(const char* what, int64_t M, int64_t h, float p, const void* keep,
                       int64_t keep_bits, int64_t keep_need, int wlayout, int dtype, const void* ws,
                       size_t ws_bytes, size_t need) {
  if (M <= 0 || h <= 0 || !dtype_ok(dtype) || (wlayout != GPTMI_W_KN && wlayout != GPTMI_W_PACKED)) {
    set_error("%s: invalid argument", what);
    return GPTMI_ERR_INVALID;
  }
  if (h % 64 != 0 || h > 8192) {
    set_error("%s: row width %lld is not a multiple of 64 up to 8192", what, (long long)h);
    return GPTMI_ERR_UNSUPPORTED;
  }
  if (!dropout_ok(p)) {
    set_error("%s: dropout probability %g outside [0, 1)", what, (double)p);
    return GPTMI_ERR_INVALID;
  }
  if (keep != nullptr && (keep_bits < keep_need || keep_need > kMaxMaskBits || ((uintptr_t)keep & 3) != 0)) {
    set_error("%s: a dropout mask of %lld bits (at most 2^32), 4-byte aligned, needed (%lld given)", what,
              (long long)keep_need, (long long)keep_bits);
    return GPTMI_ERR_INVALID;
  }
  if (ws == nullptr || ws_bytes < need || ((uintptr_t)ws & 255) != 0) {
    set_error("%s: workspace of %zu bytes, 256-byte aligned, needed (%zu given)", what, need,
              ws ? ws_bytes : (size_t)0);
    return GPTMI_ERR_WORKSPACE;
  }
  return GPTMI_OK;
}

// The limits of the product's row index and of the attention's grid.
static int check_grid(const char* what, int64_t B, int64_t L, int64_t heads) {
  if (B * heads > 0x7fffffffll || L > (1 << 24) || B * L >= (1ll << 31) - 512) {
    set_error("%s: B*heads=%lld, L=%lld or B*L=%lld beyond the grid limits", what, (long long)(B * heads),
              (long long)L, (long long)(B * L));
    return GPTMI_ERR_UNSUPPORTED;
  }
  return GPTMI_OK;
}

// The LayerNorm prologue reads rows and parameters in 16-byte units; the block functions run the
// LayerNorm kernel in front of the product where one of them lies otherwise.
static bool prologue_aligned(const void* x, const void* ln_w, const void* ln_b) {
  return (((uintptr_t)x | (uintptr_t)ln_w | (uintptr_t)ln_b) & 15) == 0;
}

// fp32 models' blocks with packed weights run their LayerNorm inside the product behind it without being asked, up to
// the rows that FusedGPT asks for it at in fp16 (gpt.LN_PROLOGUE_MAX_ROWS and those beside it; a caller declines with -1):
// a launch less, the same bits.  Forwards, two launches / one, weights from HBM, us, queued behind other work | replayed |
// waited for: 124M 1 x 24 tokens 297 / 284 | 306 / 292 | 473 / 444, 1 x 80 326 / 304 | 333 / 312 | 478 / 445, 1 x 112 348 /
// 335 | 358 / 343 | 506 / 470, 2 x 64 357 / 357 | 364 / 366 | 508 / 493, 1 x 144 371 / 364 | 379 / 373 | 522 / 500, 1 x 160 380 /
// 374 | 390 / 383 | 531 / 503, replayed 1 x 192 418 / 480; 1024 wide 1 x 8 626 / 627 | 635 / 637 | 842 / 777, 1 x 24 643 / 631 |
// 651 / 639 | 845 / 772, 1 x 64 686 / 675 | 690 / 682 | 868 / 805, 2 x 64 797 / 806 on the GPU.
static bool prologue_f32(int64_t M, int64_t h, bool packed, float p) {
  return packed && p == 0.f && h <= 1024 && M <= (h <= 768 ? 160 : 64) && gemm_layernorm_supported(M, (int)h, false);
}

}  // namespace gptmi

using namespace gptmi;

extern "C" {

int gptmi_version(void) { return GPTMI_VERSION; }

const char* gptmi_last_error(void) { return g_err; }

int gptmi_embed(const int64_t* ids, const void* wte, const void* wpe, void* out, int64_t B,
                int64_t L, int64_t V, int64_t P, int64_t H, float p, uint64_t seed,
                int dtype, void* stream) {
  if (!ids || !wte || !wpe || !out || B <= 0 || L <= 0 || V <= 0 || P <= 0 || H <= 0 ||
      !dtype_ok(dtype)) {
    set_error("embed: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (L > P) {
    set_error("embed: sequence length %lld exceeds the %lld position rows", (long long)L,
              (long long)P);
    return GPTMI_ERR_INVALID;
  }
  if (H > (1 << 24)) {
    set_error("embed: H=%lld too large", (long long)H);
    return GPTMI_ERR_UNSUPPORTED;
  }
  if (!dropout_ok(p)) {
    set_error("embed: dropout probability %g outside [0, 1)", (double)p);
    return GPTMI_ERR_INVALID;
  }
  launch_embed(ids, wte, wpe, out, B * L, L, V, (int)H, Dropout{p, seed}, dtype == GPTMI_F16,
               (hipStream_t)stream);
  return check_launch("embed");
}

int gptmi_embed_layernorm(const int64_t* ids, const void* wte, const void* wpe,
                          const void* ln_w, const void* ln_b, void* emb, void* out, int64_t B,
                          int64_t L, int64_t V, int64_t P, int64_t H, float eps, int dtype,
                          void* stream) {
  if (!ids || !wte || !wpe || !ln_w || !ln_b || !emb || !out || B <= 0 || L <= 0 || V <= 0 ||
      P <= 0 || H <= 0 || !dtype_ok(dtype)) {
    set_error("embed_layernorm: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (L > P) {
    set_error("embed_layernorm: sequence length %lld exceeds the %lld position rows",
              (long long)L, (long long)P);
    return GPTMI_ERR_INVALID;
  }
  if (H > 8192) {
    set_error("embed_layernorm: H=%lld beyond the supported 8192", (long long)H);
    return GPTMI_ERR_UNSUPPORTED;
  }
  const bool f16 = dtype == GPTMI_F16;
  hipStream_t st = (hipStream_t)stream;
  if (!launch_embed_layernorm(ids, wte, wpe, ln_w, ln_b, emb, out, B * L, L, V, (int)H, eps, f16,
                              st)) {
    // rows the fused kernel does not hold in registers: the two kernels, same results
    launch_embed(ids, wte, wpe, emb, B * L, L, V, (int)H, Dropout{0.0f, 1337}, f16, st);
    launch_layernorm(emb, ln_w, ln_b, out, B * L, (int)H, eps, f16, false, st);
  }
  return check_launch("embed_layernorm");
}

int gptmi_layernorm(const void* x, const void* w, const void* b, void* out, int64_t M,
                    int64_t H, float eps, int dtype, void* stream) {
  if (!x || !w || !b || !out || M <= 0 || H <= 0 || !dtype_ok(dtype)) {
    set_error("layernorm: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (H > 8192) {
    set_error("layernorm: H=%lld beyond the supported 8192", (long long)H);
    return GPTMI_ERR_UNSUPPORTED;
  }
  launch_layernorm(x, w, b, out, M, (int)H, eps, dtype == GPTMI_F16, false, (hipStream_t)stream);
  return check_launch("layernorm");
}

int gptmi_softmax(const void* x, void* out, int64_t M, int64_t H, int dtype, void* stream) {
  if (!x || !out || M <= 0 || H <= 0 || !dtype_ok(dtype)) {
    set_error("softmax: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (H > 8192) {
    set_error("softmax: H=%lld beyond the supported 8192", (long long)H);
    return GPTMI_ERR_UNSUPPORTED;
  }
  launch_softmax(x, out, M, (int)H, dtype == GPTMI_F16, (hipStream_t)stream);
  return check_launch("softmax");
}

size_t gptmi_linear_workspace_bytes(int64_t M, int64_t N, int64_t K, int dtype, int wlayout) {
  if (M <= 0 || N <= 0 || K <= 0 || !dtype_ok(dtype)) return 0;
  return plan_linear(M, N, K, dtype, wlayout).total;
}

size_t gptmi_packed_weight_bytes(int64_t N, int64_t K) {
  if (N <= 0 || K <= 0) return 0;
  return (size_t)round_up(N * round_up(K, 64) * 2, 256);
}

int gptmi_pack_weight(const void* W, void* packed, int64_t N, int64_t K, int wlayout, int dtype,
                      void* stream) {
  if (!W || !packed || N <= 0 || K <= 0 || !dtype_ok(dtype) ||
      (wlayout != GPTMI_W_KN && wlayout != GPTMI_W_NK) || N > (1 << 30) || K > (1 << 30)) {
    set_error("pack_weight: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (((uintptr_t)packed & 255) != 0) {
    set_error("pack_weight: destination must be 256-byte aligned");
    return GPTMI_ERR_INVALID;
  }
  const int Kp = (int)round_up(K, 64);
  if (wlayout == GPTMI_W_KN)
    launch_pack_transpose(W, packed, (int)K, (int)N, Kp, dtype == GPTMI_F16, (hipStream_t)stream);
  else
    launch_pack_rows(W, packed, N, (int)K, Kp, dtype == GPTMI_F16, (hipStream_t)stream);
  return check_launch("pack_weight");
}

int gptmi_linear(const void* x, const void* W, const void* bias, const void* residual,
                 void* out, int64_t M, int64_t N, int64_t K, int gelu, float p,
                 uint64_t seed, int wlayout, void* workspace, size_t workspace_bytes,
                 int dtype, void* stream) {
  const int rc = check_linear_args(x, W, out, M, N, K, p, wlayout, dtype);
  if (rc) return rc;
  return linear_impl(x, W, bias, residual, out, M, N, K, gelu, p, seed, wlayout, workspace,
                     workspace_bytes, dtype, (hipStream_t)stream);
}

size_t gptmi_linear_static_capacity(void) { return GPTMI_STATIC_SCRATCH_BYTES; }

int gptmi_linear_static(const void* x, const void* W, const void* bias, const void* residual,
                        void* out, int64_t M, int64_t N, int64_t K, int gelu, float p,
                        uint64_t seed, int wlayout, int dtype, void* stream) {
  const int rc = check_linear_args(x, W, out, M, N, K, p, wlayout, dtype);
  if (rc) return rc;
  // the size check comes before anything touches the device
  const size_t need = plan_linear(M, N, K, dtype, wlayout).total;
  if (need > (size_t)GPTMI_STATIC_SCRATCH_BYTES) {
    set_error("linear_static: these sizes need %zu bytes of packed operands, the built-in "
              "scratch holds %zu; use gptmi_linear with a workspace, or pack the weight once "
              "(GPTMI_W_PACKED)",
              need, (size_t)GPTMI_STATIC_SCRATCH_BYTES);
    return GPTMI_ERR_WORKSPACE;
  }
  void* ws = nullptr;
  if (need > 0) {
    ws = static_scratch();
    if (ws == nullptr) return GPTMI_ERR_LAUNCH;
  }
  return linear_impl(x, W, bias, residual, out, M, N, K, gelu, p, seed, wlayout, ws,
                     (size_t)GPTMI_STATIC_SCRATCH_BYTES, dtype, (hipStream_t)stream);
}

int gptmi_linear_qkv(const void* x, const void* W, const void* bias, void* q, void* k,
                     void* v, int64_t B, int64_t L, int64_t heads, int64_t d, int64_t K,
                     int wlayout, void* workspace, size_t workspace_bytes, int dtype,
                     void* stream) {
  if (!x || !W || !q || !k || !v || B <= 0 || L <= 0 || heads <= 0 || d <= 0 || K <= 0 ||
      !dtype_ok(dtype) || (wlayout != GPTMI_W_KN && wlayout != GPTMI_W_PACKED)) {
    set_error("linear_qkv: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (d % 8 != 0) {
    set_error("linear_qkv: head size %lld must be a multiple of 8", (long long)d);
    return GPTMI_ERR_UNSUPPORTED;
  }
  const int64_t M = B * L, N = 3 * heads * d;
  if (N > kMaxN || K > (1 << 30)) {
    set_error("linear_qkv: N=%lld beyond %d or K=%lld beyond 2^30", (long long)N, kMaxN,
              (long long)K);
    return GPTMI_ERR_UNSUPPORTED;
  }
  hipStream_t st = (hipStream_t)stream;
  GemmEpilogue ep = {};
  ep.bias = bias;
  ep.q = q;
  ep.k = k;
  ep.v = v;
  ep.L = L;
  ep.heads = (int)heads;
  ep.d = (int)d;
  ep.qkv = true;
  ep.f16 = dtype == GPTMI_F16;
  return product("linear_qkv", x, W, M, N, K, ep, wlayout, workspace, workspace_bytes, dtype, st);
}

// Shared argument checks of the two LayerNorm-prologue entry points; K = H.
static int check_layernorm_linear(const char* what, const void* x, const void* ln_w,
                                  const void* ln_b, const void* W, int64_t M, int64_t N,
                                  int64_t K, int dtype) {
  if (!x || !ln_w || !ln_b || !W || M <= 0 || N <= 0 || K <= 0 || !dtype_ok(dtype)) {
    set_error("%s: invalid argument", what);
    return GPTMI_ERR_INVALID;
  }
  if (N > kMaxN) {
    set_error("%s: N=%lld beyond %d", what, (long long)N, kMaxN);
    return GPTMI_ERR_UNSUPPORTED;
  }
  if (dtype != GPTMI_F16 || K > (1 << 20) || !gemm_layernorm_supported(M, (int)K)) {
    set_error("%s: fp16 storage and a row width that is a multiple of 64 and fits the LDS panel "
              "(gptmi_layernorm_linear_supported); use gptmi_layernorm + gptmi_linear", what);
    return GPTMI_ERR_UNSUPPORTED;
  }
  return GPTMI_OK;
}

int gptmi_layernorm_linear_supported(int64_t M, int64_t K, int dtype) {
  return dtype == GPTMI_F16 && K > 0 && K <= (1 << 20) && gemm_layernorm_supported(M, (int)K) ? 1 : 0;
}

int gptmi_layernorm_linear(const void* x, const void* ln_w, const void* ln_b, float eps,
                           const void* W_packed, const void* bias, void* out, int64_t M,
                           int64_t N, int64_t K, int gelu, int dtype, void* stream) {
  int rc = check_layernorm_linear("layernorm_linear", x, ln_w, ln_b, W_packed, M, N, K, dtype);
  if (rc) return rc;
  if (!out) {
    set_error("layernorm_linear: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  GemmEpilogue ep = {};
  ep.bias = bias;
  ep.out = out;
  ep.gelu = gelu ? 1 : 0;
  ep.drop = Dropout{0.0f, 1337};
  ep.qkv = false;
  ep.f16 = true;
  rc = launch_gemm_layernorm(x, ln_w, ln_b, eps, W_packed, M, (int)N, (int)K, ep,
                             (hipStream_t)stream);
  if (rc) return rc == -2 ? GPTMI_ERR_INVALID : rc;
  return check_launch("layernorm_linear");
}

int gptmi_layernorm_linear_qkv(const void* x, const void* ln_w, const void* ln_b, float eps,
                               const void* W_packed, const void* bias, void* q, void* k, void* v,
                               int64_t B, int64_t L, int64_t heads, int64_t d, int64_t K,
                               int dtype, void* stream) {
  if (B <= 0 || L <= 0 || heads <= 0 || d <= 0 || !q || !k || !v) {
    set_error("layernorm_linear_qkv: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (d % 8 != 0) {
    set_error("layernorm_linear_qkv: head size %lld must be a multiple of 8", (long long)d);
    return GPTMI_ERR_UNSUPPORTED;
  }
  const int64_t M = B * L, N = 3 * heads * d;
  int rc = check_layernorm_linear("layernorm_linear_qkv", x, ln_w, ln_b, W_packed, M, N, K, dtype);
  if (rc) return rc;
  GemmEpilogue ep = {};
  ep.bias = bias;
  ep.q = q;
  ep.k = k;
  ep.v = v;
  ep.L = L;
  ep.heads = (int)heads;
  ep.d = (int)d;
  ep.drop = Dropout{0.0f, 1337};
  ep.qkv = true;
  ep.f16 = true;
  rc = launch_gemm_layernorm(x, ln_w, ln_b, eps, W_packed, M, (int)N, (int)K, ep,
                             (hipStream_t)stream);
  if (rc) return rc == -2 ? GPTMI_ERR_INVALID : rc;
  return check_launch("layernorm_linear_qkv");
}

int gptmi_flash_attn(const void* q, const void* k, const void* v, void* out, int64_t B,
                     int64_t N, int64_t Lq, int64_t Lk, int64_t d, float scale, float p,
                     uint64_t seed, int olayout, int dtype, void* stream) {
  if (!q || !k || !v || !out || B <= 0 || N <= 0 || Lq <= 0 || Lk <= 0 || d <= 0 ||
      !dtype_ok(dtype) || (olayout != GPTMI_O_BNLD && olayout != GPTMI_O_BLND)) {
    set_error("flash_attn: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  if (!dropout_ok(p)) {
    set_error("flash_attn: dropout probability %g outside [0, 1)", (double)p);
    return GPTMI_ERR_INVALID;
  }
  if (((uintptr_t)q & 15) || ((uintptr_t)k & 15) || ((uintptr_t)v & 15) ||
      ((uintptr_t)out & 15)) {
    set_error("flash_attn: q, k, v and out must be 16-byte aligned");
    return GPTMI_ERR_INVALID;
  }
  int rc = launch_flash_attn(q, k, v, out, B, N, Lq, Lk, (int)d, scale, Dropout{p, seed},
                             olayout == GPTMI_O_BLND,
                             dtype == GPTMI_F16, (hipStream_t)stream);
  if (rc) return rc;
  return check_launch("flash_attn");
}

size_t gptmi_dropout_mask_bytes(int64_t n) {
  return n > 0 && n <= kMaxMaskBits ? (size_t)((n + 31) / 32 + 4) * 4 : 0;
}

int gptmi_dropout_mask(void* mask, int64_t n, float p, uint64_t seed, void* stream) {
  if (!mask || n <= 0 || n > kMaxMaskBits || ((uintptr_t)mask & 3) != 0 || !dropout_ok(p)) {
    set_error("dropout_mask: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  launch_dropout_mask(mask, (n + 31) / 32 + 4, Dropout{p, seed}, (hipStream_t)stream);
  return check_launch("dropout_mask");
}

size_t gptmi_attention_block_workspace_bytes(int64_t B, int64_t L, int64_t heads, int64_t d,
                                             int wlayout) {
  if (B <= 0 || L <= 0 || heads <= 0 || d <= 0) return 0;
  return plan_attention(nullptr, B * L, heads * d, wlayout).total;
}

// What gptmi_blocks knows of a layer: front_split, the same for all of them, and what to request ahead.
struct Stack {
  int front;
  Prefetch ahead;
};

static int attention_block(const void* x, const void* normed, const void* ln_w, const void* ln_b, float eps,
                          const void* W_qkv, const void* b_qkv, const void* W_proj, const void* b_proj,
                          void* out, int64_t B, int64_t L, int64_t heads, int64_t d, float p,
                          uint64_t seed, const void* keep, int64_t keep_bits, int fuse_layernorm, int wlayout, void* workspace,
                          size_t workspace_bytes, int dtype, void* stream, const Stack* stack) {
  const Prefetch* ahead = stack ? &stack->ahead : nullptr;
  if (!x || !ln_w || !ln_b || !W_qkv || !W_proj || !out || B <= 0 || L <= 0 || heads <= 0 || d <= 0) {
    set_error("attention_block: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  // before the product, whose scatter stores 8 columns of a head at a time
  if (d != 16 && d != 32 && d != 64 && d != 128 && d != 256) {
    set_error("attention_block: head size %lld not built (16, 32, 64, 128 and 256 are)", (long long)d);
    return GPTMI_ERR_UNSUPPORTED;
  }
  const int64_t M = B * L, h = heads * d;
  const AttentionPlan pl = plan_attention(workspace, M, h, wlayout);
  int rc = check_block("attention_block", M, h, p, keep, keep_bits, M * h > L * L ? M * h : L * L, wlayout,
                       dtype, workspace, workspace_bytes, pl.total);
  if (!rc) rc = check_grid("attention_block", B, L, heads);
  if (rc) return rc;
  const bool f16 = dtype == GPTMI_F16;
  hipStream_t st = (hipStream_t)stream;
  BlockWeights bw = {W_qkv, W_proj, pl.w_qkv, pl.w_proj, (int)h, (int)(3 * h), (int)h, (int)h,
                     wlayout == GPTMI_W_PACKED, f16};
  GemmEpilogue ep = {};
  ep.bias = b_qkv;
  ep.q = pl.q;
  ep.k = pl.k;
  ep.v = pl.v;
  ep.L = L;
  ep.heads = (int)heads;
  ep.d = (int)d;
  ep.qkv = true;
  ep.f16 = f16;
  ep.out_f16 = true;
  bool prologue = fuse_layernorm > 0 && !normed;
  if (prologue) {
    if (!f16 || !gemm_layernorm_supported(M, (int)h)) {
      set_error("attention_block: the LayerNorm prologue takes fp16 storage and the row widths of "
                "gptmi_layernorm_linear_supported");
      return GPTMI_ERR_UNSUPPORTED;
    }
  } else if (!f16 && !normed && fuse_layernorm == 0) {
    prologue = prologue_f32(M, h, bw.packed, p);
  }
  prologue = prologue && prologue_aligned(x, ln_w, ln_b);
  const Dropout drop = {p, seed, keep};
  GemmEpilogue eo = {};
  eo.bias = b_proj;
  eo.residual = x;
  eo.out = out;
  eo.drop = drop;
  eo.f16 = f16;
  bw.first_in_place = !bw.packed && !prologue && (normed || few_rows(M, h)) && gemm_reads_kn(W_qkv, M, (int)(3 * h), (int)h, ep);
  bw.second_in_place = bw.first_in_place && (normed || !layernorm_packs((int)h)) && gemm_reads_kn(W_proj, M, (int)h, (int)h, eo);
  const void *Bq = bw.first(), *Bp = bw.second();
  if (((uintptr_t)Bq & 15) || ((uintptr_t)Bp & 15)) {
    set_error("attention_block: the weights must be 16-byte aligned");
    return GPTMI_ERR_INVALID;
  }
  const float scale = (float)(1.0 / sqrt((double)d));
  // short sequences: everything in front of the projection in one launch
  const void* rows = normed ? normed : x;
  const int front = !bw.packed || p > 0.f || !prologue_aligned(rows, ln_w, ln_b) || ((uintptr_t)b_qkv & 15) != 0 ? 0
                    : stack ? stack->front : front_split(B, L, heads, d, f16, st);
  if (front > 0) {
    rc = launch_attn_front(front, rows, normed != nullptr, ln_w, ln_b, eps, Bq, b_qkv, pl.merged, B, L, heads, scale, st, ahead);
  } else if (prologue) {
    bw.build(st);
    rc = launch_gemm_layernorm(x, ln_w, ln_b, eps, Bq, M, (int)(3 * h), (int)h, ep, st);
  } else {
    const void* A = pl.normed;
    if (!normed) {
      bw.build_and_normalise(x, ln_w, ln_b, pl.normed, M, (int)h, eps, st);
    } else {
      bw.build(st);
      if (f16 && ((uintptr_t)normed & 15) == 0) A = normed;
      else launch_pack_rows(normed, pl.normed, M, (int)h, (int)h, f16, st);
    }
    rc = bw.multiply_first(A, M, ep, st);
  }
  if (rc) return rc;
  if (front == 0) {
    rc = f16 ? launch_flash_attn(pl.q, pl.k, pl.v, pl.merged, B, heads, L, L, (int)d, scale, drop, true, true, st, ahead)
             : launch_flash_attn_operands(pl.q, pl.k, pl.v, pl.merged, B, heads, L, (int)d, scale, drop, st, ahead);
    if (rc) return rc;
  }
  rc = bw.multiply_second(pl.merged, M, eo, st);
  if (rc) return rc;
  return check_launch("attention_block");
}

int gptmi_attention_block(const void* x, const void* normed, const void* ln_w, const void* ln_b, float eps,
                          const void* W_qkv, const void* b_qkv, const void* W_proj, const void* b_proj,
                          void* out, int64_t B, int64_t L, int64_t heads, int64_t d, float p, uint64_t seed,
                          const void* keep, int64_t keep_bits, int fuse_layernorm, int wlayout,
                          void* workspace, size_t workspace_bytes, int dtype, void* stream) {
  return attention_block(x, normed, ln_w, ln_b, eps, W_qkv, b_qkv, W_proj, b_proj, out, B, L, heads, d, p, seed,
                         keep, keep_bits, fuse_layernorm, wlayout, workspace, workspace_bytes, dtype, stream, nullptr);
}

size_t gptmi_mlp_block_workspace_bytes(int64_t M, int64_t H, int64_t inner, int wlayout) {
  if (M <= 0 || H <= 0 || inner <= 0) return 0;
  return plan_mlp(nullptr, M, H, inner, wlayout).total;
}

int gptmi_mlp_block(const void* x, const void* ln_w, const void* ln_b, float eps, const void* W1,
                    const void* b1, const void* W2, const void* b2, void* out, int64_t M, int64_t H,
                    int64_t inner, float p, uint64_t seed, const void* keep, int64_t keep_bits,
                    int fuse_layernorm, int wlayout, void* workspace, size_t workspace_bytes, int dtype, void* stream) {
  if (!x || !ln_w || !ln_b || !W1 || !W2 || !out || inner <= 0 || inner % 64 != 0 || inner > kMaxN) {
    set_error("mlp_block: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  const MlpPlan pl = plan_mlp(workspace, M, H, inner, wlayout);
  int rc = check_block("mlp_block", M, H, p, keep, keep_bits, M * (inner > H ? inner : H), wlayout, dtype,
                       workspace, workspace_bytes, pl.total);
  if (rc) return rc;
  const bool f16 = dtype == GPTMI_F16;
  hipStream_t st = (hipStream_t)stream;
  BlockWeights bw = {W1, W2, pl.w1, pl.w2, (int)H, (int)inner, (int)inner, (int)H,
                     wlayout == GPTMI_W_PACKED, f16};
  const Dropout drop = {p, seed, keep};
  GemmEpilogue e1 = {};
  e1.bias = b1;
  e1.out = pl.inner;
  e1.gelu = 1;
  e1.drop = drop;
  e1.f16 = f16;
  e1.out_f16 = true;
  bool prologue = fuse_layernorm > 0;
  if (prologue) {
    if (!f16 || p > 0.f || !gemm_layernorm_supported(M, (int)H)) {
      set_error("mlp_block: the LayerNorm prologue takes fp16 storage, no dropout and the row widths of "
                "gptmi_layernorm_linear_supported");
      return GPTMI_ERR_UNSUPPORTED;
    }
  } else if (!f16 && fuse_layernorm == 0) {
    prologue = prologue_f32(M, H, bw.packed, p);
  }
  prologue = prologue && prologue_aligned(x, ln_w, ln_b);
  GemmEpilogue e2 = {};
  e2.bias = b2;
  e2.residual = x;
  e2.out = out;
  e2.drop = drop;
  e2.f16 = f16;
  bw.first_in_place = !bw.packed && !prologue && few_rows(M, H) && gemm_reads_kn(W1, M, (int)inner, (int)H, e1);
  bw.second_in_place = bw.first_in_place && !layernorm_packs((int)H) && gemm_reads_kn(W2, M, (int)H, (int)inner, e2);
  const void *B1 = bw.first(), *B2 = bw.second();
  if (((uintptr_t)B1 & 15) || ((uintptr_t)B2 & 15)) {
    set_error("mlp_block: the weights must be 16-byte aligned");
    return GPTMI_ERR_INVALID;
  }
  if (prologue) {
    bw.build(st);
    rc = launch_gemm_layernorm(x, ln_w, ln_b, eps, B1, M, (int)inner, (int)H, e1, st);
  } else {
    bw.build_and_normalise(x, ln_w, ln_b, pl.normed, M, (int)H, eps, st);
    rc = bw.multiply_first(pl.normed, M, e1, st);
  }
  if (rc) return rc;
  rc = bw.multiply_second(pl.inner, M, e2, st);
  if (rc) return rc;
  return check_launch("mlp_block");
}

// What the calls of the layers would refuse one by one, with the layers in front of them launched.
static int check_blocks(const void* const* params, int64_t n, int64_t B, int64_t L, int64_t heads, int64_t h,
                        int64_t inner, int fuse_layernorm, int dtype) {
  if (inner % 64 != 0 || inner > kMaxN) {
    set_error("blocks: inner width %lld is not a multiple of 64 up to %d", (long long)inner, kMaxN);
    return GPTMI_ERR_INVALID;
  }
  for (int64_t i = 0; i < n; ++i) {
    const void* const* p = params + 12 * i;
    for (const int j : {0, 1, 2, 4, 6, 7, 8, 10})
      if (p[j] == nullptr) {
        set_error("blocks: pointer %d of layer %lld is NULL", j, (long long)i);
        return GPTMI_ERR_INVALID;
      }
    if (((uintptr_t)p[2] | (uintptr_t)p[4] | (uintptr_t)p[8] | (uintptr_t)p[10]) & 15) {
      set_error("blocks: the weights of layer %lld must be 16-byte aligned", (long long)i);
      return GPTMI_ERR_INVALID;
    }
  }
  if (fuse_layernorm > 0 && (dtype != GPTMI_F16 || !gemm_layernorm_supported(B * L, (int)h))) {
    set_error("blocks: the LayerNorm prologue takes fp16 storage and the row widths of "
              "gptmi_layernorm_linear_supported");
    return GPTMI_ERR_UNSUPPORTED;
  }
  return check_grid("blocks", B, L, heads);
}

// Two matrices of the residual stream in front of the larger block's workspace.
size_t gptmi_blocks_workspace_bytes(int64_t B, int64_t L, int64_t heads, int64_t d, int64_t inner, int dtype) {
  if (B <= 0 || L <= 0 || heads <= 0 || d <= 0 || inner <= 0 || !dtype_ok(dtype)) return 0;
  const int64_t M = B * L, h = heads * d;
  const size_t a = plan_attention(nullptr, M, h, GPTMI_W_PACKED).total;
  const size_t m = plan_mlp(nullptr, M, h, inner, GPTMI_W_PACKED).total;
  return 2 * (size_t)round_up(M * h * (dtype == GPTMI_F16 ? 2 : 4), 256) + (a > m ? a : m);
}

int gptmi_blocks(const void* x, const void* normed, const void* const* params, int64_t n, float eps,
                 void* out, int64_t B, int64_t L, int64_t heads, int64_t d, int64_t inner,
                 int fuse_layernorm, void* workspace, size_t workspace_bytes, int dtype, void* stream) {
  if (!x || !params || !out || n <= 0 || B <= 0 || L <= 0 || heads <= 0 || d <= 0 || inner <= 0 ||
      !dtype_ok(dtype)) {
    set_error("blocks: invalid argument");
    return GPTMI_ERR_INVALID;
  }
  const size_t need = gptmi_blocks_workspace_bytes(B, L, heads, d, inner, dtype);
  if (workspace == nullptr || workspace_bytes < need || ((uintptr_t)workspace & 255) != 0) {
    set_error("blocks: workspace of %zu bytes, 256-byte aligned, needed (%zu given)", need,
              workspace ? workspace_bytes : (size_t)0);
    return GPTMI_ERR_WORKSPACE;
  }
  const int64_t M = B * L, h = heads * d;
  if (const int rc = check_blocks(params, n, B, L, heads, h, inner, fuse_layernorm, dtype)) return rc;
  Carver c = {(char*)workspace, 0};
  const size_t mat = (size_t)(M * h * (dtype == GPTMI_F16 ? 2 : 4));
  void *mid = c.take(mat), *next = c.take(mat);
  char* ws = (char*)workspace + c.used;
  const size_t ws_bytes = workspace_bytes - c.used;
  Stack stack = {front_split(B, L, heads, d, dtype == GPTMI_F16, (hipStream_t)stream), Prefetch()};
  const AheadPlan plan = plan_ahead(L, B * heads > cu_count() - 64 || stack.front > 0, h, inner);
  for (int64_t i = 0; i < n; ++i) {
    const void* const* p = params + 12 * i;
    stack.ahead = weights_ahead(p, i + 1 == n, plan);
    int rc = attention_block(x, i == 0 ? normed : nullptr, p[0], p[1], eps, p[2], p[3], p[4], p[5], mid, B, L, heads,
                             d, 0.0f, 1337, nullptr, 0, fuse_layernorm, GPTMI_W_PACKED, ws, ws_bytes, dtype, stream, &stack);
    if (rc) return rc;
    // x is not read again: the layer's output may take its place
    void* y = i + 1 == n ? out : next;
    rc = gptmi_mlp_block(mid, p[6], p[7], eps, p[8], p[9], p[10], p[11], y, M, h, inner, 0.0f, 1337, nullptr, 0,
                         fuse_layernorm, GPTMI_W_PACKED, ws, ws_bytes, dtype, stream);
    if (rc) return rc;
    x = y;
  }
  return GPTMI_OK;
}

}  // extern "C"
