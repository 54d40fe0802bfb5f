// LayerNorm as the operand prologue of a product: rows normalised into an LDS panel.
#pragma once
#include "gemm_common.h"
#include "layernorm.h"

namespace gptmi {

// LayerNorm of the BM rows from m0 on into the LDS panel, as fp16 operands: element k of row r
// goes to k-slice k / 64, row r's 128 bytes there, 16-byte unit (k % 64) / 8 ^ key(r).  A row is
// spread over LPR lanes as in layernorm_vec_kernel (same sums, same bits); rows past the end
// repeat the last row.
template <int BM, int NT, int LPR, int CH, bool FULL, typename T>
__device__ __forceinline__ void normalise_rows(const T* __restrict__ x, int M, int H, int m0,
                                               const LnArgs& ln, char* panel, int tid) {
  constexpr int VN = 16 / (int)sizeof(T);  // elements of a 16-byte chunk
  typedef T V __attribute__((ext_vector_type(VN)));
  typedef _Float16 HV __attribute__((ext_vector_type(VN)));
  constexpr int RPP = NT / LPR;  // rows per pass
  constexpr int PASSES = BM / RPP;
  static_assert(PASSES >= 1 && BM % RPP == 0, "row passes");
  const int nchunks = H / VN, ll = tid & (LPR - 1), rsub = tid / LPR;
  const V* wv = reinterpret_cast<const V*>(ln.w);
  const V* bv = reinterpret_cast<const V*>(ln.b);
  // the rows of all passes and the parameters are requested together: one memory round trip
  V tw[CH], tb[CH], t[PASSES][CH];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    int row = m0 + p * RPP + rsub;
    row = row < M ? row : M - 1;
    const V* xr = reinterpret_cast<const V*>(x + (size_t)row * H);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = ll + i * LPR;
      if (FULL || c < nchunks) t[p][i] = xr[c];
      else {
#pragma unroll
        for (int j = 0; j < VN; ++j) t[p][i][j] = (T)0.f;
      }
    }
  }
#pragma unroll
  for (int i = 0; i < CH; ++i) {
    const int c = ll + i * LPR;
    if (FULL || c < nchunks) {
      tw[i] = wv[c];
      tb[i] = bv[c];
    }
  }
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int r = p * RPP + rsub;
    float d[CH][VN], rstd;
    layernorm_stats<CH, VN, LPR, FULL>(t[p], ll, nchunks, H, ln.eps, d, rstd);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = ll + i * LPR;
      if (FULL || c < nchunks) {
        HV o;
#pragma unroll
        for (int j = 0; j < VN; ++j)
          o[j] = (_Float16)layernorm_apply(d[i][j], rstd, (float)tw[i][j], (float)tb[i][j]);
        const int k = c * VN;
        *reinterpret_cast<HV*>(panel + (k >> 6) * (BM * 128) + r * 128 +
                               ((((k >> 3) & 7) ^ ((r >> 1) & 7)) << 4) + (k & 7) * 2) = o;
      }
    }
  }
}

// At most 4 chunks per lane: rows of up to 256 chunks (gemm_layernorm_supported), 64 lanes beyond 128.
template <int BM, int NT, typename T>
__device__ __forceinline__ void normalise_panel(const T* x, int M, int H, int m0, const LnArgs& ln,
                                                char* panel, int tid) {
  const int nchunks = H * (int)sizeof(T) / 16, need = (nchunks + ln.lpr - 1) / ln.lpr;  // chunks per lane
#define GPTMI_LN_ROWS(L, FULL)                                                       \
  do {                                                                               \
    if (need <= 1) normalise_rows<BM, NT, L, 1, FULL>(x, M, H, m0, ln, panel, tid);      \
    else if (need <= 2) normalise_rows<BM, NT, L, 2, FULL>(x, M, H, m0, ln, panel, tid); \
    else if (need <= 3) normalise_rows<BM, NT, L, 3, FULL>(x, M, H, m0, ln, panel, tid); \
    else normalise_rows<BM, NT, L, 4, FULL>(x, M, H, m0, ln, panel, tid);                \
  } while (0)
  if (nchunks == need * 32 && ln.lpr == 32) GPTMI_LN_ROWS(32, true);
  else if (ln.lpr == 32) GPTMI_LN_ROWS(32, false);
  else if (sizeof(T) == 4 && nchunks == need * 64) GPTMI_LN_ROWS(64, true);  // 768 floats
  else GPTMI_LN_ROWS(64, false);
#undef GPTMI_LN_ROWS
}

}  // namespace gptmi
