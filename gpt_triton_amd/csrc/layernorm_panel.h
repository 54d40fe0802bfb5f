// LayerNorm as the operand prologue of a product: rows normalised into an LDS panel.
#pragma once
#include "gemm_common.h"
#include "layernorm.h"

namespace gptmi {

// LayerNorm of the BM rows from m0 on into the LDS panel, as fp16 operands: element k of row r
// goes to k-slice k / 64, row r's 128 bytes there, 16-byte unit (k % 64) / 8 ^ key(r).  A row is
// spread over LPR lanes as in layernorm_vec_kernel (same sums, same bits); rows past the end
// repeat the last row.
template <int BM, int NT, int LPR, int CH, bool FULL>
__device__ __forceinline__ void normalise_rows(const _Float16* __restrict__ x, int M, int H, int m0,
                                               const LnArgs& ln, char* panel, int tid) {
  constexpr int RPP = NT / LPR;  // rows per pass
  constexpr int PASSES = BM / RPP;
  static_assert(PASSES >= 1 && BM % RPP == 0, "row passes");
  const int nchunks = H / 8, ll = tid & (LPR - 1), rsub = tid / LPR;
  const h8* wv = reinterpret_cast<const h8*>(ln.w);
  const h8* bv = reinterpret_cast<const h8*>(ln.b);
  // the rows of all passes and the parameters are requested together: one memory round trip
  h8 tw[CH], tb[CH], t[PASSES][CH];
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    int row = m0 + p * RPP + rsub;
    row = row < M ? row : M - 1;
    const h8* xr = reinterpret_cast<const h8*>(x + (size_t)row * H);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = ll + i * LPR;
      if (FULL || c < nchunks) t[p][i] = xr[c];
      else {
#pragma unroll
        for (int j = 0; j < 8; ++j) t[p][i][j] = (_Float16)0.f;
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
    float d[CH][8], rstd;
    layernorm_stats<CH, 8, LPR, FULL>(t[p], ll, nchunks, H, ln.eps, d, rstd);
#pragma unroll
    for (int i = 0; i < CH; ++i) {
      const int c = ll + i * LPR;
      if (FULL || c < nchunks) {
        h8 o;
#pragma unroll
        for (int j = 0; j < 8; ++j)
          o[j] = (_Float16)layernorm_apply(d[i][j], rstd, (float)tw[i][j], (float)tb[i][j]);
        *reinterpret_cast<h8*>(panel + (c >> 3) * (BM * 128) + r * 128 +
                               (((c & 7) ^ ((r >> 1) & 7)) << 4)) = o;
      }
    }
  }
}

// At most 4 chunks per lane: rows of up to 224 chunks (gemm_layernorm_supported), 64 lanes beyond 128.
template <int BM, int NT>
__device__ __forceinline__ void normalise_panel(const _Float16* x, int M, int H, int m0, const LnArgs& ln,
                                                char* panel, int tid) {
  const int need = (H / 8 + ln.lpr - 1) / ln.lpr;  // chunks per lane
#define GPTMI_LN_ROWS(L, FULL)                                                       \
  do {                                                                               \
    if (need <= 1) normalise_rows<BM, NT, L, 1, FULL>(x, M, H, m0, ln, panel, tid);      \
    else if (need <= 2) normalise_rows<BM, NT, L, 2, FULL>(x, M, H, m0, ln, panel, tid); \
    else if (need <= 3) normalise_rows<BM, NT, L, 3, FULL>(x, M, H, m0, ln, panel, tid); \
    else normalise_rows<BM, NT, L, 4, FULL>(x, M, H, m0, ln, panel, tid);                \
  } while (0)
  if (H / 8 == need * 32 && ln.lpr == 32) GPTMI_LN_ROWS(32, true);
  else if (ln.lpr == 32) GPTMI_LN_ROWS(32, false);
  else GPTMI_LN_ROWS(64, false);
#undef GPTMI_LN_ROWS
}

}  // namespace gptmi
