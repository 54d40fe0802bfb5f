// What the attention launches of layers in one call request of the weights behind them.  Nothing but arithmetic, for
// the host's compiler too.
#pragma once
#include <stddef.h>
#include <stdint.h>

#ifndef GPTMI_HOST_DEVICE
#ifdef __HIPCC__
#define GPTMI_HOST_DEVICE __attribute__((host, device, always_inline))
#else
#define GPTMI_HOST_DEVICE
#endif
#endif

namespace gptmi {

// What the launches behind this one will read (weights): an attention launch has further workgroups request it from
// HBM into the memory-side cache, on the CUs that it leaves idle.
struct Prefetch {
  const void* p[4] = {};
  size_t bytes[4] = {};
  bool may_be_cached = false;  // the memory-side cache may hold it from the model's last forward
  bool empty() const { return bytes[0] == 0; }
};

// The same as a kernel takes it, in lines of 128 bytes.
struct PrefetchArgs {
  const void* p[4];
  unsigned lines[4];  // multiples of 8, for both sides of a matrix are multiples of 64
};
inline PrefetchArgs prefetch_args(const Prefetch* ahead) {
  PrefetchArgs a = {};
  for (int k = 0; ahead != nullptr && k < 4; ++k) a.p[k] = ahead->p[k], a.lines[k] = (unsigned)(ahead->bytes[k] / 128);
  return a;
}
// What goes through one of the 8 XCDs: an eighth of each matrix, in order (the part that the products of few rows read
// there, which then lies in its L2 as well), one matrix behind the other.
class AheadLines {
 public:
  GPTMI_HOST_DEVICE AheadLines(const PrefetchArgs& pf, unsigned xcd) {
    unsigned all = 0;
#pragma GCC unroll 4
    for (int k = 0; k < 4; ++k) {
      const unsigned eighth = pf.lines[k] >> 3;
      base_[k] = (uintptr_t)pf.p[k] + ((uintptr_t)xcd * eighth - all) * 128;
      all += eighth;
      end_[k] = all;
    }
  }
  GPTMI_HOST_DEVICE unsigned all() const { return end_[3]; }
  GPTMI_HOST_DEVICE uintptr_t at(unsigned n) const {  // address of the n-th of them
    return (n < end_[0] ? base_[0] : n < end_[1] ? base_[1] : n < end_[2] ? base_[2] : base_[3]) + (uintptr_t)n * 128;
  }

 private:
  uintptr_t base_[4];
  unsigned end_[4];
};

// Workgroups for it behind the `workers` of the front kernel (LayerNorm, product and attention of short sequences), which
// pull their weights through CUs of their own, one workgroup each: requests from all idle CUs at once stand in their way,
// from 64 they do not, and from few what they ask for is late.  With fewer than 32 CUs idle they wait for the workers to
// end, and more of them are through sooner.  Forwards of 124M that the GPU sets the pace of, all idle CUs (beyond 192
// workers 128) / 128 / 64 / 32, us: 1 x 8 tokens 276 / 271 / 264 / 263, 1 x 24 with logits 301 / 296 / 289 / 288, weights from HBM 1 x
// 24 294 / 288 / 285 / 286, 8 x 24 360 / 358 / 354 / 357, 16 x 32 412 / 413 / 412 / 414, 18 x 32 434 / 434 / 427 / 421, 19 x 32
// 456 / 455 / 464 / 498, 21 x 32 505 / 506 / 524 / 557.
inline int front_ahead_workgroups(const Prefetch* ahead, int64_t workers, int cus) {
  return ahead == nullptr || ahead->empty() ? 0 : workers <= cus - 32 ? 64 : 128;
}

// Sizes that are the same for all layers of a call; rows: of a key, lasting: see weights_ahead.
struct AheadPlan {
  size_t square, wide, most;  // bytes of W_proj, W1 or W2; of all that is requested behind W2
  bool any, may_be_cached;
};
// The MLP's second product first, which has the longest columns, then the next layer's first product, then what follows at
// once; half a matrix saves nothing, and what the launch has to wait for costs what it saves.  How much is a fit to
// what was measured: launches of as many workgroups as CUs and those of the front kernel (lasting) take some 15 MB and
// 40 KB more for each key row, launches of few pairs 120 KB a key row, and the second product alone is worth a wait of
// its 14 MB or less.  Forwards that find their weights in HBM (four models in turn; wider ones always do), us,
// nothing / the second product alone / this: 124M 1 x 24 tokens 342 / 335 / 303, 2 x 64 370 / 357 / 356 (15 MB: 368),
// 7 x 211 751 / 724 / 674, 1 x 800 713 / 695 / 651; 100 x 40 1274 / - / 1164 (120 KB a row: 1217); 1024 wide 1 x 41 707 /
// 698 / 697 (15 MB: 715), 4 x 160 1390 / - / 1237, 2 x 200 1168 / 1148 / 1115; 1280 wide 2 x 60 1641 / 1545, 2 x 200
// 2376 / 2320 / 2239; 1600 wide 1 x 41 1925 / 1959 / 1925, 1 x 150 2616 / 2478 / 2478, 1 x 300 3349 / 3174 / 3100, 1 x 500
// 4287 / 3851 / 3851 (60 MB: 3972).
// One 124M model over and over, whose 170 MB the memory-side cache holds, nothing / this: 1 x 24 298 / 297, 2 x 64 344 /
// 343, 1 x 300 434 / 428, 7 x 211 669 / 667, 16 x 300 1302 / 1253, 21 x 64 610 / 614, 100 x 40 1192 / 1203, 32 x 300
// 2282 / 2140.  Widths between those of the fit, 8 shapes each: 640 (12 layers) 1 x 24 278 / 279, 7 x 211 559 / 554, 100 x 40
// 974 / 1001, 896 (24) 797 / 795 to 1606 / 1526, 1152 2187 / 2068, 1408 1515 / 1394, 1792 (12) 1016 / 917, others equal.
inline AheadPlan plan_ahead(int64_t rows, bool lasting, int64_t h, int64_t inner) {
  AheadPlan plan;
  plan.square = (size_t)(h * h * 2);
  plan.wide = (size_t)(h * inner * 2);
  const size_t alone = 15000000 + 40000 * (size_t)rows;
  const size_t by_row = 120000 * (size_t)rows < 40000000 ? 120000 * (size_t)rows : 40000000;
  plan.most = lasting && alone > by_row ? alone : by_row;
  plan.any = plan.wide <= alone;
  // 12 layers, the fewest of the GPT-2 sizes, in 256 MB
  plan.may_be_cached = 12 * (4 * plan.square + 2 * plan.wide) <= (size_t)256 << 20;
  return plan;
}

// layer: its 12 pointers as gptmi_blocks lists them, those of the next one behind them unless it is the last.
inline Prefetch weights_ahead(const void* const* layer, bool last, const AheadPlan& plan) {
  Prefetch ahead;
  if (!plan.any) return ahead;
  const struct {
    const void* p;
    size_t bytes;
  } wanted[4] = {{layer[10], plan.wide}, {last ? nullptr : layer[12 + 2], 3 * plan.square}, {layer[8], plan.wide},
                 {layer[4], plan.square}};
  ahead.may_be_cached = plan.may_be_cached;
  size_t sum = 0;
  for (int k = 0; k < 4; ++k) {
    if (wanted[k].p == nullptr) continue;
    sum += wanted[k].bytes;
    if (k > 0 && sum > plan.most) break;
    ahead.p[k] = wanted[k].p, ahead.bytes[k] = wanted[k].bytes;
  }
  return ahead;
}

}  // namespace gptmi
