// How the (batch, head) pairs and query blocks of the long-sequence attention kernels (flash_attn.hip) are dealt to
// workgroups.  Nothing but arithmetic, for the host's compiler too.
#pragma once
#include <stdint.h>

#ifndef GPTMI_HOST_DEVICE
#ifdef __HIPCC__
#define GPTMI_HOST_DEVICE __attribute__((host, device, always_inline))
#else
#define GPTMI_HOST_DEVICE
#endif
#endif

namespace gptmi {

// Which (batch, head) pair and which query block (of q_blocks) a workgroup works on.  Workgroup ids are dealt
// round-robin over the 8 XCDs, so ids equal modulo 8 share one: all blocks of a pair go to the same, whose L2 then
// holds the K and V that they share.  Up to 7 pairs, those beyond a multiple of 8, are tied to none, so that every
// XCD gets the same number of blocks (`pairs` is Deal's, which may count some that are none).  Pairs are taken in groups of `group`, a multiple of
// 8 (0: fewer than 8 pairs), of each group the heaviest (latest) block of every pair first, then all next ones; the
// untied are part of the first group, for a heavy block that starts last is waited for.  Pairs tied without exception
// / so, us: d = 64 1 pair of 16384 rows 331 / 225, 9 of 8192 165 / 131, 42 of 4096 174 / 144, 257 of 512 23.6 / 21.3;
// d = 256 1 of 16384 1597 / 747, 9 of 8192 822 / 522, 257 of 512 115 / 90.
struct WorkItem {
  int bh, qb;  // bh: less than Deal's pairs
};
GPTMI_HOST_DEVICE inline WorkItem work_item(int workgroup, int pairs, int q_blocks, int group) {
  const int front = group + (pairs & 7), behind = workgroup - front * q_blocks;
  int base = 0, size = front, at = workgroup;
  if (behind >= 0) {
    const int g = behind / (group * q_blocks);
    base = front + g * group;
    size = group < pairs - base ? group : pairs - base;
    at = behind - g * group * q_blocks;
  }
  const int late = at / size, s = at - late * size;
  // 8 ids in a row are one of each XCD
  return {base + (s < (size & ~7) ? (s & ~7) + (workgroup & 7) : s), q_blocks - 1 - late};
}

// Groups of some 256 workgroups, half of what the chip holds: their K and V stay in the XCDs' 4 MB L2s until the last
// block has read them (all pairs' heaviest blocks first, every block fetches them anew; 64 x 25 pairs of 1024 rows:
// 445 us, groups of 8, 16, 32, 64, 128 pairs 417, 398, 376, 383, 394; 512 x 6 of 300 rows, d = 128: 308, 229, 231, 226,
// 224, 233).  Below two rounds of workgroups the order decides when the last one ends, and all heaviest go first
// (8 x 12 pairs of 1024 rows 25.6 us, groups of 32 26.8).
// Of more than 64 pairs for each that is missing to a multiple of 8, the last are tied too, for what that leaves empty is
// less than what untied pairs fetch anew (127 pairs of 2048 rows, d = 256: 553 us, 510 tied; d = 64 114, 112).
struct Deal {
  unsigned grid;
  int pairs, group;
};
// false: more workgroups than a grid takes (memory holds at most some 5 million blocks' q, k, v and output)
inline bool deal_blocks(int64_t pairs, int q_blocks, Deal* deal) {
  const int64_t missing = -pairs & 7;
  if (missing * 64 <= pairs) pairs += missing;
  const int64_t all = pairs * q_blocks, tied = pairs & ~(int64_t)7, some = 8 * ((32 + q_blocks - 1) / q_blocks);
  if (all >= 1 << 24) return false;
  deal->group = (int)(all < 1024 || tied < some ? tied : some);
  deal->grid = (unsigned)all;
  deal->pairs = (int)pairs;
  return true;
}

}  // namespace gptmi
