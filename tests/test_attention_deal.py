"""How the long-sequence attention kernels' work is dealt, on the host from the kernels' own header: every block of every
pair goes to one workgroup, and but for a 64th of them every workgroup has one, so that the 8 XCDs (workgroup id modulo
8) get the same number; all blocks of a pair go to one XCD but for up to 7 pairs; heavy blocks come first in a group."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpt_triton_amd", "csrc")
PROGRAM = r"""
#include <stdio.h>
#include <vector>
#include "attn_deal.h"
using namespace gptmi;
int main() {
  const int sizes[][2] = {{1, 1}, {1, 128}, {1, 2000}, {2, 64}, {7, 3}, {7, 200}, {8, 3}, {8, 128}, {9, 64}, {9, 128}, {15, 80},
                          {42, 6}, {42, 20}, {60, 8}, {65, 32}, {96, 8}, {127, 16}, {333, 3}, {343, 3}, {447, 5}, {503, 9}, {1600, 8},
                          {1601, 3}, {4095, 2}};
  for (const auto& s : sizes) {
    const int pairs = s[0], q_blocks = s[1];
    Deal deal;
    if (!deal_blocks(pairs, q_blocks, &deal)) return 1;
    if (deal.grid != (unsigned)(deal.pairs * q_blocks) || deal.pairs < pairs || (deal.pairs - pairs) * 64 > pairs) return printf("%d x %d: %u workgroups\n", pairs, q_blocks, deal.grid), 1;
    std::vector<int> seen(pairs * q_blocks), xcd(pairs, -1);
    int apart = 0, rises = 0, done = 0;
    for (int id = 0, last = q_blocks; id < (int)deal.grid; ++id) {
      const WorkItem w = work_item(id, deal.pairs, q_blocks, deal.group);
      if (w.bh >= pairs && w.bh < deal.pairs) continue;
      ++done;
      if (w.bh < 0 || w.bh >= pairs || w.qb < 0 || w.qb >= q_blocks || seen[w.bh * q_blocks + w.qb]++)
        return printf("%d x %d: workgroup %d\n", pairs, q_blocks, id), 1;
      if (xcd[w.bh] == -1) xcd[w.bh] = id % 8;
      if (xcd[w.bh] >= 0 && xcd[w.bh] != id % 8) xcd[w.bh] = -2, ++apart;
      rises += w.qb > last;
      last = w.qb;
    }
    if (done != pairs * q_blocks) return printf("%d x %d: %d done\n", pairs, q_blocks, done), 1;
    if (apart > pairs % 8) return printf("%d x %d: %d pairs apart\n", pairs, q_blocks, apart), 1;
    const int groups = deal.group ? (deal.pairs / 8 * 8 + deal.group - 1) / deal.group : 1;
    if (rises >= groups || (deal.grid < 1024 && rises)) return printf("%d x %d: %d rises\n", pairs, q_blocks, rises), 1;
  }
  Deal deal;
  return deal_blocks(1 << 24, 1, &deal) || deal_blocks(1ll << 40, 3, &deal);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_deal(tmp_path):
    source = tmp_path / "deal.cpp"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, "-o", tmp_path / "deal", source], check=True)
    done = subprocess.run([tmp_path / "deal"], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
