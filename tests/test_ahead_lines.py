"""Which lines of memory the workgroups that request weights ahead read, on the host from the library's own header: over the
8 XCDs every line of every matrix once, and none that is not of a matrix."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpt_triton_amd", "csrc")
PROGRAM = r"""
#include <stdio.h>
#include <set>
#include "weights_ahead.h"
using namespace gptmi;
int main() {
  const size_t sizes[] = {0, 64 * 64 * 2, 3 * 64 * 64 * 2, 64 * 192 * 2, 128 * 448 * 2};
  for (int c = 0; c < 5 * 5 * 5 * 5; ++c) {
    Prefetch f;
    std::set<uintptr_t> left;
    for (int k = 0, r = c; k < 4; ++k, r /= 5) {
      f.bytes[k] = sizes[r % 5];
      f.p[k] = f.bytes[k] ? (const void*)(uintptr_t)((4 - k) * (size_t)1000000 + 256) : nullptr;  // in falling order
      for (size_t i = 0; i < f.bytes[k]; i += 128) left.insert((uintptr_t)f.p[k] + i);
    }
    const PrefetchArgs args = prefetch_args(&f);
    for (unsigned xcd = 0; xcd < 8; ++xcd) {
      const AheadLines lines(args, xcd);
      for (unsigned n = 0; n < lines.all(); ++n)
        if (left.erase(lines.at(n)) != 1) return printf("case %d, XCD %u, line %u\n", c, xcd, n), 1;
    }
    if (!left.empty()) return printf("case %d: %zu lines left\n", c, left.size()), 1;
  }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_every_line_once(tmp_path):
    source = tmp_path / "lines.cpp"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, "-o", tmp_path / "lines", source], check=True)
    done = subprocess.run([tmp_path / "lines"], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout


WORKGROUPS = r"""
#include <stdio.h>
#include "weights_ahead.h"
using namespace gptmi;
int main() {
  Prefetch none, some;
  some.p[0] = "", some.bytes[0] = 1 << 20;
  for (int workers = 1; workers <= 256; ++workers) {
    if (front_ahead_workgroups(nullptr, workers, 256) != 0 || front_ahead_workgroups(&none, workers, 256) != 0) return 1;
    const int n = front_ahead_workgroups(&some, workers, 256);
    if (n < 8 || n % 8 != 0) return printf("%d workgroups: not the same number on every XCD\n", n), 1;
    if (workers + n <= 256 ? n > 64 : workers <= 192 || workers + n < 256) return printf("%d beside %d\n", n, workers), 1;
  }
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_few_workgroups_beside_the_front_kernels(tmp_path):
    """64 beside its workers and no more: with 244 of them 1 x 24 tokens with logits took 301 us in place of 289."""
    source = tmp_path / "workgroups.cpp"
    source.write_text(WORKGROUPS)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I", CSRC, "-o", tmp_path / "workgroups", source], check=True)
    done = subprocess.run([tmp_path / "workgroups"], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
    with open(os.path.join(CSRC, "attn_front.hip")) as f:
        assert "workers + front_ahead_workgroups(ahead, workers, cus)" in f.read()
