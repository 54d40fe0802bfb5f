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
