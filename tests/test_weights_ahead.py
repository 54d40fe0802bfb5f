"""What the layers of one call request ahead of the weights behind them, on the host from the library's own header: whole
matrices at their own addresses, the next layer's only where there is one, and nothing where nothing is chosen."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "gpt_triton_amd", "csrc")
PROGRAM = r"""
#include <stdio.h>
#include <initializer_list>
#include "weights_ahead.h"
using namespace gptmi;
int main() {
  static char memory[24];
  const void* params[24];
  for (int i = 0; i < 24; ++i) params[i] = memory + i;
  int some = 0, none = 0, next = 0;
  for (int64_t h = 64; h <= 8192; h += 64)
    for (int64_t inner : {h, 4 * h, 4 * h + 64})
      for (int64_t L : {1, 24, 64, 137, 138, 300, 1024, 5000})
        for (int flags = 0; flags < 4; ++flags) {
          const bool lasting = flags & 1, last = flags & 2;
          const Prefetch a = weights_ahead(params, last, plan_ahead(L, lasting, h, inner));
          size_t sum = 0;
          for (int k = 0; k < 4; ++k) {
            sum += a.bytes[k];
            if ((a.p[k] == nullptr) != (a.bytes[k] == 0)) return printf("bytes without a place\n"), 1;
            if (a.p[k] == nullptr) continue;
            const long j = (const char*)a.p[k] - memory;
            const size_t whole = j == 10 || j == 8 ? 2 * h * inner : j == 4 ? 2 * h * h : j == 14 && !last ? 6 * h * h : 0;
            if (a.bytes[k] != whole) return printf("%zu bytes of matrix %ld, width %d\n", a.bytes[k], j, (int)h), 1;
            next += j == 14;
          }
          if (a.empty() != (sum == 0)) return printf("not the second product first\n"), 1;
          (sum ? some : none) += 1;
          if (sum > 2u * h * inner && sum > 15000000 + 40000u * L && sum > 40000000) return printf("%zu bytes\n", sum), 1;
        }
  return !(some && none && next);
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_whole_matrices(tmp_path):
    source = tmp_path / "ahead.cpp"
    source.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-Wno-sign-compare", "-I", CSRC, "-o", tmp_path / "ahead",
                    source], check=True)
    done = subprocess.run([tmp_path / "ahead"], capture_output=True, text=True)
    assert done.returncode == 0, done.stdout
