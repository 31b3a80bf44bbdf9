"""bvllm_fast_div.h: division by multiplication, exact over its whole range (compiled for the host)."""

import os
import subprocess
from pathlib import Path

CSRC = Path(__file__).resolve().parents[1] / "baby-vllm_amd" / "csrc"

SOURCE = r"""
#include <cstdio>
#include <random>
#include "bvllm_fast_div.h"
int main() {
  std::mt19937 r(1);
  const int32_t top = 0x7fffffff;
  for (int64_t i = 0; i < 60000; ++i) {
    // 1 .. 4096, powers of two and their neighbours, then any divisor
    int64_t d = i < 4096 ? i + 1 : i < 4096 + 93 ? ((int64_t)1 << ((i - 4096) / 3)) + (i - 4096) % 3 - 1 : 1 + r() % top;
    if (d < 1 || d > top) continue;
    const bvllm::FastDiv by = bvllm::fast_div((int32_t)d);
    for (int k = 0; k < 60; ++k) {
      const int64_t q = r() % (top / d + 1);
      const int64_t around[] = {0, 1, d - 1, d, top, top - 1, q * d - 1, q * d, q * d + d - 1, (int64_t)(r() & top)};
      for (int64_t n : around)
        if (n >= 0 && n <= top && by((int32_t)n) != n / d) return std::printf("%ld / %ld = %d\n", (long)n, (long)d, by((int32_t)n)), 1;
    }
  }
  return 0;
}
"""


def test_quotients_are_exact(tmp_path):
    src = tmp_path / "t.cpp"
    src.write_text(SOURCE)
    exe = tmp_path / "t"
    subprocess.run([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-I", str(CSRC), str(src), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True)
    assert out.returncode == 0, out.stdout
