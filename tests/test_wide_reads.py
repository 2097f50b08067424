"""The reads of the GEMM with dequantised operands stay inside the weight and its staged
metadata for every column tile, the ragged last one included: the kernel's own offset functions
(csrc/mtl_w4wide_reads.h) in a host program that walks them (CPU)."""
import os
import shutil
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                    "moss-tts-lite_amd", "csrc")

# Every wave of every 256-column tile, its 4 strips, first and last block of each half of K (the
# offsets grow with the block), each group size.  Sizes as WideLayout and the strip layout give them.
PROGRAM = r"""
#include <cstdio>
#include <initializer_list>
#include "mtl_w4wide_reads.h"
using namespace mtl;
int main() {
  long walked = 0;
  for (int N = 16; N <= 2064; N += 16)
    for (int K : {256, 512, 768, 4096, 16640})
      for (int g : {32, 64, 128, 256}) {
        const int kb = K / 128, mb = g >= 128 ? 1 : 128 / g, krec = K / (g > 128 ? 256 : 128);
        const int zc = (K / g + 31) / 32;
        const long wbytes = (long)N * K / 2, sbytes = (long)K / g * N * 2, zbytes = N / 16l * zc * 1024;
        for (int strip = 0; strip < (N + 255) / 256 * 16; ++strip) {
          const int s = wide_strip(strip, N / 16);
          if (strip < N / 16 && s != strip) return 2;
          for (int b : {0, kb / 2 - 1, kb / 2, kb - 1}) {
            const long w = wide_weight_at(s, kb, b), m = wide_scale_at(s, krec, kb, b, mb);
            if (w < 0 || w + 1024 > wbytes || m < 0 || m + 32 * mb > sbytes) {
              std::printf("N=%d K=%d g=%d strip %d block %d\n", N, K, g, strip, b);
              return 1;
            }
          }
          const long z = wide_zero_at(s, zc, zc - 1);
          if (z < 0 || z + 1024 > zbytes) { std::printf("zeros N=%d K=%d g=%d\n", N, K, g); return 1; }
          ++walked;
        }
      }
  std::printf("walked %ld\n", walked);
  return 0;
}
"""


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
def test_wide_reads_stay_inside(tmp_path):
    src, exe = tmp_path / "walk.cpp", tmp_path / "walk"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-O2", "-std=c++17", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout.startswith("walked"), r.stdout
