"""The fused transport's block numbering and row-block rule, compiled from the
header for the host: every (block, round) pair is reached once, the rounds of a
block keep its number modulo 8, and the rows per block stay in their range."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")

SRC = r"""
#include "fused_tp.h"
#include <cstdio>
#include <vector>
int main() {
  for (int nb = 1; nb < 70; nb++)
    for (int rounds = 1; rounds < 17; rounds++) {
      std::vector<int> seen(nb * rounds, 0);
      for (int x = 0; x < nb * rounds; x++) {
        int b = x, r = 0;
        fv3::fused_block_round(x, nb, rounds, b, r);
        if (b < 0 || b >= nb || r < 0 || r >= rounds || seen[r * nb + b]++) return 1;
        if (b < (nb & ~7) && (b & 7) != (x & 7)) return 2;
      }
    }
  for (int rows = 1; rows < 1600; rows = rows < 40 ? rows + 1 : rows * 5 / 4)
    for (long long units = 1; units < 40000; units *= 3)
      for (int slots : {512, 768})        // FP64, FP32
        for (double warm : {4.0, 6.0}) {  // with interior strips, without
          const int h = fv3::fused_block_rows(rows, units, slots, warm);
          if (h < 12 || h > 60 || h % 6) return 3;
        }
  std::puts("ok");
  return 0;
}
"""


def test_blocks_and_rows(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    src = tmp_path / "blocks.cpp"
    src.write_text(SRC)
    exe = tmp_path / "blocks"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-w", "-x", "hip", str(src), "-I",
                    os.path.join(ROOT, "fv3atm_amd", "csrc"), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and "ok" in r.stdout, r.returncode


# Every strip and row block of a tile with three halo cells: one that holds a
# corner cell (corner_src, the exact rule) has to be marked as reading corners.
# Rows per block as the transport derives them and every other value up to 60.
CORNERS = r"""
#include "fused_tp.h"
#include <algorithm>
#include <cstdio>
using namespace fv3;
int main() {
  for (int n = 8; n <= 260; n++)
    for (int H0 = -5; H0 <= 60; H0++) {
      if (H0 == 0) continue;
      // H0 < 0: the rule, at -H0 levels, FP32 or FP64, one or a few tracers
      const int ns = (n + FT_BX - 1) / FT_BX;
      const int H = std::min(n, H0 > 0 ? H0 : fused_block_rows(n, (long long)ns * -H0 * 16, H0 & 1 ? 768 : 512, 2.0 * NG));
      for (int s = 0; s < ns; s++)
        for (int b = 0; b * H < n; b++) {
          const int i0 = 1 + s * FT_BX, j0 = 1 + b * H, h = std::min(H, n + 1 - j0);
          bool holds = false;
          for (int l = 0; l < FT_LANES && !holds; l++)
            for (int j = j0 - NG; j <= j0 + h - 1 + NG && !holds; j++) {
              int si, sj;
              const int i = std::min(i0 - NG + l, n + NG);
              holds = corner_src(i, j, n + 1, n + 1, 1, 15u, si, sj);
            }
          if (holds && !fused_reads_corners(i0, j0, h, 1, n, 1, n)) {
            std::printf("n %d rows %d strip %d block %d\n", n, H, s, b);
            return 1;
          }
        }
    }
  std::puts("ok");
  return 0;
}
"""


def test_corner_blocks(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    src = tmp_path / "corners.cpp"
    src.write_text(CORNERS)
    exe = tmp_path / "corners"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-w", "-x", "hip", str(src), "-I",
                    os.path.join(ROOT, "fv3atm_amd", "csrc"), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and "ok" in r.stdout, r.stdout
