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
    for (long long units = 1; units < 40000; units *= 3) {
      const int h = fv3::fused_block_rows(rows, units, 768, 2.5);
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
