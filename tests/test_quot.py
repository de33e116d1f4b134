"""The remap's division by tabulated divisors (quot.h), compiled for the host: bit
for bit the division, for float, double and both components of (value, tangent)
pairs, over random operands of the elimination's and the layer sums' ranges; the
tangent beside a value that is not finite is a NaN, as the division's."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")

SRC = r"""
#include "quot.h"
#include <cmath>
#include <cstdio>
#include <cstring>
#include <random>
using namespace fv3;
template <typename R>
bool same(R a, R b) { return std::memcmp(&a, &b, sizeof(R)) == 0 || (a == R(0) && b == R(0)); }
template <typename R>
int check(std::mt19937_64 &g) {
  std::uniform_real_distribution<double> u(-1.0, 1.0), lb(-3.0, 12.0), la(-12.0, 9.0);
  for (int n = 0; n < 4000000; n++) {
    const R b = R(std::exp2(lb(g))), a = R(u(g) * std::exp2(la(g))), y = R(1) / b;
    if (!same(quot(a, b, y), R(a / b))) return 1;
  }
  return 0;
}
int main() {
  std::mt19937_64 g(7);
  if (check<double>(g)) return 1;
  if (check<float>(g)) return 2;
  std::uniform_real_distribution<double> u(-1.0, 1.0), lb(-3.0, 12.0);
  for (int n = 0; n < 4000000; n++) {
    const double b = std::exp2(lb(g)), y = 1.0 / b;
    Dual<1> a(u(g));
    a.d[0] = u(g);
    const Dual<1> q = quot(a, b, y), r = a / Dual<1>(b);
    if (!same(q.v, r.v) || !same(q.d[0], r.d[0])) return 3;
  }
  // a tangent beside a value that is not finite, or over a divisor that is not one
  const double inf = INFINITY, odd[] = {inf, -inf, NAN};
  for (double v : odd) {
    Dual<1> a(v);
    a.d[0] = 0.5;
    if (!std::isnan(quot(a, 3.0, 1.0 / 3.0).d[0]) || !std::isnan((a / Dual<1>(3.0)).d[0])) return 4;
  }
  Dual<1> a(1.0);
  a.d[0] = 0.5;
  if (!std::isnan(quot(a, NAN, NAN).d[0]) || !std::isnan((a / Dual<1>(NAN)).d[0])) return 5;
  std::puts("ok");
  return 0;
}
"""


def test_equals_division(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    src = tmp_path / "quot.cpp"
    src.write_text(SRC)
    exe = tmp_path / "quot"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O2", "-std=c++17", "-ffp-contract=off", "-w", "-x", "hip", str(src),
                    "-I", os.path.join(ROOT, "fv3atm_amd", "csrc"), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and "ok" in r.stdout, r.returncode
