"""The per-device setup of the kernels' LDS limits (DeviceOnce), compiled for the host
with a stand-in for the current device: once for each device, from several threads,
and again after a failure."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")

SRC = r"""
#include "fv3_internal.h"
#include <atomic>
#include <cstdio>
#include <thread>
thread_local int current = 0;
extern "C" hipError_t hipGetDevice(int *d) {
  *d = current;
  return hipSuccess;
}
int main() {
  fv3::DeviceOnce once;
  std::atomic<int> runs[2] = {};
  std::vector<std::thread> t;
  for (int n = 0; n < 16; n++)
    t.emplace_back([&, n] {
      current = n & 1;
      for (int m = 0; m < 100; m++) once([&] { runs[current]++; return hipSuccess; });
    });
  for (auto &x : t) x.join();
  if (runs[0] != 1 || runs[1] != 1) return 1;
  fv3::DeviceOnce fails;
  int tries = 0;
  for (int m = 0; m < 3; m++)
    if (fails([&] { return ++tries < 2 ? hipErrorInvalidValue : hipSuccess; }) != (m == 0 ? hipErrorInvalidValue : hipSuccess))
      return 2;
  if (tries != 2) return 3;
  std::puts("ok");
  return 0;
}
"""


def test_once_for_each_device(tmp_path):
    if not os.path.exists(HIPCC):
        pytest.skip("hipcc not found")
    src = tmp_path / "once.cpp"
    src.write_text(SRC)
    exe = tmp_path / "once"
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-O1", "-std=c++17", "-w", "-x", "hip", str(src), "-I",
                    os.path.join(ROOT, "fv3atm_amd", "csrc"), "-lpthread", "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and "ok" in r.stdout, r.returncode
