"""The launch shape of strided level-1 updates (hcblas_amd/csrc/level1_plan.hpp,
host code): every element is covered, and short vectors of a large batch share
workgroups instead of taking a nearly empty one each."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r'''
#include <cstdio>
#include "level1_plan.hpp"
int main() {
  const long long T = hcb::kLevel1Threads;
  for (long long n : {1ll, 3ll, 16ll, 100ll, 191ll, 192ll, 255ll, 256ll, 257ll,
                      383ll, 384ll, 520ll, 1000ll, 5000ll, 1ll << 20, 1ll << 31})
    for (long long batch : {1ll, 2ll, 70ll, 10000ll, 65535ll, 65536ll, 1000000ll}) {
      const hcb::StridedGrid g = hcb::plan_strided(n, batch);
      // lanes launched in one pass, and the elements they have among them
      const long long lanes = g.x * T * g.y;
      const long long rows = g.y < batch ? g.y : batch;
      const long long used = g.rows ? (n < g.x * T ? n : g.x * T) * rows
                                    : (n * batch < lanes ? n * batch : lanes);
      const bool ok = g.x >= 1 && g.y >= 1 && g.y <= 65535 &&
                      (g.rows || g.y == 1) &&
                      (batch == 1 || lanes <= T || 4 * used >= 3 * lanes ||
                       (!g.rows && lanes - used < T));
      if (!ok) {
        std::printf("%lld x %lld: %d %d %d\n", n, batch, (int)g.rows, g.x, g.y);
        return 1;
      }
    }
  std::printf("ok\n");
  return 0;
}
'''


def test_strided_grid(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(PROBE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "hcblas_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0 and p.stdout == "ok\n", p.stdout + p.stderr
