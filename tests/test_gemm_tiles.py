"""The GEMM's tile choice (hcblas_amd/csrc/gemm_tiles.hpp, host code) on the CPU, at
256 CUs: the sizes of the GPU tests run on the tiles that they are there for, short
K loops on tiles that measured fastest, and K slices of a split product cover
K."""
import os
import shutil
import subprocess

import pytest

from gemm_tile_cases import CASES, FORMS

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r'''
#include <cstdio>
#include <cstdlib>
#include "gemm_tiles.hpp"
using namespace hcb;
// type (s d h) M N K batch r-contiguous operands: tile
int main(int argc, char **argv) {
  for (int i = 1; i + 5 < argc; i += 6) {
    const long long m = atoll(argv[i + 1]), n = atoll(argv[i + 2]),
                    k = atoll(argv[i + 3]), b = atoll(argv[i + 4]);
    const int rc = atoi(argv[i + 5]);
    const MacroTile &t =
        argv[i][0] == 's'   ? pick_tile<Elem::F32>(m, n, k, b, 256, rc)
        : argv[i][0] == 'd' ? pick_tile<Elem::F64>(m, n, k, b, 256, rc)
                            : pick_tile<Elem::F16>(m, n, k, b, 256, rc);
    std::printf("%dx%d\n", t.bm, t.bn);
  }
  if (argc > 1) return 0;
  for (int m : {1, 31, 33, 128, 515, 1000, 4096})
    for (int n : {1, 64, 513, 2000})
      for (int k : {1, 512, 2047, 2048, 2049, 2305, 3001, 8192, 36864, 1 << 20})
        for (int bk : {64, 128}) {
          const SplitK s = splitk_plan(m, n, k, 256, bk, 32);
          const long long last = k - (long long)(s.splits - 1) * s.ks;
          if (s.splits < 1 || last < 1 || last > s.ks || s.splits > 8 ||
              (s.splits > 1 && (k < 2048 || s.ks % 32 || s.ks < 256))) {
            std::printf("%d %d %d: %d x %d\n", m, n, k, s.splits, s.ks);
            return 1;
          }
        }
  // rows and K against a 16-byte vector, in each orientation
  if (is_narrow(4, 4, 4, true, true, 1, 4) || !is_narrow(4, 4, 3, true, false, 1, 4) ||
      is_narrow(4, 4, 3, false, false, 1, 4) ||
      !is_narrow(3, 4, 9, false, true, 1, 4) ||
      !is_narrow(9, 7, 9, true, false, 1, 2) || is_narrow(4, 1, 4, true, true, 2, 4) ||
      !is_narrow(2, 9, 8, false, true, 2, 4) || is_narrow(2, 1, 2, false, false, 2, 8))
    return 1;
  std::printf("ok\n");
  return 0;
}
'''

# Short K loops (K <= 50), and products for which a rate has to win over a lead:
# type, M, N, K, batch, r-contiguous operands, tiles within 4% of the fastest.
MEASURED = [("d", 586, 46, 16, 7, 0, "32x32"), ("d", 421, 2944, 26, 1, 1, "64x64"),
            ("d", 5516, 1312, 29, 1, 1, "64x64"), ("d", 4096, 4096, 4096, 1, 1, "256x128"),
            ("d", 827, 5055, 167, 1, 1, "64x64"), ("s", 1584, 2240, 32, 1, 0, "64x64"),
            ("s", 203, 698, 84, 120, 1, "64x64"), ("s", 255, 257, 517, 8, 1, "32x32"),
            ("s", 5632, 2816, 448, 1, 0, "256x256"), ("s", 4096, 4096, 4096, 1, 1, "256x256"),
            ("s", 260, 130, 80, 120, 0, "64x64"), ("h", 7520, 6272, 16, 1, 1, "128x128"),
            ("h", 8192, 8192, 8192, 1, 1, "256x256")]


@pytest.fixture(scope="module")
def probe(tmp_path_factory):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    d = tmp_path_factory.mktemp("tiles")
    src, exe = d / "probe.cpp", d / "probe"
    src.write_text(PROBE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "hcblas_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)

    def run(rows=()):
        p = subprocess.run([str(exe)] + [str(v) for r in rows for v in r],
                           capture_output=True, text=True)
        assert p.returncode == 0, p.stdout
        return p.stdout.split()
    return run


def test_sizes_of_the_gpu_tests(probe):
    rows, want = [], []
    for p, m, n, k, tile in CASES:
        for ta, tb in FORMS:
            cx = p in "cz"
            # (column-major: op(A) = A and op(B) = B^T have contiguous rows; a
            # complex product's real form is read k-contiguous)
            rc = 0 if cx else (ta == 0) + (tb == 1)
            rows.append(({"c": "s", "z": "d", "b": "h"}.get(p, p), m * (1 + cx), n,
                         k * (1 + cx), 1, rc))
            want.append(tile if isinstance(tile, str) else tile[ta, tb])
    got = probe(rows)
    assert got == want, [(r, g, w) for r, g, w in zip(rows, got, want) if g != w]


def test_measured_choices(probe):
    got = probe([r[:6] for r in MEASURED])
    assert got == [r[6] for r in MEASURED]


def test_split_plan_and_narrow_operands(probe):
    assert probe() == ["ok"]
