"""Which GEMV kernel the plan (hcblas_amd/csrc/gemv_plan.hpp, host code) takes for
sizes at which one of them measured clearly ahead, at 256 CUs: short row bands whose
lanes would idle, narrow matrices read along their rows, and those that a second
launch would slow down."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PROBE = r'''
#include <cstdio>
#include <cstdlib>
#include "gemv_plan.hpp"
int main(int argc, char **argv) {
  const char *names[] = {"bandn", "panel", "band", "band", "column"};
  for (int i = 1; i + 4 < argc; i += 5) {
    const int es = atoi(argv[i + 3]);
    const long long R = atoll(argv[i + 1]);
    const hcb::GemvPlan p =
        hcb::plan_gemv(256, atoi(argv[i]) != 0, R, atoll(argv[i + 2]), R >= 16 / es,
                       16 / es, es, atoll(argv[i + 4]));
    std::printf("%s %d %d\n", names[(int)p.kernel], p.waves, p.splits > 1);
  }
  return 0;
}
'''
# row-contiguous case, R, Cc, element bytes, batch: kernel, waves, split
RULES = [
    # two steps with half their lanes idle (4.9 us, bands 6.5) and all at work
    ((0, 1052, 4224, 4, 1), ("column", 4, 0)), ((0, 2011, 1773, 4, 1), ("band", 4, 0)),
    ((0, 384, 2528, 8, 1), ("column", 4, 0)), ((0, 1536, 4195, 4, 1), ("column", 4, 0)),
    # a large matrix of one full step (61 us, column kernel 77)
    ((0, 1024, 100000, 4, 1), ("band", 4, 0)),
    # three steps in one band (5.5 us, 6.8 in two), many steps in several
    ((0, 2700, 87, 4, 1), ("band", 4, 0)), ((0, 20011, 64, 4, 1), ("band", 4, 1)),
    # up to 128 columns (3.6 us, sixteen waves 4.0), up to 512, and more
    ((1, 3904, 96, 4, 1), ("panel", 4, 0)), ((1, 168, 100, 8, 1), ("panel", 4, 0)),
    ((1, 3904, 300, 4, 1), ("panel", 16, 0)),
    ((1, 1024, 225, 8, 43), ("panel", 4, 0)),  # 13.7 us, in bands 20.1
    ((1, 3904, 600, 4, 1), ("bandn", 4, 1)), ((1, 24, 4276, 4, 1), ("panel", 4, 1)),
]


def test_measured_choices(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(PROBE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "hcblas_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe)] + [str(v) for r, _ in RULES for v in r],
                         capture_output=True, text=True, check=True).stdout
    got = [(k, int(w), int(s)) for k, w, s in
           (line.split() for line in out.strip().split("\n"))]
    assert got == [w for _, w in RULES], [
        (r, g, w) for (r, w), g in zip(RULES, got) if g != w]
