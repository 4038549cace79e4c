"""The blocks that hold the partial sums of split reductions
(hcblas_amd/csrc/partial_blocks.hpp, host code) on the CPU, over an allocator
that records what is live: no block serves two queues, a capture and an eager
call, or two captures; growing frees nothing; everything is bounded and freed at
the end. The GEMV plan without partials is checked beside it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROBE = r'''
#include <cstdio>
#include <cstdlib>
#include <map>
#include <set>
#include "gemv_plan.hpp"
#include "partial_blocks.hpp"
using hcb::PartialBlocks;
static std::map<void *, size_t> live;
static int frees = 0;
static bool dry = false;
static void *take(size_t n) {
  if (dry) return nullptr;
  void *p = std::malloc(1);
  live[p] = n;
  return p;
}
static void give(void *p) {
  if (!live.erase(p)) std::abort();
  ++frees;
  std::free(p);
}
#define CHECK(c) if (!(c)) { std::printf("line %d: %s\n", __LINE__, #c); return 1; }
static const void *q(size_t i) { return reinterpret_cast<void *>(8 * i); }
int main() {
  {
    PartialBlocks b(take, give);
    // one block per queue, kept while it is large enough
    void *p0 = b.get(q(0), false, 0, 1000), *p1 = b.get(q(1), false, 0, 1000);
    CHECK(p0 && p1 && p0 != p1);
    CHECK(b.get(q(0), false, 0, 500) == p0 && b.get(q(1), false, 0, 1000) == p1);
    // growing leaves the old block alone (work on it may be under way), and
    // all that was replaced is smaller than what is in use
    void *g = b.get(q(0), false, 0, 1100);
    CHECK(g != p0 && g != p1 && live.count(p0) && live[g] >= 2 * live[p0]);
    CHECK(frees == 0 && b.get(q(1), false, 0, 1) == p1);
    // captures: their own blocks, one per queue of each
    void *c0 = b.get(q(0), true, 1, 800), *c1 = b.get(q(1), true, 1, 800),
         *c2 = b.get(q(0), true, 2, 800);
    std::set<void *> all{p0, p1, g, c0, c1, c2};
    CHECK(all.size() == 6 && !all.count(nullptr));
    CHECK(b.get(q(0), true, 1, 700) == c0);
    void *c3 = b.get(q(0), true, 1, 4000);
    CHECK(!all.count(c3) && live.count(c0) && live.count(c2));
    for (size_t n = 64; n < (1u << 20); n *= 2) b.get(q(0), false, 0, n);
    CHECK(live.count(c0) && live.count(c1) && live.count(c2) && live.count(c3));
    CHECK(b.get(q(0), true, 2, 800) == c2 && frees == 0);
    // no memory: no block, and what there was still serves
    dry = true;
    CHECK(!b.get(q(9), false, 0, 10) && !b.get(q(0), true, 3, 10));
    CHECK(!b.get(q(1), false, 0, 1 << 20) && b.get(q(1), false, 0, 9) == p1);
    dry = false;
  }
  CHECK(live.empty());
  {  // captures are bounded, and their blocks stay
    PartialBlocks b(take, give);
    const size_t part = PartialBlocks::kCaptureBytes / 8;
    std::set<void *> all;
    for (int i = 0; i < 8; ++i) all.insert(b.get(q(0), true, i, part));
    CHECK(all.size() == 8 && !all.count(nullptr));
    CHECK(!b.get(q(0), true, 8, 1) && all.count(b.get(q(0), true, 3, 1)));
    CHECK(b.get(q(0), false, 0, part) != nullptr);
    CHECK(!b.get(q(0), true, 9, ~(size_t)0 - 4096));
  }
  CHECK(live.empty());
  {  // queues are bounded: the one used longest ago gives all it has back
    PartialBlocks b(take, give);
    for (size_t i = 0; i < PartialBlocks::kQueues; ++i) b.get(q(i), false, 0, 100);
    void *p1 = b.get(q(1), false, 0, 100);
    b.get(q(0), false, 0, 1000);  // replaces one
    CHECK(live.size() == PartialBlocks::kQueues + 1);
    for (size_t i = 0; i < 3 * PartialBlocks::kQueues; ++i) {
      b.get(q(1000 + i), false, 0, 100);
      CHECK(b.get(q(1), false, 0, 100) == p1);
    }
    CHECK(live.size() == PartialBlocks::kQueues);
  }
  CHECK(live.empty());
  // the GEMV plan without partials
  for (int panel = 0; panel < 2; ++panel)
    for (long long R = 1; R < (1ll << 31); R = R * 5 / 3 + 1)
      for (long long C : {1, 7, 64, 100, 513, 4099, 1 << 20})
        for (int es : {4, 8})
          for (int batch : {1, 3, 1000}) {
            const int vn = 16 / es;
            const hcb::GemvPlan p = hcb::plan_gemv(256, panel, R, C, R >= vn, vn,
                                                   es, batch, false);
            const hcb::GemvPlan s = hcb::plan_gemv(256, panel, R, C, R >= vn, vn,
                                                   es, batch);
            CHECK(p.splits == 1 && p.partial_bytes == 0 && p.oblocks > 0);
            // a band kernel's splits are its bands
            if (p.kernel == hcb::GemvKernel::kBand16 ||
                p.kernel == hcb::GemvKernel::kBand8)
              CHECK(p.xr <= 16 && (long long)p.xr * 256 * vn >= R);
            if (s.splits == 1)
              CHECK(p.kernel == s.kernel && p.xr == s.xr && p.oblocks == s.oblocks);
          }
  std::printf("ok\n");
  return 0;
}
'''


def test_partial_blocks(tmp_path):
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not available")
    src, exe = tmp_path / "probe.cpp", tmp_path / "probe"
    src.write_text(PROBE)
    subprocess.run([gxx, "-std=c++17", "-O1", "-g", "-Wall", "-Werror",
                    "-Wno-dangling-else", "-I",
                    os.path.join(ROOT, "hcblas_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    p = subprocess.run([str(exe)], capture_output=True, text=True)
    assert p.returncode == 0 and p.stdout == "ok\n", p.stdout + p.stderr
