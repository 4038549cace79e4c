// Launch plan of the GEMV kernels (host only, no HIP dependency): which
// kernel runs, its grid, the reduction split count and the bytes of split
// partials it needs. Shared by level2.hip and the CPU test that checks the
// partials of the allocation-free entry against its fixed scratch.
#pragma once

#include <algorithm>
#include <cstddef>
#include <cstdint>

namespace hcb {

// Kernel geometry constants of level2.hip.
constexpr int kGemvThreads = 256;
constexpr int kCPW = 4;           // columns per wave of the column kernel
constexpr int kColsPerBlock = 4 * kCPW;
constexpr int kBandCols = 8;      // columns per workgroup of the band kernel

// kBand16: the band kernel with 16 row steps; kBand8: with 1 to 14.
enum class GemvKernel { kBandN, kPanel, kBand16, kBand8, kColumn };

struct GemvPlan {
  GemvKernel kernel;
  int xr;           // row steps of a band (band kernels)
  int waves;        // waves per workgroup (panel kernel)
  int64_t oblocks;  // output blocks (grid x, or grid y for band-N)
  int splits;       // reduction splits (grid y, or grid x for band-N)
  size_t partial_bytes;  // split partials (0 when splits == 1)
};

inline int64_t plan_cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// panel: the reduction runs along the contiguous storage rows' columns
// (y has R entries); otherwise along the rows (y has Cc entries). vec: rows
// are read 16 bytes at a time (vn elements; R >= vn). esize: element bytes.
//
// Every rule aims at a grid that covers the GPU (what a memory-bound kernel
// lacks on a small or narrow matrix is loads in flight, not their width) but
// not at a few workgroups more than the GPU holds side by side: 258 bands of
// a 12000^2 SGEMV-N took 120 us, 255 took 91.
// split = false: the same without split reductions (there is no memory for the
// partials).
inline GemvPlan plan_gemv(int num_cus, bool panel, int64_t R, int64_t Cc,
                          bool vec, int vn, size_t esize, int64_t batch,
                          bool split = true) {
  const int64_t len_y = panel ? R : Cc;
  const int64_t target = (int64_t)num_cus * 4;  // workgroups to aim for
  GemvPlan p{GemvKernel::kColumn, 0, 4, 1, 1, 0};
  const int64_t step = (int64_t)kGemvThreads * vn;  // rows of one band step
  const int64_t steps = plan_cdiv(R, step);
  // Below three quarters of a step a band would leave a whole wave idle.
  const bool band = vec && 4 * R >= 3 * step;
  // Row-contiguous case of 129 to 512 columns and at most 32 MB: sixteen waves per
  // 64 vectors of rows, a wave's columns in at most two trips, one launch. (Each
  // workgroup reads 1 KiB of every column; the split form's second launch
  // costs more than the CUs that stay idle. Up to 128 columns four waves do: 3.6
  // us in the mean against 4.0.)
  const int64_t pblocks = plan_cdiv(R, 64 * (int64_t)(vec ? vn : 1));
  const bool short_sums = panel && Cc > 128 && Cc <= 512 &&
                          pblocks * batch < 2 * (int64_t)num_cus &&
                          R * Cc * (int64_t)esize * batch <= (32ll << 20);
  // Column case. A band of up to 16 steps, all bands alike (R = 20011, 20
  // steps: two bands of 10 instead of 16 and 4), and more, shorter bands
  // where the column blocks are few: up to one workgroup per CU, bands of at
  // least 2 steps, from 5 steps on (below, the second launch costs more than they
  // save: 3 steps 5.5 us in one band, 6.8 in two).
  // Up to 128 MB the column kernel is ahead where a band's lanes idle: more than a
  // quarter of them (0.86 to 0.9 of the band's time, 1 to 3 steps; with few idle
  // ones up to 1.1), and of rows that are whole vectors up to 1.8 steps (0.86 to
  // 0.93; above 1.0). Larger matrices stream faster in bands at any row count
  // (1024 x 100000 fp32 61 us, 77).
  const bool columns = R * Cc * (int64_t)esize * batch < (128ll << 20) &&
                       (4 * R < 3 * steps * step ||
                        (R % vn == 0 && 5 * R < 9 * step));
  int64_t bands = plan_cdiv(steps, 16);
  if (split && steps >= 5) {
    const int64_t blocks = plan_cdiv(Cc, kBandCols) * batch;
    bands = std::max(bands,
                     std::min((int64_t)num_cus / blocks, (steps + 1) / 2));
  }
  if (!panel && band && !columns && bands <= (split ? 65535 : 1)) {
    int64_t xr = plan_cdiv(steps, bands);
    if (xr > 4) xr = (xr + 1) / 2 * 2;  // instances: 1..4, 6, 8, .. 16
    p.kernel = xr == 16 ? GemvKernel::kBand16 : GemvKernel::kBand8;
    p.xr = (int)xr;
    p.oblocks = plan_cdiv(Cc, kBandCols);
    p.splits = (int)plan_cdiv(steps, xr);
  } else if (panel && band && Cc > 512 && steps <= 65535) {
    // Row-contiguous case (up to 512 columns the panel kernel is as fast or
    // faster: 1024 x 225 fp64 in a batch of 43 13.7 us, here 20.1): bands of 4
    // steps (16 KiB of each column in one run) where they waste at most an
    // eighth of their lanes and, with at least 64 columns per block, still give
    // every CU a workgroup; else 2 or 1. Column blocks: about one workgroup per CU (at 16384^2 fp32 256
    // workgroups took 152 us, 128 178 us, 512 159 us), at least 32 columns.
    // (4096^2 fp32 used one band of 4 steps in 16 blocks: 16 workgroups,
    // 75 us.)
    int xr = 1;
    for (int x : {4, 2}) {
      const int64_t b = plan_cdiv(steps, x);
      if (8 * R >= 7 * b * x * step &&
          b * batch * plan_cdiv(Cc, 64) >= num_cus) {
        xr = x;
        break;
      }
    }
    p.kernel = GemvKernel::kBandN;
    p.xr = xr;
    p.oblocks = plan_cdiv(steps, xr);
    p.splits = (int)std::max<int64_t>(
        1, std::min(plan_cdiv(Cc, 32), num_cus / (p.oblocks * batch)));
  } else if (panel) {
    p.kernel = GemvKernel::kPanel;
    p.oblocks = pblocks;
    // Otherwise, above 128 columns, splits of at least 8 columns for each of
    // four waves, or of 32 where the row blocks give every CU a workgroup.
    if (short_sums)
      p.waves = 16;
    else if (Cc > 128)
      p.splits = (int)std::min<int64_t>(
          plan_cdiv(target, p.oblocks * batch),
          std::min<int64_t>(256, Cc / (p.oblocks * batch < num_cus ? 32 : 128)));
  } else {
    p.kernel = GemvKernel::kColumn;
    p.oblocks = plan_cdiv(Cc, kColsPerBlock);
    const int64_t rsteps = plan_cdiv(R, 64 * (vec ? vn : 1));
    const int64_t max_split = std::max<int64_t>(1, rsteps / 16);
    p.splits = (int)std::min<int64_t>(
        std::max<int64_t>(1, plan_cdiv(target, p.oblocks * batch)),
        std::min<int64_t>(256, max_split));
  }
  if (!split) p.splits = 1;
  if (p.splits > 1)
    p.partial_bytes = esize * (size_t)p.splits * (size_t)len_y *
                      (size_t)std::min<int64_t>(batch, 65535);
  return p;
}

// Launch plan of the GEMV pair kernel (both products of one matrix in one
// pass): bands of `xr` row steps x blocks of columns; xr == 0 where the two
// GEMVs are to run instead.
struct PairPlan {
  int xr;
  int64_t bands, blocks;
  size_t partial_bytes;
};

// Matrices of 4 MB on whose rows fill a band step to three quarters: below, a
// GEMV is a launch and little else. Bands as in plan_gemv's row-contiguous case,
// blocks of 32 to 512 columns for about one workgroup per CU (fp32 4500 x 1000
// 11.8 us with at least 32 columns, 13.0 with 16, 18.3 with 8 and four
// workgroups per CU; 4096^2 21.0, 21.0 and 27.5). Against the two GEMVs, both
// finish launches included: fp32 4096^2 28.2 -> 21.0 us, 1100 x 1000 12.8 -> 9.1,
// 2500^2 18.4 -> 15.2; fp64 4096^2 48.1 -> 30.4, 700 x 3000 19.0 -> 14.2.
inline PairPlan plan_gemv_pair(int num_cus, int64_t R, int64_t Cc, int vn,
                               size_t esize) {
  PairPlan p{0, 0, 0, 0};
  const int64_t step = (int64_t)kGemvThreads * vn;
  const int64_t steps = plan_cdiv(R, step);
  if (4 * R < 3 * step || Cc < 64 || steps > 65535 ||
      R * Cc * (int64_t)esize < (4ll << 20))
    return p;
  p.xr = 1;
  for (int x : {4, 2}) {
    const int64_t b = plan_cdiv(steps, x);
    if (8 * R >= 7 * b * x * step && b * plan_cdiv(Cc, 32) >= num_cus) {
      p.xr = x;
      break;
    }
  }
  p.bands = plan_cdiv(steps, p.xr);
  p.blocks = std::max<int64_t>(
      2, std::min(plan_cdiv(Cc, 32), num_cus / p.bands));
  p.blocks = std::max(p.blocks, plan_cdiv(Cc, 512));
  p.partial_bytes =
      esize * (size_t)(p.blocks * R + (p.bands > 1 ? p.bands * Cc : 0));
  return p;
}

}  // namespace hcb
