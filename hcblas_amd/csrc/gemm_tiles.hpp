// Tile choice and split-K plan of the MFMA GEMM (host only, no HIP dependency):
// shared by the launcher and the CPU test that checks which tiles the sizes of the
// GPU tests run on.
#pragma once

#include <algorithm>
#include <cstdint>

namespace hcb {

enum class Elem { F32, F64, F16, BF16, I8 };

inline int64_t ceil_div(int64_t a, int64_t b) { return (a + b - 1) / b; }

// Macro tiles, largest first, and the rate of each in TF/s over a grid of many
// tiles (8192 x 8192 x 1024 on MI355X), with 0, 1 or 2 operands r-contiguous
// (transposed on their way into LDS):
//   FP32  256x256x32, 8 waves of 128x64 on 32x32 MFMA blocks (146-148 TF/s at
//         8192^3, 93-94% of peak), 256x128 8 waves, 128x128, 64x64 and 32x32 4
//         waves;
//   FP64  256x128x16, 8 waves of 64x64 (71.6 TF/s at 8192^3, 91%), 128x64, 64x64
//         8 waves, 32x32 4 waves;
//   F16 / BF16 256x256x64, 8 waves on 32x32 blocks, 128x128 8 waves of 64x32,
//         64x64 4 waves (8192 x 8192 x 1024 HGEMM NN 292 us against 655 with 8,
//         whose r-contiguous tiles go to LDS by elements), 32x32 4 waves.
// (FP64 256x128 counts 70 for its lead at a long K: 4096^3 1960 us, 1995 on
// 128x64).
//
// `lead`: time of a tile beside its K loop, in k. The largest tiles fill a CU's
// LDS, so that nothing runs beside their first loads and their epilogue: a 16-bit
// 256x256 tile's are as long as 128 k. (BF16 12x 807x775x189 30 us on 256x256 tiles,
// 21 on 128x128; HGEMM 64x 446x732x224 36 and 31; but 64x 512^3 30 and 35, 120x
// 913x750x666 236 and 303. DGEMM 5516x1312x29 22.8 on 256x128, 21.4 on 128x64, 18.8
// on 64x64, 23.7 on 32x32.) A 32x32 FP32 tile pays more for its area than a 64x64
// one (SGEMM 120x 203x698x84 79 and 54 us, CGEMM 120x 130x130x40 28 and 24; but SGEMM
// 8x 255x257x517 16.3 and 17.1, CGEMM 64x 96^3 11.2 and 13.1). The FP32 and FP64
// leads were chosen on 1500 sizes (K from 16 to 2047, batches up to 256) timed on
// every tile: the choice loses 0.5% and 0.4% against the best tile in the mean. With
// 20 (FP64 10) for all tiles, 60 (35) for 32x32, it lost 1.6% and 1.2%, 10 to 20%
// at short K: DGEMM 7x 586x46x16 4.7 -> 3.9 us, 421x2944x26 9.0 -> 8.2, SGEMM 79x
// 128x352x17 10.1 -> 9.0.
struct MacroTile {
  int bm, bn;
  int rate[3];
  int lead = 0;
};
template <Elem E>
inline constexpr MacroTile kTiles[] = {{256, 256, {1180, 1110, 916}, 128},
                                       {128, 128, {1017, 820, 589}},
                                       {64, 64, {610, 465, 304}},
                                       {32, 32, {330, 238, 152}}};
template <>
inline constexpr MacroTile kTiles<Elem::F32>[] = {
    {256, 256, {140, 140, 133}, 60},
    {256, 128, {128, 128, 129}, 30},
    {128, 128, {133, 129, 127}, 40},
    {64, 64, {120, 117, 114}, 20},
    {32, 32, {105, 97, 80}, 55}};
template <>
inline constexpr MacroTile kTiles<Elem::F64>[] = {
    {256, 128, {70, 70, 70}, 40},
    {128, 64, {68, 68, 67}, 25},
    {64, 64, {66, 65, 65}, 20},
    {32, 32, {57, 54, 52}, 30}};

// The tile with the least time on the CU that gets the most tiles,
// ceil(tiles / CUs) * area * (K + lead) / rate: tiles past the edge of C and a
// last round that leaves most CUs idle count in full. (Taking the largest tile
// whose grid covers every CU instead: 3072 x 3072 x 1024 SGEMM NN 267 us on 288
// tiles of 256x128, 180 on 2304 of 64x64; 5512 x 6720 x 1024 738 on 256x256, 658
// on 128x128; a batch of 212 512 x 37 x 32 DGEMMs 36 us on 256x128, 21 on 64x64;
// 529 x 192 x 1152 28.8 on 27 tiles of 64x64, 12.1 on 32x32.)
template <Elem E>
inline const MacroTile &pick_tile(int64_t M, int64_t N, int64_t K,
                                  int64_t batch, int num_cus,
                                  int r_contiguous) {
  const MacroTile *best = nullptr;
  double least = 0;
  for (const MacroTile &t : kTiles<E>) {
    const int64_t tiles = ceil_div(M, t.bm) * ceil_div(N, t.bn) * batch;
    const double time = (double)ceil_div(tiles, num_cus) * t.bm * t.bn *
                        (double)(K + t.lead) / t.rate[r_contiguous];
    if (best == nullptr || time < least) {
      best = &t;
      least = time;
    }
  }
  return *best;
}

// An operand shorter than one 16-byte vector along its contiguous dimension, of a
// product of `ce` (1, complex: 2) reals per element and esize bytes per real; M and
// K are the real form's.
inline bool is_narrow(int M, int N, int K, bool a_k, bool b_k, int ce,
                      int esize) {
  const int vec = 16 / (ce * esize);
  return (a_k ? K : M) / ce < vec || (b_k ? K / ce : N) < vec;
}

// How a single problem's K is split: `splits` slices of `ks`, on tiles of
// `tile` x `tile`; splits == 1 where it does not pay.
struct SplitK {
  int splits, ks, tile;
};

// It pays when the 64x64 tiles leave at least half the CUs idle and K is long:
// the second launch and the partials cost 3-5 us, which K = 2048 on one wave of
// workgroups just earns back (SGEMM NN, unsplit 32x32 tiles against split:
// 128 x 128 x 2048 18.6 and 8.9 us, 16 x 2000 x 2000 19.0 and 10.1,
// 512 x 512 x 2048 19.2 and 18.0, 1000 x 128 x 1024 10.7 and 9.3). Up to 8
// slices, aiming at four workgroups per CU: of at least 256 on 32x32 tiles where
// those still leave a CU idle, else of at least 512 on 64x64 tiles. (1024^3,
// with one tile per CU, measured slower split: 30 us against 26.)
inline SplitK splitk_plan(int M, int N, int K, int num_cus, int bk32,
                          int bk64) {
  auto tiles = [&](int t) {
    return ((int64_t)M + t - 1) / t * (((int64_t)N + t - 1) / t);
  };
  SplitK sk{1, K, 64};
  if (K < 2048 || 2 * tiles(64) > num_cus) return sk;
  if (tiles(32) < num_cus) sk.tile = 32;
  int64_t S = std::min<int64_t>(8, 4 * (int64_t)num_cus / tiles(sk.tile));
  S = std::min<int64_t>(S, K / (sk.tile == 32 ? 256 : 512));
  if (S < 2) return sk;
  const int bk = sk.tile == 32 ? bk32 : bk64;
  sk.ks = (int)((K + S - 1) / S);
  sk.ks = (sk.ks + bk - 1) / bk * bk;
  sk.splits = (K + sk.ks - 1) / sk.ks;
  return sk;
}

}  // namespace hcb
