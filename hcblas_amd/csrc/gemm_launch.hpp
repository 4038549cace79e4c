// Host launcher for the generic MFMA GEMM kernel: picks a macro-tile shape
// and the template instance matching the operand orientations.
#pragma once

#include "gemm_kernel.hpp"

namespace hcb {

// Launches C = alpha*A'*B' + beta*C for `batch` problems described by p
// (column-major storage; a_k / b_k give the operand orientations); CX: the real
// embedding of a complex product, formed by the tile loaders.
template <Elem E, typename OutT, bool CX = false>
hcblasStatus_t launch_gemm(hipStream_t stream, int num_cus, GemmParams p,
                           bool a_k, bool b_k, int64_t batch);

// How a single problem's K is split: `splits` slices of `ks`, on tiles of
// `tile` x `tile`; splits == 1 where it does not pay.
struct SplitK {
  int splits, ks, tile;
};

// Split-K form for one problem (no batch, no pointer arrays): partial tiles of
// the K slices into W (splits * M * N accumulators), then the reduction into C.
template <Elem E, typename OutT, bool CX = false>
hcblasStatus_t launch_gemm_splitk(hipStream_t stream, int num_cus,
                                  GemmParams p, bool a_k, bool b_k,
                                  const SplitK &sk,
                                  typename ElemT<E>::Acc *W);

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
