// Definition of launch_gemm; included once per element type so the template
// instances compile in parallel translation units.
#pragma once

#include "gemm_launch.hpp"

namespace hcb {

// K steps: of the large tiles (BK_BIG); of 64x64 and 32x32 tiles; and of 32x32
// tiles that leave CUs idle, from K = LONG_K on (few steps hide little of the
// load latency; a long step pads a short K): 529 x 192 x 1152 FP64 NN 20.6 us
// with 64 against 24.7 with 16, 529 x 1152 x 192 12.3 against 11.0.
template <Elem E>
struct TileCfg;
template <>
struct TileCfg<Elem::F32> {
  static constexpr int BK_BIG = 32, BK_64 = 32;
  static constexpr int BK_32 = 64, BK_32_LONG = 128, LONG_K = 1024;
};
template <>
struct TileCfg<Elem::F64> {
  static constexpr int BK_BIG = 16, BK_64 = 16;
  static constexpr int BK_32 = 32, BK_32_LONG = 64, LONG_K = 512;
};
template <>
struct TileCfg<Elem::F16> {
  static constexpr int BK_BIG = 64, BK_64 = 64;
  static constexpr int BK_32 = 64, BK_32_LONG = 128, LONG_K = 1024;
};
template <>
struct TileCfg<Elem::BF16> : TileCfg<Elem::F16> {};

template <Elem E, typename OutT, int BM, int BN, int BK, int WM, int WN,
          int MI = 16, bool CX = false, bool NARROW = false>
hcblasStatus_t launch_tiles(hipStream_t stream, GemmParams p, bool a_k,
                            bool b_k, int64_t batch) {
  p.tiles_m = (int)cdiv(p.M, BM);
  p.tiles_n = (int)cdiv(p.N, BN);
  const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n);
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
    GemmParams q = p;
    const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
    if (b0) {
      // Advance strided bases / pointer arrays to this chunk of the batch.
      if (q.Aptrs) q.Aptrs += b0;
      else q.A = (const char *)q.A + b0 * q.strideA * sizeof(typename ElemT<E>::T);
      if (q.Bptrs) q.Bptrs += b0;
      else q.B = (const char *)q.B + b0 * q.strideB * sizeof(typename ElemT<E>::T);
      if (q.Cptrs) q.Cptrs += b0;
      else q.C = (char *)q.C + b0 * q.strideC * sizeof(OutT);
    }
    dim3 grid(tiles, 1, (unsigned)nb);
#define HCB_GEMM_CASE(AK, BKC)                                             \
  if (a_k == AK && b_k == BKC)                                             \
    gemm_mfma_kernel<E, OutT, AK, BKC, BM, BN, BK, WM, WN, MI, CX, NARROW> \
        <<<grid, 64 * WM * WN, 0, stream>>>(q);
    HCB_GEMM_CASE(false, false)
    HCB_GEMM_CASE(false, true)
    HCB_GEMM_CASE(true, false)
    HCB_GEMM_CASE(true, true)
#undef HCB_GEMM_CASE
    hcblasStatus_t st = launch_status();
    if (st != HCBLAS_STATUS_SUCCESS) return st;
  }
  return HCBLAS_STATUS_SUCCESS;
}

// 64x64 (or, with `t32`, 32x32) tiles, `tiles` of them.
template <Elem E, typename OutT, bool CX, bool NARROW>
hcblasStatus_t launch_small(hipStream_t stream, int num_cus, GemmParams p,
                            bool a_k, bool b_k, int64_t batch, bool t32,
                            int64_t tiles) {
  using C = TileCfg<E>;
  if (t32) {
    if (p.K >= C::LONG_K && tiles <= num_cus)
      return launch_tiles<E, OutT, 32, 32, C::BK_32_LONG, 2, 2, 16, CX, NARROW>(
          stream, p, a_k, b_k, batch);
    // (16-bit r-contiguous tiles of 128-deep steps are transposed in
    // registers: 8192 x 8192 x 1024 HGEMM NN 564 us against 743)
    if (sizeof(typename ElemT<E>::T) == 2 && !(a_k && b_k))
      return launch_tiles<E, OutT, 32, 32, C::BK_32_LONG, 2, 2, 16, CX, NARROW>(
          stream, p, a_k, b_k, batch);
    return launch_tiles<E, OutT, 32, 32, C::BK_32, 2, 2, 16, CX, NARROW>(
        stream, p, a_k, b_k, batch);
  }
  // 64x64 tiles. At most one tile per CU leaves nothing else to cover a tile's
  // load latency: FP32 then runs 8 waves and long K steps (1024^3 NN 22.8 us
  // with 128, 23.7 with 64, 27.5 with 4 waves and 32), FP64 32-deep ones
  // (1024^3 42.3 against 44.1). With more tiles than CUs, 4 waves and short
  // steps are ahead for FP32 (4096 x 4096 x 256 NN 84 us against 89 with 8
  // waves and 92 with 64-deep steps), and so they are where one step is all.
  // FP32 tiles of a single 32-deep step, and narrow 16-bit ones, take 8 waves,
  // which share its loads and the epilogue: SGEMM 3025 x 96 x 1 4.6 -> 3.8 us,
  // 3200 x 256 x 23 5.0 -> 4.1, HGEMM 1000 x 1000 x 4 4.1 -> 3.8 (but HGEMM 2000 x
  // 1000 x 48 4.6 -> 5.5, CGEMM 500 x 300 x 16 4.4 -> 5.8).
  if constexpr (!CX && (E == Elem::F32 || (NARROW && E != Elem::F64))) {
    if (p.K <= C::BK_64)
      return launch_tiles<E, OutT, 64, 64, C::BK_64, 2, 4, 16, CX, NARROW>(
          stream, p, a_k, b_k, batch);
  }
  if constexpr (E == Elem::F32) {
    if (p.K >= 512 && tiles <= num_cus)
      return launch_tiles<E, OutT, 64, 64, 128, 2, 4, 16, CX, NARROW>(
          stream, p, a_k, b_k, batch);
    if (tiles <= num_cus)
      return launch_tiles<E, OutT, 64, 64, 64, 2, 4, 16, CX, NARROW>(
          stream, p, a_k, b_k, batch);
  }
  if constexpr (E == Elem::F64) {
    if (tiles <= num_cus && p.K > C::BK_64)
      return launch_tiles<E, OutT, 64, 64, 32, 2, 4, 16, CX, NARROW>(
          stream, p, a_k, b_k, batch);
    return launch_tiles<E, OutT, 64, 64, C::BK_64, 2, 4, 16, CX, NARROW>(
        stream, p, a_k, b_k, batch);
  } else {
    return launch_tiles<E, OutT, 64, 64, C::BK_64, 2, 2, 16, CX, NARROW>(
        stream, p, a_k, b_k, batch);
  }
}

template <Elem E, typename OutT, bool CX>
hcblasStatus_t launch_gemm(hipStream_t stream, int num_cus, GemmParams p,
                           bool a_k, bool b_k, int64_t batch) {
  using C = TileCfg<E>;
  const MacroTile &t =
      pick_tile<E>(p.M, p.N, p.K, batch, num_cus,
                   CX ? 0 : (a_k ? 0 : 1) + (b_k ? 0 : 1));
  auto tiles = [&](int bm, int bn) {
    return cdiv(p.M, bm) * cdiv(p.N, bn) * batch;
  };
  // Narrow operands are a few rows or a K below one vector: the small tiles do
  // for them, and for 16-bit ones those of 128x128 (8192 x 8192 x 4 HGEMM 42 us,
  // on 64x64 tiles 58; SGEMM 72 on 64x64).
  if (is_narrow(p.M, p.N, p.K, a_k, b_k, CX ? 2 : 1,
                (int)sizeof(typename ElemT<E>::T))) {
    if constexpr (sizeof(typename ElemT<E>::T) == 2) {
      if (t.bm >= 128)
        return launch_tiles<E, OutT, 128, 128, C::BK_BIG, 2, 4, 32, CX, true>(
            stream, p, a_k, b_k, batch);
    }
    const bool t32 = t.bm == 32;
    return launch_small<E, OutT, CX, true>(
        stream, num_cus, p, a_k, b_k, batch, t32,
        t32 ? tiles(32, 32) : tiles(64, 64));
  }
  if constexpr (E == Elem::F64) {
    if (t.bm == 256)
      return launch_tiles<E, OutT, 256, 128, C::BK_BIG, 4, 2, 16, CX>(
          stream, p, a_k, b_k, batch);
    if (t.bm == 128)
      return launch_tiles<E, OutT, 128, 64, C::BK_BIG, 2, 4, 16, CX>(
          stream, p, a_k, b_k, batch);
  } else {
    if (t.bn == 256)
      return launch_tiles<E, OutT, 256, 256, C::BK_BIG, 2, 4, 32, CX>(
          stream, p, a_k, b_k, batch);
    if constexpr (E == Elem::F32) {
      if (t.bm == 256)
        return launch_tiles<E, OutT, 256, 128, C::BK_BIG, 2, 4, 16, CX>(
            stream, p, a_k, b_k, batch);
      if (t.bm == 128)
        return launch_tiles<E, OutT, 128, 128, C::BK_BIG, 2, 2, 16, CX>(
            stream, p, a_k, b_k, batch);
    } else {
      // 8 waves of 64 x 32 (fragment read-ahead, two-vector transposed loads):
      // 2048^3 HGEMM NN 38.6 against 44.4 us with 4 waves of 64 x 64.
      if (t.bm == 128)
        return launch_tiles<E, OutT, 128, 128, C::BK_BIG, 2, 4, 32, CX>(
            stream, p, a_k, b_k, batch);
    }
  }
  return launch_small<E, OutT, CX, false>(stream, num_cus, p, a_k, b_k, batch,
                                          t.bm == 32, tiles(t.bm, t.bn));
}

template <Elem E, int T, int BK, int WM, int WN, bool CX>
void launch_splitk_tiles(hipStream_t stream, GemmParams p, bool a_k, bool b_k,
                         const SplitK &sk, typename ElemT<E>::Acc *W) {
  p.tiles_m = (int)cdiv(p.M, T);
  p.tiles_n = (int)cdiv(p.N, T);
  dim3 grid((unsigned)(p.tiles_m * p.tiles_n), 1, (unsigned)sk.splits);
  const bool narrow = is_narrow(p.M, p.N, p.K, a_k, b_k, CX ? 2 : 1,
                                (int)sizeof(typename ElemT<E>::T));
#define HCB_SPLITK_CASE(AK, BKC)                                           \
  if (a_k == AK && b_k == BKC)                                             \
    (narrow ? gemm_splitk_kernel<E, AK, BKC, T, T, BK, WM, WN, 16, CX, true>   \
            : gemm_splitk_kernel<E, AK, BKC, T, T, BK, WM, WN, 16, CX, false>) \
        <<<grid, 64 * WM * WN, 0, stream>>>(p, sk.ks, W);
  HCB_SPLITK_CASE(false, false)
  HCB_SPLITK_CASE(false, true)
  HCB_SPLITK_CASE(true, false)
  HCB_SPLITK_CASE(true, true)
#undef HCB_SPLITK_CASE
}

template <Elem E, typename OutT, bool CX>
hcblasStatus_t launch_gemm_splitk(hipStream_t stream, int num_cus,
                                  GemmParams p, bool a_k, bool b_k,
                                  const SplitK &sk,
                                  typename ElemT<E>::Acc *W) {
  using Acc = typename ElemT<E>::Acc;
  // (64x64 FP64 256 x 128 x 16384 96 us with 8 waves of 32 x 16 against 123 with
  // 4 of 32 x 32)
  if (sk.tile == 32)
    launch_splitk_tiles<E, 32, TileCfg<E>::BK_32_LONG, 2, 2, CX>(stream, p, a_k,
                                                             b_k, sk, W);
  else
    launch_splitk_tiles<E, 64, TileCfg<E>::BK_64, 2,
                        sizeof(typename ElemT<E>::T) == 2 ? 2 : 4, CX>(
        stream, p, a_k, b_k, sk, W);
  hcblasStatus_t st = launch_status();
  if (st != HCBLAS_STATUS_SUCCESS) return st;
  const int64_t MN = (int64_t)p.M * p.N;
  const int64_t nb = cdiv(MN, 256);
  const unsigned g = (unsigned)(nb < 4 * num_cus ? nb : 4 * num_cus);
  splitk_reduce_kernel<Acc, OutT><<<g, 256, 0, stream>>>(
      sk.splits, p.M, p.N, W, static_cast<OutT *>(p.C) + p.cOff, p.ldc,
      (Acc)p.alpha, (Acc)p.beta);
  return launch_status();
}

}  // namespace hcb
