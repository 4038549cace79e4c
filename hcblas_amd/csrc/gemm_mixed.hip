// Mixed BF16 / FP32 GEMM for the adjoints of the BF16 batched GEMM (no
// reference counterpart): C = alpha * A' * B' in FP32 where one operand is
// FP32 (the cotangent dC) and the other BF16 (the forward's A or B), read as
// they lie in memory -- no widened and no transposed copy.
//
// The FP32 operand is split on its way into LDS into three BF16 planes,
// x = hi + mid + lo with each part the BF16 rounding of the remaining
// residual (exact for finite x: 3 x 8 bits hold the 24-bit significand), so
// hi*b + mid*b + lo*b equals x*b exactly for a BF16 b. Each K chunk issues
// the three products on v_mfma_f32_32x32x16_bf16 from one BF16 fragment of
// the other operand (smallest first) into one FP32 accumulator: the sums are
// those of an FP32 GEMM of the exact products, at three BF16 MFMAs per 16 k
// instead of eight FP32 MFMAs (v_mfma_f32_32x32x2f32 takes 2 k).
//
// Tile: 256 x 256 x 32 over 8 waves of 64 x 128, 128 x 128 x 32 over 4 waves of
// 64 x 64 or 64 x 64 x 32 over 2 waves of 32 x 64, LDS double-buffered like the
// plain kernel (the FP32 operand's tile is three planes), epilogue through LDS
// with the plain kernels' arithmetic; the result is rounded once to BF16.
//
// What bounds it: the MFMAs, and beside them the split's VALU work on the same
// SIMDs, the LDS, and the prologue and epilogue of a tile that fills a CU.
// (Counters of 256 x 256x1024x512: MFMAs busy 53% of dA, 189 us, and 38% of dB, 268
// us of 8 K steps a tile; 43-46% of wave time in s_waitcnt; 11-14% of the LDS
// cycles are conflicts. With the planes' writes two to a bank and integer
// rounding in the epilogue, 8 operations per output, dA took 223 us where it then
// took 204, dB 293 and 246.) v_cvt_pk_bf16_f32 rounds two values at once, about 8
// operations per element where integer rounding took 18. An operand stored with the inner index as its row index (both
// operands of dB = op(A)^T dC) is transposed in registers by the tile loader: a
// thread holds a 4 x 4 block of FP32 or two k-lines of 8 BF16 rows and writes
// along k, as many LDS writes as the k-contiguous form. (Transposed copies of dC
// and A in a workspace took 115 us of the 256 x 256x1024x512 backward's 700.)
#include "gemm_common.hpp"

namespace hcb {
namespace {

__device__ __forceinline__ float bf16_val(uint16_t b) {
  return __uint_as_float((uint32_t)b << 16);
}

// Two floats rounded to BF16 (nearest even), packed: v_cvt_pk_bf16_f32.
__device__ __forceinline__ uint32_t cvt_pk_bf16(float a, float b) {
  typedef float floatx2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return bitcast<uint32_t>(__builtin_convertvector(floatx2{a, b}, bf16x2));
}

// x = hi + mid + lo for a pair (packed BF16 bits); non-finite x keeps hi =
// bf16(x) (NaN stays NaN) and zero residual planes.
__device__ __forceinline__ void split3_pair(float x0, float x1, uint32_t &h,
                                            uint32_t &m, uint32_t &l) {
  h = cvt_pk_bf16(x0, x1);
  float r0 = x0 - __uint_as_float(h << 16);
  float r1 = x1 - __uint_as_float(h & 0xFFFF0000u);
  r0 = __builtin_isfinite(x0) ? r0 : 0.f;
  r1 = __builtin_isfinite(x1) ? r1 : 0.f;
  m = cvt_pk_bf16(r0, r1);
  l = cvt_pk_bf16(r0 - __uint_as_float(m << 16),
                  r1 - __uint_as_float(m & 0xFFFF0000u));
}

// Global -> register loader of an FP32 tile (the plain kernel's loader) whose
// store writes three BF16 planes [ROWS][BK] (row stride BK*2 + 16 bytes,
// planes PLANE bytes apart) in the BF16 operand's LDS layout.
template <int ROWS, int BK, bool KCONT, int NTH>
struct SplitPlaneLoader : TileLoader<float, ROWS, BK, KCONT, NTH> {
  using L = TileLoader<float, ROWS, BK, KCONT, NTH>;
  // The loader's vectors in an order in which the 8-byte LDS writes of 16 and of
  // 32 consecutive lanes fall on distinct banks (rows are 80 bytes apart):
  // k-contiguous, 32 lanes take rows 0, 4, 8, 12 (64 bytes each at offsets 0,
  // 64, 128, 192 of 256) instead of 0 .. 3; 4 x 4 blocks, 4 r-vectors (64 bytes
  // apart) by all 8 k-quads instead of twice 4.
  __device__ __forceinline__ static int order(int t) {
    static_assert(BK == 32, "eight vectors along k");
    if (KCONT) return (t & ~0x78) | ((t >> 2) & 0x18) | ((t << 2) & 0x60);
    return ((t >> 3) & 3) | ((t & 3) << 2) | ((t >> 5) << 4) |
           (((t >> 2) & 1) * ROWS);  // 16 threads per group, ROWS / 16 groups
  }
  __device__ __forceinline__ explicit SplitPlaneLoader(int t) : L(order(t)) {}
  static_assert(KCONT || L::TRANS4, "4 x 4 blocks");
  static_assert(L::NV % NTH == 0, "whole vectors per thread");
  static constexpr int ROWB = BK * 2 + 16;
  static constexpr int PLANE = ROWS * ROWB;
  __device__ __forceinline__ void store(char *lds) const {
#pragma unroll
    for (int i = 0; i < L::PER_THREAD; ++i) {
      // four consecutive k of one row: 8 bytes per plane
      int r, k;
      L::vec_pos(KCONT ? this->tid + i * NTH : this->tid, r, k);
      uint32_t v[4];
#pragma unroll
      for (int e = 0; e < 4; ++e)
        v[e] = KCONT ? this->reg[i][e] : this->reg[e][i];
      char *p = lds + (KCONT ? r : r + i) * ROWB + k * 2;
      uint32_t h[2], m[2], l[2];
#pragma unroll
      for (int e = 0; e < 2; ++e)
        split3_pair(__uint_as_float(v[2 * e]), __uint_as_float(v[2 * e + 1]),
                    h[e], m[e], l[e]);
      *reinterpret_cast<vec2u *>(p) = vec2u{h[0], h[1]};
      *reinterpret_cast<vec2u *>(p + PLANE) = vec2u{m[0], m[1]};
      *reinterpret_cast<vec2u *>(p + 2 * PLANE) = vec2u{l[0], l[1]};
    }
  }
};

constexpr int kMBK = 32;
constexpr int kMRowB = kMBK * 2 + 16;
// LDS bytes of one K step: the FP32 operand's three planes and the BF16
// operand's tile; two of them double-buffer the main loop.
template <bool AF, int BM, int BN>
constexpr int mixed_buf_bytes() {
  return ((AF ? 3 : 1) * BM + (AF ? 1 : 3) * BN) * kMRowB;
}

// BF16 output element (bits), rounded to nearest even from FP32; NaN stays
// a quiet NaN.
struct Bf16Out {
  uint16_t bits;
};
}  // namespace
template <>
__device__ __forceinline__ Bf16Out to_out<Bf16Out, float>(float v) {
  return Bf16Out{(uint16_t)cvt_pk_bf16(v, v)};
}
template <>
__device__ __forceinline__ float from_out<float, Bf16Out>(Bf16Out v) {
  return bf16_val(v.bits);
}
namespace {

struct MixedParams {
  int M, N, K;
  const void *A;
  int64_t lda, strideA;
  const void *B;
  int64_t ldb, strideB;
  void *C;
  int64_t ldc, strideC;
  float alpha;
  int tiles_m, tiles_n;
};

// AF: A' is the FP32 operand (else B' is). A_K / B_K: k-contiguous operands.
// BM x BN tile over WM x WN waves.
template <bool AF, bool A_K, bool B_K, int BM, int BN, int WM, int WN>
__global__ __launch_bounds__(64 * WM * WN) void gemm_mixed_kernel(
    MixedParams p) {
  constexpr int NTH = 64 * WM * WN, MI = 32;
  using WT = WaveTile<Elem::BF16, BM, BN, WM, WN, MI>;
  constexpr int FM = WT::FM, FN = WT::FN, WTM = WT::WTM, WTN = WT::WTN;
  constexpr int PLANE_A = BM * kMRowB, PLANE_B = BN * kMRowB;
  constexpr int BUF = mixed_buf_bytes<AF, BM, BN>(), LDS = 2 * BUF;
  __shared__ __attribute__((aligned(16))) char lds[LDS];
  using FL_A = SplitPlaneLoader<BM, kMBK, A_K, NTH>;
  using FL_B = SplitPlaneLoader<BN, kMBK, B_K, NTH>;
  using HL_A = TileLoader<uint16_t, BM, kMBK, A_K, NTH>;
  using HL_B = TileLoader<uint16_t, BN, kMBK, B_K, NTH>;
  using LA = typename std::conditional<AF, FL_A, HL_A>::type;
  using LB = typename std::conditional<AF, HL_B, FL_B>::type;
  using TA = typename std::conditional<AF, float, uint16_t>::type;
  using TB = typename std::conditional<AF, uint16_t, float>::type;
  // LDS buffer: A region (3 planes if FP32, else 1) then B region
  constexpr int A_BYTES = (AF ? 3 : 1) * PLANE_A;

  int z, pid;
  batch_tile(p.tiles_m * p.tiles_n, z, pid);
  const TA *A = static_cast<const TA *>(p.A) + (int64_t)z * p.strideA;
  const TB *B = static_cast<const TB *>(p.B) + (int64_t)z * p.strideB;
  Bf16Out *C = static_cast<Bf16Out *>(p.C) + (int64_t)z * p.strideC;
  int tile_m, tile_n;
  tile_coords(pid, p.tiles_m, p.tiles_n, tile_m, tile_n, gridDim.z < 8);
  const int m0 = tile_m * BM, n0 = tile_n * BN;

  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int lrow = lane % MI, lgrp = lane / MI;
  typename WT::AccV acc[FM][FN];
#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = typename WT::AccV{};

  LA la(threadIdx.x);
  LB lb(threadIdx.x);
  const int K = p.K;
  const int nk = (K + kMBK - 1) / kMBK;
  const int nfull =
      LA::wide(p.M, K) && LB::wide(p.N, K) ? K / kMBK : 0;  // no K tail
  auto buf = [&](int kt) { return lds + (kt & 1) * BUF; };
  auto load = [&](int k, bool full) {
    la.load_step(A, p.lda, m0, k * kMBK, p.M, K, full);
    lb.load_step(B, p.ldb, n0, k * kMBK, p.N, K, full);
  };
  auto store = [&](int k) {
    la.store(buf(k));
    lb.store(buf(k) + A_BYTES);
  };
  // MFMAs of one K step; hook() is issued with the first chunk's fragments.
  auto compute = [&](const char *cur, auto hook) {
    const char *As = cur + (wm * WTM + lrow) * kMRowB;
    const char *Bs = cur + A_BYTES + (wn * WTN + lrow) * kMRowB;
#pragma unroll
    for (int c = 0; c < kMBK / 16; ++c) {
      const int kbyte = (c * 16 + lgrp * 8) * 2;
      vec4u af[AF ? 3 : 1][FM], bf[AF ? 1 : 3][FN];
#pragma unroll
      for (int q = 0; q < (AF ? 3 : 1); ++q)
#pragma unroll
        for (int i = 0; i < FM; ++i)
          af[q][i] = *reinterpret_cast<const vec4u *>(
              As + q * PLANE_A + i * MI * kMRowB + kbyte);
#pragma unroll
      for (int q = 0; q < (AF ? 1 : 3); ++q)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          bf[q][j] = *reinterpret_cast<const vec4u *>(
              Bs + q * PLANE_B + j * MI * kMRowB + kbyte);
      if (c == 0) hook();
      // lo, mid, hi of the FP32 operand against the BF16 fragment
#pragma unroll
      for (int q = 2; q >= 0; --q)
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            mfma_step<Elem::BF16, MI, 0>(af[AF ? q : 0][i], bf[AF ? 0 : q][j],
                                         acc[i][j]);
    }
  };
  if (nk > 0) {
    load(0, nfull > 0);
    store(0);
    if (nk > 1) load(1, 1 < nfull);
    __syncthreads();
    int kt = 0;
    for (; kt + 2 < nfull; ++kt) {
      compute(buf(kt), [&] {
        store(kt + 1);
        load(kt + 2, true);
      });
      __syncthreads();
    }
    for (; kt < nk; ++kt) {
      if (kt + 1 < nk) store(kt + 1);
      if (kt + 2 < nk) load(kt + 2, kt + 2 < nfull);
      __builtin_amdgcn_sched_barrier(0);
      compute(buf(kt), [] {});
      __syncthreads();
    }
  }
  store_tile_lds<Elem::BF16, Bf16Out, BM, BN, WM, WN, MI, LDS, false>(
      acc, C, p.ldc, p.M, p.N, m0, n0, (double)p.alpha, 0.0, threadIdx.x, lds,
      LA::edge_row(p.M), LA::edge_shift(p.M), LB::edge_row(p.N),
      LB::edge_shift(p.N));
}

template <bool AF, int BM, int BN, int WM, int WN>
hcblasStatus_t launch_mixed_cfg(hipStream_t s, MixedParams p, bool a_k,
                                bool b_k, int64_t batch) {
  p.tiles_m = (int)cdiv(p.M, BM);
  p.tiles_n = (int)cdiv(p.N, BN);
  const unsigned tiles = (unsigned)(p.tiles_m * p.tiles_n);
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
    MixedParams q = p;
    const int64_t nb = batch - b0 < 65535 ? batch - b0 : 65535;
    q.A = static_cast<const char *>(q.A) +
          b0 * q.strideA * (AF ? sizeof(float) : sizeof(uint16_t));
    q.B = static_cast<const char *>(q.B) +
          b0 * q.strideB * (AF ? sizeof(uint16_t) : sizeof(float));
    q.C = static_cast<Bf16Out *>(q.C) + b0 * q.strideC;
    dim3 grid(tiles, 1, (unsigned)nb);
#define HCB_MIXED(AK, BKC)                                      \
  if (a_k == AK && b_k == BKC)                                  \
    gemm_mixed_kernel<AF, AK, BKC, BM, BN, WM, WN>              \
        <<<grid, 64 * WM * WN, 0, s>>>(q);
    HCB_MIXED(false, false)
    HCB_MIXED(false, true)
    HCB_MIXED(true, false)
    HCB_MIXED(true, true)
#undef HCB_MIXED
    const hcblasStatus_t st = launch_status();
    if (st != HCBLAS_STATUS_SUCCESS) return st;
  }
  return HCBLAS_STATUS_SUCCESS;
}
// Tiles: 256 x 256 over 8 waves of 64 x 128 (FP32 operand along the wave
// tile's short side: 10 fragment reads per 24 MFMAs of a 16-k chunk, against
// 8 per 12 for 64 x 64 wave tiles), 128 x 128 over 4 waves of 64 x 64, 64 x 64
// over 2 waves of 32 x 64. Taken by the time on the CU with the most tiles,
// ceil(tiles / CUs) * area / rate (rates relative, from the times below; with
// 256 x 256 wherever both sides reach it a few large tiles ran on a few CUs):
//   dB of                          256   128   64 (us, tile edge)
//   256x 256 x 1024 x 512          245   313   464
//   100x 300 x 300 x 300            64    42    44
//   1x 1024 x 1024 x 1024           67    41    30
//   7x 900 x 900 x 900              66    51    71
//   16x 1000 x 700 x 900            76    89   110
//   33x 200 x 130 x 600             24    16    13
template <bool AF>
hcblasStatus_t launch_mixed(hipStream_t s, int num_cus, MixedParams p,
                            bool a_k, bool b_k, int64_t batch) {
  auto time = [&](int64_t t, int rate) {
    return cdiv(cdiv(p.M, t) * cdiv(p.N, t) * batch, num_cus) * t * t / rate;
  };
  const int64_t t256 = time(256, 125), t128 = time(128, 90), t64 = time(64, 48);
  if (t256 <= t128 && t256 <= t64) {
    if constexpr (AF)
      return launch_mixed_cfg<AF, 256, 256, 4, 2>(s, p, a_k, b_k, batch);
    else
      return launch_mixed_cfg<AF, 256, 256, 2, 4>(s, p, a_k, b_k, batch);
  }
  if (t128 <= t64)
    return launch_mixed_cfg<AF, 128, 128, 2, 2>(s, p, a_k, b_k, batch);
  if constexpr (AF)
    return launch_mixed_cfg<AF, 64, 64, 2, 1>(s, p, a_k, b_k, batch);
  else
    return launch_mixed_cfg<AF, 64, 64, 1, 2>(s, p, a_k, b_k, batch);
}

}  // namespace

hcblasStatus_t gemm_mixed_bf16(hcblasHandle_t h, const Canon &c, bool a_f32,
                               float alpha, void *C, int64_t ldc,
                               int64_t strideC, int64_t batch) {
  if (c.M == 0 || c.N == 0 || batch == 0) return HCBLAS_STATUS_SUCCESS;
  if (hipSetDevice(h->device) != hipSuccess)
    return HCBLAS_STATUS_EXECUTION_FAILED;
  MixedParams p{};
  p.M = c.M;
  p.N = c.N;
  p.K = c.K;
  p.A = static_cast<const char *>(c.A) + c.aOff * (a_f32 ? 4 : 2);
  p.lda = c.lda;
  p.strideA = c.strideA;
  p.B = static_cast<const char *>(c.B) + c.bOff * (a_f32 ? 2 : 4);
  p.ldb = c.ldb;
  p.strideB = c.strideB;
  p.C = C;
  p.ldc = ldc;
  p.strideC = strideC;
  p.alpha = alpha;
  return a_f32 ? launch_mixed<true>(h->stream, h->num_cus, p, c.a_k, c.b_k,
                                    batch)
               : launch_mixed<false>(h->stream, h->num_cus, p, c.a_k, c.b_k,
                                     batch);
}

}  // namespace hcb
