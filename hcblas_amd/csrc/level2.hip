// Level-2 BLAS on gfx950: {S,D}gemv and {S,D}ger, plain and batched.
//
// Reference kernels replaced (rocmarchive/hcBLAS):
//   gemv_TransA    lib/src/blas/sgemv/sgemv_array.cpp:30-147  (one WG / column)
//   gemv_NoTransA  lib/src/blas/sgemv/sgemv_array.cpp:520-563 (one thread / row)
//   gemv_alpha0_*  lib/src/blas/sgemv/sgemv_array.cpp:709-825
//   ger_HC         lib/src/blas/sger/sger_array.cpp:27-98     (one element / thread)
//
// Every matrix is handled as column-major STORAGE S (R contiguous rows, Cc
// columns, leading dimension ld). Row-major A is column-major A^T, so
//   col-major N, row-major T  ->  "panel" kernel:  y[r] = sum_c S[r,c] x[c]
//   col-major T, row-major N  ->  "column" kernel: y[c] = sum_r S[r,c] x[r]
// with a "band" variant of each for tall operands (a workgroup reads each
// column of its row band as one contiguous run; x or the band's sums stay in
// registers). All stream S once with 16-byte loads and split the reduction
// across workgroups when the output alone cannot fill 256 CUs; split partials
// go to a block of the handle's and a small finish kernel on the same stream
// sums them in a fixed order, so results are deterministic.
//
// GER updates S[r,c] = fma(v[r], alpha*w[c], S[r,c]) where w is the vector
// that indexes storage columns; with v = x, w = y for column-major and
// v = y, w = x for row-major this is bit-identical to CBLAS (netlib
// "temp = alpha*y(j); a(i,j) += x(i)*temp", row-major by argument swap).
#include <type_traits>
#include <utility>

#include "common.hpp"
#include "gemv_plan.hpp"

namespace hcb {
namespace {

constexpr int kThreads = 256;
static_assert(kThreads == kGemvThreads, "plan and kernels agree");

typedef float f4v __attribute__((ext_vector_type(4)));
typedef double d2v __attribute__((ext_vector_type(2)));

// 16 bytes of T. `type` for registers and the library's own buffers; `any` for
// the caller's operands, at any multiple of the element size: gfx950 serves a
// global_load / store_dwordx4 at any address, so an odd leading dimension,
// offset or row count does not leave the vector path.
template <typename T>
struct VecT;
template <>
struct VecT<float> {
  using type = f4v;
  typedef f4v any __attribute__((aligned(4)));
  static constexpr int n = 4;
};
template <>
struct VecT<double> {
  using type = d2v;
  typedef d2v any __attribute__((aligned(8)));
  static constexpr int n = 2;
};

template <typename T>
__device__ __forceinline__ T vlane(const typename VecT<T>::type &v, int i) {
  return v[i];
}

// 16-byte load, non-temporal when NT (operands far larger than the caches).
template <bool NT, typename T>
__device__ __forceinline__ typename VecT<T>::type vld(const T *p) {
  using A = typename VecT<T>::any;
  if constexpr (NT)
    return __builtin_nontemporal_load(reinterpret_cast<const A *>(p));
  else
    return *reinterpret_cast<const A *>(p);
}
template <bool NT, typename T>
__device__ __forceinline__ void vst(T *p, typename VecT<T>::type v) {
  using A = typename VecT<T>::any;
  if constexpr (NT)
    __builtin_nontemporal_store(v, reinterpret_cast<A *>(p));
  else
    *reinterpret_cast<A *>(p) = v;
}

// Operands at least this large (bytes) are streamed non-temporally.
constexpr int64_t kStreamBytes = 64ll << 20;

__device__ __forceinline__ int64_t bidx(int64_t i, int64_t n, int64_t inc) {
  return inc > 0 ? i * inc : (n - 1 - i) * (-inc);
}

template <typename T>
__device__ __forceinline__ T wave_sum(T v) {
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) v += __shfl_xor(v, off, 64);
  return v;
}

template <typename T>
__device__ __forceinline__ T fma_t(T a, T b, T c);
template <>
__device__ __forceinline__ float fma_t(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}
template <>
__device__ __forceinline__ double fma_t(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

struct GemvShape {
  int64_t R, Cc, ld;    // storage rows (contiguous), columns, leading dim
  int64_t incx, incy;   // BLAS increments of x (reduction) and y (output)
  int64_t sA, sx, sy;   // batch strides (elements)
  int splits;           // reduction split count (>= 1)
};

// Final value of one output element: y = alpha*sum + beta*y; beta == 0 does
// not read y (CBLAS: y need not be initialised).
template <typename T>
__device__ __forceinline__ void store_y(T *y, T sum, T alpha, T beta) {
  T r = alpha * sum;
  if (beta != T(0)) r = fma_t(beta, *y, r);
  *y = r;
}

// Split reductions: every workgroup stores its partial sums with plain
// stores to part[split][output], and gemv_finish_kernel, launched next on the
// same stream, adds them and writes y. A workgroup takes 64 outputs and its
// four waves every fourth split, eight loads in flight per thread; the order
// is fixed, so results are deterministic. (An in-kernel last-arriver reduction
// needs an agent-scope release per workgroup, which on a multi-XCD MI355X is
// an L2 write-back each: measured 5.1 against 6.4 TB/s for SGEMV-N 16384^2
// with 1024 workgroups.)
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_finish_kernel(
    int64_t len_y, int splits, const T *__restrict__ part, int64_t spart,
    T *y, int64_t incy, int64_t sy, T alpha, T beta) {
  __shared__ T red[4][64];
  const int64_t z = blockIdx.z;
  part += z * spart;
  y += z * sy;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  for (int64_t o0 = (int64_t)blockIdx.x * 64; o0 < len_y;
       o0 += (int64_t)gridDim.x * 64) {
    const int64_t o = o0 + lane < len_y ? o0 + lane : len_y - 1;
    T s[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) s[j] = T(0);
    int k = wave;
    for (; k + 28 < splits; k += 32) {
#pragma unroll
      for (int j = 0; j < 8; ++j)
        s[j] += part[(int64_t)(k + 4 * j) * len_y + o];
    }
#pragma unroll
    for (int j = 0; j < 7; ++j)
      if (k + 4 * j < splits) s[j] += part[(int64_t)(k + 4 * j) * len_y + o];
#pragma unroll
    for (int w = 4; w >= 1; w >>= 1)
#pragma unroll
      for (int j = 0; j < w; ++j) s[j] = s[j] + s[j + w];
    red[wave][lane] = s[0];
    __syncthreads();
    if (wave == 0 && o0 + lane < len_y)
      store_y(&y[bidx(o, len_y, incy)],
              (red[0][lane] + red[1][lane]) + (red[2][lane] + red[3][lane]),
              alpha, beta);
    __syncthreads();
  }
}

// ---------------------------------------------------------------------------
// Panel kernel: y[r] = alpha * sum_c S[r,c] x[c] + beta*y[r], for fewer rows
// than a band. Workgroup = NW waves over the same 64*VN rows (one 16-byte
// vector per lane); the waves interleave the workgroup's columns
// (c = c0 + wave + NW u) with U loads in flight per lane, and LDS sums the
// waves. blockIdx.y splits the columns across workgroups. Sixteen waves and no
// split serve small matrices in one launch. The last vector of a row count
// that is not a whole number of vectors is read from row R - VN on, and its
// lane stores only the rows that no other lane has.
// ---------------------------------------------------------------------------
template <typename T, bool VEC, bool NT, int NW>
__global__ __launch_bounds__(64 * NW) void gemv_panel_kernel(
    GemvShape s, const T *__restrict__ A, const T *__restrict__ x, T *y,
    T alpha, T beta, T *part) {
  constexpr int VN = VEC ? VecT<T>::n : 1;
  constexpr int ROWS = 64 * VN, TH = 64 * NW;
  constexpr int U = NW == 16 ? 16 : 8;
  __shared__ T red[NW][ROWS];
  const int64_t z = blockIdx.z;
  A += z * s.sA;
  x += z * s.sx;
  y += z * s.sy;
  // wave is uniform across the wave: readfirstlane lets the compiler fetch
  // x[c] with scalar loads instead of a vector load per A load.
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  const int64_t rb = (int64_t)blockIdx.x * ROWS;
  const int64_t r0 = rb + (int64_t)lane * VN;
  const int split = blockIdx.y;
  const int64_t cper = cdiv_dev(s.Cc, s.splits);
  const int64_t c_begin = split * cper;
  const int64_t c_end = c_begin + cper < s.Cc ? c_begin + cper : s.Cc;
  // Rows this lane reads: r0 .. or, at the edge, the last VN.
  const int64_t rr = r0 + VN <= s.R ? r0 : s.R - VN;

  T acc[VN];
#pragma unroll
  for (int e = 0; e < VN; ++e) acc[e] = T(0);

  if (r0 < s.R) {
    const T *col = A + rr;
    int64_t c = c_begin + wave;
    if constexpr (VEC) {
      using V = typename VecT<T>::type;
      // N of the wave's columns from c: all loads, then all FMAs. (A last
      // trip of U with the missing columns masked was slower: 9000 x 300 fp32
      // 9.3 us against 6.9.)
      auto columns = [&](auto n) {
        constexpr int N = decltype(n)::value;
        V a[N];
        T xv[N];
#pragma unroll
        for (int u = 0; u < N; ++u) {
          a[u] = vld<NT>(col + (c + NW * u) * s.ld);
          xv[u] = x[bidx(c + NW * u, s.Cc, s.incx)];
        }
#pragma unroll
        for (int u = 0; u < N; ++u)
#pragma unroll
          for (int e = 0; e < VN; ++e) acc[e] = fma_t(a[u][e], xv[u], acc[e]);
        c += NW * N;
      };
      while (c + NW * (U - 1) < c_end) columns(std::integral_constant<int, U>{});
      while (c + NW * 3 < c_end) columns(std::integral_constant<int, 4>{});
      while (c < c_end) columns(std::integral_constant<int, 1>{});
    } else {
      for (; c < c_end; c += NW)
        acc[0] = fma_t(col[c * s.ld], x[bidx(c, s.Cc, s.incx)], acc[0]);
    }
#pragma unroll
    for (int e = 0; e < VN; ++e)
      if (rr + e >= r0) red[wave][rr + e - rb] = acc[e];
  }
  __syncthreads();
  // Sum of the waves in wave order.
  T *pp = part + (z * s.splits + split) * s.R;
  for (int i = threadIdx.x; i < ROWS && rb + i < s.R; i += TH) {
    T v = red[0][i];
#pragma unroll
    for (int w = 1; w < NW; ++w) v += red[w][i];
    if (s.splits == 1)
      store_y(&y[bidx(rb + i, s.R, s.incy)], v, alpha, beta);
    else
      pp[rb + i] = v;
  }
}

// ---------------------------------------------------------------------------
// Band-N kernel: the panel kernel's job for operands of at least three
// quarters of a band of 256*VN rows. Workgroup = (one band of XR*256*VN rows,
// one block of columns): the band's sums stay in registers (XR vectors per
// thread) while the workgroup walks its columns UC at a time, each column's
// band being one contiguous run (XR * 4 KiB) read by all 256 threads; x[c] is
// wave-uniform (scalar loads). The loads of UC columns (32 per thread) are all
// issued before their FMAs (a scheduling barrier keeps the compiler from
// interleaving them one by one). Column blocks are sized so that bands x
// blocks is about one workgroup per CU with at least 32 columns per block, so
// the partials cost at most 2/32 of the traffic (XR = 4 bands of a large
// matrix: 2/256). Measured on MI355X at 16384^2: 155 us fp32 (6.9 TB/s) and
// 308 us fp64 against 166 / 315 us for the panel kernel. Lanes past the edge
// read the last VN rows; the rows no other lane has are stored.
// ---------------------------------------------------------------------------

template <typename T, int XR, bool NT>
__global__ __launch_bounds__(kThreads) void gemv_bandn_kernel(
    GemvShape s, const T *__restrict__ A, const T *__restrict__ x, T *y,
    T alpha, T beta, T *part) {
  using V = typename VecT<T>::type;
  constexpr int VN = VecT<T>::n;
  constexpr int UC = 32 / XR;
  constexpr int64_t STEP = (int64_t)kThreads * VN;
  const int64_t z = blockIdx.z;
  A += z * s.sA;
  x += z * s.sx;
  y += z * s.sy;
  // blockIdx.x walks the column blocks and blockIdx.y the bands: consecutive
  // workgroups (spread over the XCDs in turn) then share a band (measured
  // 155 against 164 us at 16384^2 fp32 with the axes swapped).
  const int64_t rt = (int64_t)blockIdx.y * XR * STEP +
                     (int64_t)threadIdx.x * VN;
  int64_t roff[XR];
#pragma unroll
  for (int u = 0; u < XR; ++u) {
    const int64_t r = rt + u * STEP;
    roff[u] = r + VN <= s.R ? r : s.R - VN;
  }
  const int split = blockIdx.x;
  const int64_t cper = cdiv_dev(s.Cc, s.splits);
  const int64_t c_begin = split * cper;
  const int64_t c_end = c_begin + cper < s.Cc ? c_begin + cper : s.Cc;
  T acc[XR][VN];
#pragma unroll
  for (int u = 0; u < XR; ++u)
#pragma unroll
    for (int e = 0; e < VN; ++e) acc[u][e] = T(0);
  int64_t c = c_begin;
  // N columns from c: all loads, then all FMAs.
  auto columns = [&](auto n) {
    constexpr int N = decltype(n)::value;
    V a[N][XR];
    T xv[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      xv[j] = x[bidx(c + j, s.Cc, s.incx)];
      const T *col = A + (c + j) * s.ld;
#pragma unroll
      for (int u = 0; u < XR; ++u) a[j][u] = vld<NT>(col + roff[u]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < N; ++j)
#pragma unroll
      for (int u = 0; u < XR; ++u)
#pragma unroll
        for (int e = 0; e < VN; ++e)
          acc[u][e] = fma_t(vlane<T>(a[j][u], e), xv[j], acc[u][e]);
    c += N;
  };
  while (c + UC <= c_end) columns(std::integral_constant<int, UC>{});
  while (c + 4 <= c_end) columns(std::integral_constant<int, 4>{});
  while (c < c_end) columns(std::integral_constant<int, 1>{});
#pragma unroll
  for (int u = 0; u < XR; ++u) {
    const int64_t r = rt + u * STEP;
    if (r >= s.R) continue;
    T *pp = part + (z * s.splits + split) * s.R;
    if (s.splits > 1 && r + VN <= s.R) {
      V v;
#pragma unroll
      for (int e = 0; e < VN; ++e) v[e] = acc[u][e];
      vst<false>(pp + r, v);
      continue;
    }
#pragma unroll
    for (int e = 0; e < VN; ++e) {
      const int64_t re = roff[u] + e;
      if (re < r) continue;
      if (s.splits == 1)
        store_y(&y[bidx(re, s.R, s.incy)], acc[u][e], alpha, beta);
      else
        pp[re] = acc[u][e];
    }
  }
}

// ---------------------------------------------------------------------------
// Column kernel: y[c] = alpha * sum_r S[r,c] x[r] + beta*y[c].
// Workgroup = 4 waves x CPW columns; each wave reduces CPW columns over its
// row range with 16-byte loads, reusing each x load for the CPW columns.
// blockIdx.y selects a contiguous range of rows (split).
// ---------------------------------------------------------------------------

template <typename T, bool VEC, bool NT>
__global__ __launch_bounds__(kThreads) void gemv_column_kernel(
    GemvShape s, const T *__restrict__ A, const T *__restrict__ x, T *y,
    T alpha, T beta, T *part) {
  constexpr int VN = VEC ? VecT<T>::n : 1;
  const int64_t z = blockIdx.z;
  A += z * s.sA;
  x += z * s.sx;
  y += z * s.sy;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane_id = threadIdx.x & 63;
  const int64_t cbase = (int64_t)blockIdx.x * kColsPerBlock + wave * kCPW;
  const int split = blockIdx.y;
  // Row range of this split, a multiple of the 64*VN step.
  const int64_t step = 64 * VN;
  const int64_t rsteps = cdiv_dev(s.R, step);
  const int64_t sper = cdiv_dev(rsteps, s.splits);
  const int64_t r_begin = split * sper * step;
  int64_t r_end = r_begin + sper * step;
  if (r_end > s.R) r_end = s.R;

  T acc[kCPW][VN];
#pragma unroll
  for (int j = 0; j < kCPW; ++j)
#pragma unroll
    for (int e = 0; e < VN; ++e) acc[j][e] = T(0);

  const T *cols[kCPW];
  bool colok[kCPW];
#pragma unroll
  for (int j = 0; j < kCPW; ++j) {
    colok[j] = cbase + j < s.Cc;
    cols[j] = A + (colok[j] ? (cbase + j) : 0) * s.ld;
  }

  if constexpr (VEC) {
    using V = typename VecT<T>::type;
    const bool xunit = s.incx == 1;
    int64_t r = r_begin + lane_id * VN;
    if (xunit) {
      // Two row steps per iteration: 2 * kCPW loads of A in flight per lane.
      for (; r + step + VN <= r_end; r += 2 * step) {
        const V t0 = vld<false>(x + r);
        const V t1 = vld<false>(x + r + step);
        V a0[kCPW], a1[kCPW];
#pragma unroll
        for (int j = 0; j < kCPW; ++j) {
          a0[j] = vld<NT>(cols[j] + r);
          a1[j] = vld<NT>(cols[j] + r + step);
        }
#pragma unroll
        for (int j = 0; j < kCPW; ++j) {
          if (!colok[j]) continue;
#pragma unroll
          for (int e = 0; e < VN; ++e)
            acc[j][e] = fma_t(vlane<T>(a0[j], e), vlane<T>(t0, e), acc[j][e]);
#pragma unroll
          for (int e = 0; e < VN; ++e)
            acc[j][e] = fma_t(vlane<T>(a1[j], e), vlane<T>(t1, e), acc[j][e]);
        }
      }
    }
    for (; r < r_end; r += step) {
      // A vector that reaches past R is read from R - VN on; the rows below r
      // belong to another lane and count as zeros here.
      const int64_t rr = r + VN <= s.R ? r : s.R - VN;
      T xv[VN];
      V a[kCPW];
#pragma unroll
      for (int j = 0; j < kCPW; ++j) a[j] = vld<NT>(cols[j] + rr);
#pragma unroll
      for (int e = 0; e < VN; ++e) xv[e] = x[bidx(rr + e, s.R, s.incx)];
#pragma unroll
      for (int e = 0; e < VN; ++e) xv[e] = rr + e >= r ? xv[e] : T(0);
#pragma unroll
      for (int j = 0; j < kCPW; ++j)
#pragma unroll
        for (int e = 0; e < VN; ++e)
          acc[j][e] = fma_t(rr + e >= r ? vlane<T>(a[j], e) : T(0), xv[e],
                            acc[j][e]);
    }
  } else {
    for (int64_t r = r_begin + lane_id; r < r_end; r += step) {
      const T xv = x[bidx(r, s.R, s.incx)];
      T a[kCPW];
#pragma unroll
      for (int j = 0; j < kCPW; ++j) a[j] = cols[j][r];
#pragma unroll
      for (int j = 0; j < kCPW; ++j) acc[j][0] = fma_t(a[j], xv, acc[j][0]);
    }
  }

  T sums[kCPW];
#pragma unroll
  for (int j = 0; j < kCPW; ++j) {
    T t = T(0);
#pragma unroll
    for (int e = 0; e < VN; ++e) t += acc[j][e];
    sums[j] = wave_sum(t);
  }

  if (s.splits == 1) {
    if (lane_id == 0) {
#pragma unroll
      for (int j = 0; j < kCPW; ++j)
        if (colok[j])
          store_y(&y[bidx(cbase + j, s.Cc, s.incy)], sums[j], alpha, beta);
    }
    return;
  }
  if (lane_id == 0) {
    T *pp = part + (z * s.splits + split) * s.Cc;
#pragma unroll
    for (int j = 0; j < kCPW; ++j)
      if (colok[j]) pp[cbase + j] = sums[j];
  }
}

// ---------------------------------------------------------------------------
// Band kernel: the column kernel's job for operands of at least three
// quarters of a row step of 256*VN. Workgroup = (CPB consecutive columns, one
// band of XR row steps). The band's x is loaded once into registers (thread t
// keeps the vectors at rows t*VN + u*256*VN, u < XR) and each column is then
// one contiguous run of the band read by all 256 threads, with no x traffic
// and at least 16 loads per thread in flight (short bands read several
// columns together). A column's sum crosses the wave by shuffles while the next
// columns load, and the four waves are added at the end in order. Measured on MI355X at 16384^2:
// 6.9 TB/s fp32 and 7.0 TB/s fp64, against 6.2 / 6.5 for the column kernel,
// whose four columns per wave and per-step x loads cost bandwidth.
// ---------------------------------------------------------------------------

template <typename T, int XR, bool NT>
__global__ __launch_bounds__(kThreads) void gemv_band_kernel(
    GemvShape s, const T *__restrict__ A, const T *__restrict__ x, T *y,
    T alpha, T beta, T *part) {
  using V = typename VecT<T>::type;
  constexpr int VN = VecT<T>::n;
  constexpr int CPB = kBandCols;
  // Columns read together: at least 16 vectors in flight per thread.
  constexpr int CG = XR >= 12 ? 1 : XR >= 6 ? 2 : XR >= 3 ? 4 : 8;
  constexpr int64_t STEP = (int64_t)kThreads * VN;
  __shared__ T red[4][CPB];
  const int64_t z = blockIdx.z;
  A += z * s.sA;
  x += z * s.sx;
  y += z * s.sy;
  const int split = blockIdx.y;
  const int64_t r_begin = (int64_t)split * XR * STEP;
  const int64_t rt = r_begin + (int64_t)threadIdx.x * VN;
  const bool full = r_begin + XR * STEP <= s.R;
  // Lanes past the edge read the last VN rows; rows that another lane (or
  // none) has count as zeros, in x and in A.
  auto row = [&](int u) {
    const int64_t r = rt + u * STEP;
    return full || r + VN <= s.R ? r : s.R - VN;
  };
  V xr[XR];
#pragma unroll
  for (int u = 0; u < XR; ++u) {
    const int64_t rr = row(u);
    if (s.incx == 1) {
      xr[u] = vld<false>(x + rr);
    } else {
#pragma unroll
      for (int e = 0; e < VN; ++e) xr[u][e] = x[bidx(rr + e, s.R, s.incx)];
    }
    if (!full) {
#pragma unroll
      for (int e = 0; e < VN; ++e)
        if (rr + e < rt + u * STEP) xr[u][e] = T(0);
    }
  }
  const int64_t c0 = (int64_t)blockIdx.x * CPB;
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  V a[CG][XR];
  auto load = [&](int j0) {
#pragma unroll
    for (int j = 0; j < CG; ++j) {
      // (columns past the last read the last one; their sums are dropped)
      const int64_t c = c0 + j0 + j < s.Cc ? c0 + j0 + j : s.Cc - 1;
      const T *col = A + c * s.ld;
#pragma unroll
      for (int u = 0; u < XR; ++u) a[j][u] = vld<NT>(col + row(u));
    }
  };
  load(0);
  // A rolled loop: one group's vectors in registers, the next group's loads in
  // flight while this group's sums cross the wave.
#pragma unroll 1
  for (int j0 = 0; j0 < CPB; j0 += CG) {
    T t[CG];
#pragma unroll
    for (int j = 0; j < CG; ++j) {
      if (!full) {
#pragma unroll
        for (int u = 0; u < XR; ++u)
#pragma unroll
          for (int e = 0; e < VN; ++e)
            if (row(u) + e < rt + u * STEP) a[j][u][e] = T(0);
      }
      T acc[VN];
#pragma unroll
      for (int e = 0; e < VN; ++e) acc[e] = T(0);
#pragma unroll
      for (int u = 0; u < XR; ++u)
#pragma unroll
        for (int e = 0; e < VN; ++e)
          acc[e] = fma_t(vlane<T>(a[j][u], e), vlane<T>(xr[u], e), acc[e]);
      t[j] = T(0);
#pragma unroll
      for (int e = 0; e < VN; ++e) t[j] += acc[e];
    }
    if (j0 + CG < CPB) load(j0 + CG);
#pragma unroll
    for (int j = 0; j < CG; ++j) {
      const T v = wave_sum(t[j]);
      if (lane == 0) red[wave][j0 + j] = v;
    }
  }
  __syncthreads();
  if (threadIdx.x >= CPB) return;
  const int j = threadIdx.x;
  const int64_t c = c0 + j;
  if (c >= s.Cc) return;
  const T v = ((red[0][j] + red[1][j]) + red[2][j]) + red[3][j];
  if (s.splits == 1)
    store_y(&y[bidx(c, s.Cc, s.incy)], v, alpha, beta);
  else
    part[(z * s.splits + split) * s.Cc + c] = v;
}

// alpha == 0 (or an empty reduction): y = beta*y without reading A or x
// (reference gemv_alpha0_col, sgemv_array.cpp:709-734).
template <typename T>
__global__ __launch_bounds__(kThreads) void gemv_scale_y_kernel(
    int64_t len, int64_t incy, int64_t sy, T *y, T beta) {
  y += (int64_t)blockIdx.z * sy;
  for (int64_t i = (int64_t)blockIdx.x * kThreads + threadIdx.x; i < len;
       i += (int64_t)gridDim.x * kThreads) {
    T *p = &y[bidx(i, len, incy)];
    *p = beta == T(0) ? T(0) : beta * *p;
  }
}

// ---------------------------------------------------------------------------
// GER: D[r,c] = fma(v[r], alpha*w[c], S[r,c]), in place (D = S) or into another
// matrix; alpha == 0 copies. HBM bound: one read of S, one write of D. Each
// thread owns VN consecutive rows (one 16-byte vector) and walks kGerCols
// columns, so v stays in registers and every store is a full 16-byte store.
// (The differentiable update copied S first and updated the copy in place, two
// reads and two writes: 4096^2 fp32 copy 26 us and update 22; now one launch of
// 22, 5.9 TB/s.)
// ---------------------------------------------------------------------------
constexpr int kGerCols = 16;

template <typename T, bool VEC, bool NT, bool ADD>
__global__ __launch_bounds__(kThreads) void ger_kernel(
    int64_t R, int64_t Cc, const T *S, int64_t lds, T *D, int64_t ldd,
    int64_t sA, const T *__restrict__ v, int64_t incv, int64_t sv,
    const T *__restrict__ w, int64_t incw, int64_t sw, T alpha) {
  constexpr int VN = VEC ? VecT<T>::n : 1;
  using V = typename std::conditional<VEC, typename VecT<T>::type, T>::type;
  const int64_t z = blockIdx.z;
  S += z * sA;
  D += z * sA;
  v += z * sv;
  w += z * sw;
  const int64_t r0 = ((int64_t)blockIdx.x * kThreads + threadIdx.x) * VN;
  if (r0 >= R) return;
  const int64_t c0 = (int64_t)blockIdx.y * kGerCols;
  const int64_t cend = c0 + kGerCols < Cc ? c0 + kGerCols : Cc;
  // The last rows, if they are no whole vector, are read from row R - VN on; of
  // that vector only they are stored (the others are another lane's).
  const int64_t rr = r0 + VN <= R ? r0 : R - VN;
  // Every load is issued before the first store, so kGerCols loads are in
  // flight per lane (the stores would otherwise order each next load behind
  // them: the compiler cannot prove the columns disjoint). Columns past the
  // last read it again and are not stored. (Edge rows and columns one load and
  // store after another: SGER 179 x 125 9.9 us, now 3.8; 1904 x 26 8.5, 3.6.)
  auto columns = [&](auto whole) {
    constexpr bool W = decltype(whole)::value;
    auto col = [&](int j) { return W || c0 + j < cend ? c0 + j : cend - 1; };
    V a[kGerCols];
    T vr[VN];
#pragma unroll
    for (int j = 0; j < kGerCols; ++j) {
      if constexpr (VEC)
        a[j] = vld<NT>(S + rr + col(j) * lds);
      else
        a[j] = S[rr + col(j) * lds];
    }
    if constexpr (ADD) {
#pragma unroll
      for (int e = 0; e < VN; ++e) vr[e] = v[bidx(rr + e, R, incv)];
    }
    auto update = [&](int j, T wj) {
      if constexpr (ADD) {
        const T t = alpha * wj;
        if constexpr (VEC) {
#pragma unroll
          for (int e = 0; e < VN; ++e) a[j][e] = fma_t(vr[e], t, a[j][e]);
        } else {
          a[j] = fma_t(vr[0], t, a[j]);
        }
      }
    };
    auto wcol = [&](int j) { return ADD ? w[bidx(col(j), Cc, incw)] : T(0); };
    if (W && rr == r0) {
#pragma unroll
      for (int j = 0; j < kGerCols; ++j) {
        update(j, wcol(j));
        if constexpr (VEC)
          vst<NT>(D + rr + (c0 + j) * ldd, a[j]);
        else
          D[rr + (c0 + j) * ldd] = a[j];
      }
      return;
    }
    T wv[kGerCols];
#pragma unroll
    for (int j = 0; j < kGerCols; ++j) wv[j] = wcol(j);
#pragma unroll
    for (int j = 0; j < kGerCols; ++j) update(j, wv[j]);
    if (rr == r0) {
#pragma unroll
      for (int j = 0; j < kGerCols; ++j) {
        if (c0 + j >= cend) break;
        if constexpr (VEC)
          vst<NT>(D + rr + (c0 + j) * ldd, a[j]);
        else
          D[rr + (c0 + j) * ldd] = a[j];
      }
    } else if constexpr (VEC) {
#pragma unroll
      for (int e = 1; e < VN; ++e) {
        if (rr + e < r0) continue;
#pragma unroll
        for (int j = 0; j < kGerCols; ++j) {
          if (!W && c0 + j >= cend) break;
          D[rr + e + (c0 + j) * ldd] = a[j][e];
        }
      }
    }
  };
  if (cend - c0 == kGerCols)
    columns(std::true_type{});
  else
    columns(std::false_type{});
}

// ---------------------------------------------------------------------------
// GEMV pair: both products of one matrix in one pass over it,
//   yr[r] = alpha * sum_c S[r,c] q[c]   and   yc[c] = alpha * sum_r S[r,c] p[r]
// (the adjoint of GER). HBM bound, and S is read once instead of twice. A
// workgroup owns a band of XR row steps and a block of columns, as in the
// band-N kernel: the band's p and its row sums stay in registers; 32 vectors
// per thread are in flight, all issued before their FMAs. A column's sum over
// the band crosses the wave by shuffles into LDS. Both results leave as
// partials (rows: one per column block, columns: one per band), except the
// column sums of a single band.
// ---------------------------------------------------------------------------
constexpr int kPairCols = 512;  // columns of a block at most

template <typename T, int XR, bool NT>
__global__ __launch_bounds__(kThreads) void gemv_pair_kernel(
    int64_t R, int64_t Cc, int64_t ld, const T *__restrict__ S,
    const T *__restrict__ p, int64_t incp, const T *__restrict__ q,
    int64_t incq, T alpha, T *yc, T *row_part, T *col_part) {
  using V = typename VecT<T>::type;
  constexpr int VN = VecT<T>::n;
  constexpr int UC = 32 / XR;
  constexpr int64_t STEP = (int64_t)kThreads * VN;
  __shared__ T red[4][kPairCols];
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int64_t rt = (int64_t)blockIdx.y * XR * STEP +
                     (int64_t)threadIdx.x * VN;
  const bool full = ((int64_t)blockIdx.y + 1) * XR * STEP <= R;
  // Lanes past the edge read the last VN rows; rows below their own belong to
  // another lane: they count as zeros in the column sums (in p and in S), and
  // their row sums are not stored.
  int64_t roff[XR];
  V pv[XR];
#pragma unroll
  for (int u = 0; u < XR; ++u) {
    const int64_t r = rt + u * STEP;
    roff[u] = r + VN <= R ? r : R - VN;
#pragma unroll
    for (int e = 0; e < VN; ++e)
      pv[u][e] = roff[u] + e >= r ? p[bidx(roff[u] + e, R, incp)] : T(0);
  }
  const int64_t cper = cdiv_dev(Cc, (int64_t)gridDim.x);
  const int64_t c_begin = (int64_t)blockIdx.x * cper;
  const int64_t c_end = c_begin + cper < Cc ? c_begin + cper : Cc;
  T acc[XR][VN];
#pragma unroll
  for (int u = 0; u < XR; ++u)
#pragma unroll
    for (int e = 0; e < VN; ++e) acc[u][e] = T(0);
  int64_t c = c_begin;
  // N columns from c: all loads, then all FMAs.
  auto columns = [&](auto n) {
    constexpr int N = decltype(n)::value;
    V a[N][XR];
    T qv[N], sum[N];
#pragma unroll
    for (int j = 0; j < N; ++j) {
      qv[j] = q[bidx(c + j, Cc, incq)];
      const T *col = S + (c + j) * ld;
#pragma unroll
      for (int u = 0; u < XR; ++u) a[j][u] = vld<NT>(col + roff[u]);
    }
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int j = 0; j < N; ++j) {
      T t[VN];
#pragma unroll
      for (int e = 0; e < VN; ++e) t[e] = T(0);
#pragma unroll
      for (int u = 0; u < XR; ++u)
#pragma unroll
        for (int e = 0; e < VN; ++e) {
          const T x = vlane<T>(a[j][u], e);
          acc[u][e] = fma_t(x, qv[j], acc[u][e]);
          const bool own = full || roff[u] + e >= rt + u * STEP;
          t[e] = fma_t(own ? x : T(0), vlane<T>(pv[u], e), t[e]);
        }
      sum[j] = t[0];
#pragma unroll
      for (int e = 1; e < VN; ++e) sum[j] += t[e];
    }
    // The N column sums cross the wave together: each halving of the lanes
    // also halves the columns a lane holds (N = 16: 17 shuffles, not 96).
    int width = 32;
#pragma unroll
    for (int h = N / 2; h >= 1; h /= 2, width /= 2)
#pragma unroll
      for (int i = 0; i < h; ++i) {
        const bool up = lane & width;
        const T give = up ? sum[i] : sum[i + h];
        sum[i] = (up ? sum[i + h] : sum[i]) + __shfl_xor(give, width, 64);
      }
#pragma unroll
    for (; width >= 1; width /= 2) sum[0] += __shfl_xor(sum[0], width, 64);
    constexpr int LPC = 64 / N;  // lanes that hold a column's sum
    if (lane % LPC == 0) red[wave][c - c_begin + lane / LPC] = sum[0];
    c += N;
  };
  while (c + UC <= c_end) columns(std::integral_constant<int, UC>{});
  while (c + 4 <= c_end) columns(std::integral_constant<int, 4>{});
  while (c < c_end) columns(std::integral_constant<int, 1>{});
  T *rp = row_part + (int64_t)blockIdx.x * R;
#pragma unroll
  for (int u = 0; u < XR; ++u) {
    const int64_t r = rt + u * STEP;
    if (r >= R) continue;
#pragma unroll
    for (int e = 0; e < VN; ++e)
      if (roff[u] + e >= r) rp[roff[u] + e] = acc[u][e];
  }
  __syncthreads();
  for (int j = threadIdx.x; j < (int)(c_end - c_begin); j += kThreads) {
    const T v = ((red[0][j] + red[1][j]) + red[2][j]) + red[3][j];
    if (gridDim.y == 1)
      yc[c_begin + j] = alpha * v;
    else
      col_part[(int64_t)blockIdx.y * Cc + c_begin + j] = v;
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
template <typename T, int NW>
void launch_panel(dim3 grid, hipStream_t stream, bool vec, bool nt,
                  const GemvShape &s, const T *A, const T *x, T *y, T alpha,
                  T beta, T *part) {
  (!vec ? gemv_panel_kernel<T, false, false, NW>
   : nt ? gemv_panel_kernel<T, true, true, NW>
        : gemv_panel_kernel<T, true, false, NW>)
      <<<grid, 64 * NW, 0, stream>>>(s, A, x, y, alpha, beta, part);
}

template <typename T>
hcblasStatus_t run_gemv(hcblasHandle_t h, bool panel, int64_t R, int64_t Cc,
                        T alpha, const T *A, int64_t ld, const T *x,
                        int64_t incx, T beta, T *y, int64_t incy, int64_t sA,
                        int64_t sx, int64_t sy, int64_t batch,
                        void *fixed_part = nullptr, size_t fixed_bytes = 0) {
  const int64_t len_y = panel ? R : Cc;
  const int64_t len_x = panel ? Cc : R;
  if (len_y == 0 || batch == 0) return HCBLAS_STATUS_SUCCESS;
  if (alpha == T(0) || len_x == 0) {
    if (beta == T(1)) return HCBLAS_STATUS_SUCCESS;
    dim3 g((unsigned)std::min<int64_t>(cdiv(len_y, kThreads), 4096), 1,
           (unsigned)batch);
    gemv_scale_y_kernel<T><<<g, kThreads, 0, h->stream>>>(len_y, incy, sy, y,
                                                          beta);
    return launch_status();
  }
  constexpr int VN = VecT<T>::n;
  // Rows are read 16 bytes at a time unless there is not even one vector, or, in
  // the column kernel, one element for each lane of a wave reaches them all
  // (SGEMV-T 37 x 576 3.9 us by vectors, 3.0).
  bool vec = panel ? R >= VN : R > 64;
  const bool nt = (int64_t)sizeof(T) * R * Cc * batch >= kStreamBytes;
  GemvShape s{R, Cc, ld, incx, incy, sA, sx, sy, 1};
  GemvPlan plan =
      plan_gemv(h->num_cus, panel, R, Cc, vec, VN, sizeof(T), batch);
  // Bands of a column-contiguous matrix can need more partials than the
  // allocation-free entry's scratch holds from about 68 GB on (FP64 8193 x
  // 1048577: 16 bytes more; FP32 from twice that). Where the operands are not
  // 16-byte aligned both entries then read by elements, whose splits fit.
  if (batch == 1 && plan.partial_bytes > kNoAllocScratchBytes &&
      (!aligned16(A) || ld % VN || R % VN ||
       (!panel && incx == 1 && !aligned16(x)))) {
    vec = false;
    plan = plan_gemv(h->num_cus, panel, R, Cc, vec, VN, sizeof(T), batch);
  }
  s.splits = plan.splits;
  T *part = nullptr;
  if (s.splits > 1) {
    if (fixed_part) {
      // Allocation-free entry: the same split (so the same summation order
      // and results as the workspace path) or an error, never fewer splits.
      if (plan.partial_bytes > fixed_bytes) return HCBLAS_STATUS_INVALID_VALUE;
      part = static_cast<T *>(fixed_part);
    } else {
      part = static_cast<T *>(partials(h, plan.partial_bytes));
      if (part == nullptr) {
        plan = plan_gemv(h->num_cus, panel, R, Cc, vec, VN, sizeof(T), batch,
                         false);
        s.splits = 1;
      }
    }
  }
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
    int64_t nb = std::min<int64_t>(65535, batch - b0);
    dim3 grid((unsigned)plan.oblocks, (unsigned)s.splits, (unsigned)nb);
    if (plan.kernel == GemvKernel::kBandN) std::swap(grid.x, grid.y);
    const T *Ab = A + b0 * sA;
    const T *xb = x + b0 * sx;
    T *yb = y + b0 * sy;
#define HCB_GEMV(KERNEL, TH, ...)                                          \
  (nt ? KERNEL<T, __VA_ARGS__, true> : KERNEL<T, __VA_ARGS__, false>)      \
      <<<grid, TH, 0, h->stream>>>(s, Ab, xb, yb, alpha, beta, part)
#define HCB_BAND(XR)                                                       \
  case XR:                                                                 \
    HCB_GEMV(gemv_band_kernel, kThreads, XR);                              \
    break
    switch (plan.kernel) {
      case GemvKernel::kBandN:
        if (plan.xr == 4)
          HCB_GEMV(gemv_bandn_kernel, kThreads, 4);
        else if (plan.xr == 2)
          HCB_GEMV(gemv_bandn_kernel, kThreads, 2);
        else
          HCB_GEMV(gemv_bandn_kernel, kThreads, 1);
        break;
      case GemvKernel::kPanel:
        if (plan.waves == 16)
          launch_panel<T, 16>(grid, h->stream, vec, nt, s, Ab, xb, yb, alpha,
                              beta, part);
        else
          launch_panel<T, 4>(grid, h->stream, vec, nt, s, Ab, xb, yb, alpha,
                             beta, part);
        break;
      case GemvKernel::kBand16:
      case GemvKernel::kBand8:
        switch (plan.xr) {
          HCB_BAND(1);
          HCB_BAND(2);
          HCB_BAND(3);
          HCB_BAND(4);
          HCB_BAND(6);
          HCB_BAND(8);
          HCB_BAND(10);
          HCB_BAND(12);
          HCB_BAND(14);
          HCB_BAND(16);
          default:
            return HCBLAS_STATUS_INTERNAL_ERROR;
        }
        break;
      case GemvKernel::kColumn:
        if (!vec)
          gemv_column_kernel<T, false, false><<<grid, kThreads, 0, h->stream>>>(
              s, Ab, xb, yb, alpha, beta, part);
        else
          HCB_GEMV(gemv_column_kernel, kThreads, true);
        break;
    }
#undef HCB_BAND
#undef HCB_GEMV
    if (s.splits > 1) {
      dim3 fg((unsigned)std::min<int64_t>(cdiv(len_y, 64), 4096), 1,
              (unsigned)nb);
      gemv_finish_kernel<T><<<fg, kThreads, 0, h->stream>>>(
          len_y, s.splits, part, (int64_t)s.splits * len_y, yb, incy, sy,
          alpha, beta);
    }
    hcblasStatus_t st = launch_status();
    if (st != HCBLAS_STATUS_SUCCESS) return st;
  }
  return HCBLAS_STATUS_SUCCESS;
}

// Common argument handling for gemv in the reference's (order, trans) terms.
template <typename T>
hcblasStatus_t gemv_entry(hcblasHandle_t h, hcblasOrder_t order,
                          hcblasOperation_t trans, int M, int N,
                          const T *alpha, const T *A, int64_t aOffset,
                          int64_t lda, const T *x, int64_t xOffset,
                          int64_t incx, const T *beta, T *y, int64_t yOffset,
                          int64_t incy, int64_t batch, bool ref_batch_strides,
                          int64_t sA_in = 0, int64_t sx_in = 0,
                          int64_t sy_in = 0, bool noalloc = false) {
  if (!handle_ok(h)) return HCBLAS_STATUS_NOT_INITIALIZED;
  if (M < 0 || N < 0 || incx == 0 || incy == 0 || batch < 0)
    return HCBLAS_STATUS_INVALID_VALUE;
  if (order != HCBLAS_ROW_MAJOR && order != HCBLAS_COL_MAJOR)
    return HCBLAS_STATUS_INVALID_VALUE;
  if (canon_op(trans) < 0) return HCBLAS_STATUS_INVALID_VALUE;
  const bool notrans = canon_op(trans) == HCBLAS_OP_N;
  const int64_t len_x = notrans ? N : M, len_y = notrans ? M : N;
  // Storage is column-major R x Cc.
  const bool col = order == HCBLAS_COL_MAJOR;
  const int64_t R = col ? M : N, Cc = col ? N : M;
  if (lda < std::max<int64_t>(1, R)) return HCBLAS_STATUS_INVALID_VALUE;
  if (M == 0 || N == 0 || batch == 0) {
    if (len_y == 0 || batch == 0) return HCBLAS_STATUS_SUCCESS;
  }
  if (alpha == nullptr || beta == nullptr || y == nullptr)
    return HCBLAS_STATUS_INVALID_VALUE;
  if (*alpha != T(0) && len_x > 0 && (A == nullptr || x == nullptr))
    return HCBLAS_STATUS_INVALID_VALUE;
  // Batch strides as in hcblas.cpp:1008-1019 (x by len(x), y by len(y), A by
  // M*N), or the caller's explicit batch offsets.
  int64_t sA = ref_batch_strides ? (int64_t)M * N : sA_in;
  int64_t sx = ref_batch_strides ? len_x : sx_in;
  int64_t sy = ref_batch_strides ? len_y : sy_in;
  const bool panel = col == notrans;
  return run_gemv<T>(h, panel, R, Cc, *alpha, A ? A + aOffset : nullptr, lda,
                     x ? x + xOffset : nullptr, incx, *beta, y + yOffset, incy,
                     sA, sx, sy, batch, noalloc ? h->noalloc_scratch : nullptr,
                     noalloc ? kNoAllocScratchBytes : 0);
}

template <typename T>
hcblasStatus_t ger_entry(hcblasHandle_t h, hcblasOrder_t order, int M, int N,
                         const T *alpha, const T *x, int64_t xOffset,
                         int64_t incx, const T *y, int64_t yOffset,
                         int64_t incy, T *A, int64_t aOffset, int64_t lda,
                         int64_t batch, bool ref_batch_strides = true,
                         int64_t sA_in = 0, int64_t sx_in = 0,
                         int64_t sy_in = 0, const T *src = nullptr,
                         int64_t lds = 0) {
  if (!handle_ok(h)) return HCBLAS_STATUS_NOT_INITIALIZED;
  if (M < 0 || N < 0 || incx == 0 || incy == 0 || batch < 0)
    return HCBLAS_STATUS_INVALID_VALUE;
  if (order != HCBLAS_ROW_MAJOR && order != HCBLAS_COL_MAJOR)
    return HCBLAS_STATUS_INVALID_VALUE;
  const bool col = order == HCBLAS_COL_MAJOR;
  const int64_t R = col ? M : N, Cc = col ? N : M;
  if (lda < std::max<int64_t>(1, R)) return HCBLAS_STATUS_INVALID_VALUE;
  if (M == 0 || N == 0 || batch == 0) return HCBLAS_STATUS_SUCCESS;
  if (alpha == nullptr || x == nullptr || y == nullptr || A == nullptr)
    return HCBLAS_STATUS_INVALID_VALUE;
  if (src == nullptr) {
    if (*alpha == T(0)) return HCBLAS_STATUS_SUCCESS;  // netlib quick return
    src = A + aOffset;
    lds = lda;
  }
  // Batch strides as in hcblas.cpp:1160-1167 (x by M, y by N, A by M*N), or
  // the caller's explicit batch offsets.
  const bool multi = batch > 1;
  const int64_t sA = !multi ? 0 : ref_batch_strides ? (int64_t)M * N : sA_in;
  const int64_t sxv = !multi ? 0 : ref_batch_strides ? M : sx_in;
  const int64_t syv = !multi ? 0 : ref_batch_strides ? N : sy_in;
  const T *v = col ? x + xOffset : y + yOffset;
  const T *w = col ? y + yOffset : x + xOffset;
  const int64_t incv = col ? incx : incy, incw = col ? incy : incx;
  const int64_t sv = col ? sxv : syv, sw = col ? syv : sxv;
  T *Ab = A + aOffset;
  constexpr int VN = VecT<T>::n;
  const bool vec = R >= VN;
  const int64_t rows_per_block = (int64_t)kThreads * (vec ? VN : 1);
  // A matrix larger than the 256 MB last-level cache (MALL) streams through
  // with non-temporal accesses: caching it cannot keep it for the next call
  // and only adds write-back traffic (DGER 8192^2: 6.09 against 5.6 TB/s).
  // One that fits keeps the cached path, which the next call re-reads from
  // the MALL (SGER 8192^2: 6.87 cached against 6.10 non-temporal).
  // (Into another matrix both count.)
  const int64_t footprint = src == A + aOffset ? lda : lda + lds;
  const bool nt = footprint * Cc * batch * (int64_t)sizeof(T) > (256ll << 20);
  for (int64_t b0 = 0; b0 < batch; b0 += 65535) {
    int64_t nb = std::min<int64_t>(65535, batch - b0);
    dim3 grid((unsigned)cdiv(R, rows_per_block),
              (unsigned)cdiv(Cc, kGerCols), (unsigned)nb);
    auto kernel = [&](auto add) {
      constexpr bool ADD = decltype(add)::value;
      return !vec ? ger_kernel<T, false, false, ADD>
             : nt ? ger_kernel<T, true, true, ADD>
                  : ger_kernel<T, true, false, ADD>;
    };
    (*alpha != T(0) ? kernel(std::true_type{}) : kernel(std::false_type{}))
        <<<grid, kThreads, 0, h->stream>>>(
            R, Cc, src + b0 * sA, lds, Ab + b0 * sA, lda, sA, v + b0 * sv, incv,
            sv, w + b0 * sw, incw, sw, *alpha);
    hcblasStatus_t st = launch_status();
    if (st != HCBLAS_STATUS_SUCCESS) return st;
  }
  return HCBLAS_STATUS_SUCCESS;
}

// GER from one matrix into another, D = alpha * x * y^T + A.
template <typename T>
hcblasStatus_t ger_out_entry(hcblasHandle_t h, hcblasOrder_t order, int M,
                             int N, const T *alpha, const T *x, int64_t incx,
                             const T *y, int64_t incy, const T *A, int64_t lda,
                             T *D, int64_t ldd) {
  if (!handle_ok(h)) return HCBLAS_STATUS_NOT_INITIALIZED;
  if (order != HCBLAS_ROW_MAJOR && order != HCBLAS_COL_MAJOR)
    return HCBLAS_STATUS_INVALID_VALUE;
  if (lda < std::max(1, order == HCBLAS_COL_MAJOR ? M : N))
    return HCBLAS_STATUS_INVALID_VALUE;
  if (M > 0 && N > 0 && A == nullptr) return HCBLAS_STATUS_INVALID_VALUE;
  return ger_entry<T>(h, order, M, N, alpha, x, 0, incx, y, 0, incy, D, 0, ldd,
                      1, true, 0, 0, 0, A, lda);
}

// Adjoint of A_out = alpha * x * y^T + A_in (no reference counterpart): for
// a cotangent dA (M x N in the given order) the GEMV pair
//   dx = alpha * dA * y,   dy = alpha * dA^T * x
// (dA_in = dA is the identity and needs no work). dx / dy are written with
// unit stride; either may be NULL. With both wanted of a matrix that the pair
// kernel covers, dA is read once.
template <typename T>
hcblasStatus_t ger_backward_entry(hcblasHandle_t h, hcblasOrder_t order,
                                         int M, int N, const T *alpha,
                                         const T *x, int64_t incx, const T *y,
                                         int64_t incy, const T *dA,
                                         int64_t ldda, T *dx, T *dy) {
  if (!handle_ok(h)) return HCBLAS_STATUS_NOT_INITIALIZED;
  const T zero = T(0);
  hcblasStatus_t st = HCBLAS_STATUS_SUCCESS;
  const bool col = order == HCBLAS_COL_MAJOR;
  const int64_t R = col ? M : N, Cc = col ? N : M;
  if (dx && dy && x && y && dA && alpha && *alpha != zero && M > 0 && N > 0 &&
      incx != 0 && incy != 0 && ldda >= R &&
      (col || order == HCBLAS_ROW_MAJOR)) {
    const PairPlan plan =
        plan_gemv_pair(h->num_cus, R, Cc, VecT<T>::n, sizeof(T));
    // (the two GEMVs where there is no memory for the partials)
    T *row_part =
        plan.xr ? static_cast<T *>(partials(h, plan.partial_bytes)) : nullptr;
    if (row_part != nullptr) {
      const T *p = col ? x : y, *q = col ? y : x;
      const int64_t incp = col ? incx : incy, incq = col ? incy : incx;
      T *yr = col ? dx : dy, *yc = col ? dy : dx;
      T *col_part = row_part + plan.blocks * R;
      const dim3 grid((unsigned)plan.blocks, (unsigned)plan.bands);
      const bool nt = (int64_t)sizeof(T) * R * Cc >= kStreamBytes;
#define HCB_PAIR(XR)                                                         \
  (nt ? gemv_pair_kernel<T, XR, true> : gemv_pair_kernel<T, XR, false>)      \
      <<<grid, kThreads, 0, h->stream>>>(R, Cc, ldda, dA, p, incp, q, incq,  \
                                         *alpha, yc, row_part, col_part)
      if (plan.xr == 4)
        HCB_PAIR(4);
      else if (plan.xr == 2)
        HCB_PAIR(2);
      else
        HCB_PAIR(1);
#undef HCB_PAIR
      if ((st = launch_status()) != HCBLAS_STATUS_SUCCESS) return st;
      auto finish = [&](int64_t len, int64_t splits, const T *part, T *out) {
        gemv_finish_kernel<T>
            <<<(unsigned)std::min<int64_t>(cdiv(len, 64), 4096), kThreads, 0,
               h->stream>>>(len, (int)splits, part, 0, out, 1, 0, *alpha, zero);
      };
      finish(R, plan.blocks, row_part, yr);
      if (plan.bands > 1) finish(Cc, plan.bands, col_part, yc);
      return launch_status();
    }
  }
  if (dx) {
    st = gemv_entry<T>(h, order, HCBLAS_OP_N, M, N, alpha, dA, 0, ldda, y, 0,
                       incy, &zero, dx, 0, 1, 1, false);
    if (st != HCBLAS_STATUS_SUCCESS) return st;
  }
  if (dy)
    st = gemv_entry<T>(h, order, HCBLAS_OP_T, M, N, alpha, dA, 0, ldda, x, 0,
                       incx, &zero, dy, 0, 1, 1, false);
  return st;
}

}  // namespace
}  // namespace hcb

using namespace hcb;

extern "C" {

hcblasStatus_t hcblasSgemv(hcblasHandle_t handle, hcblasOperation_t trans,
                           int m, int n, const float *alpha, const float *A,
                           int lda, const float *x, int incx, const float *beta,
                           float *y, int incy) {
  return gemv_entry<float>(handle, HCBLAS_COL_MAJOR, trans, m, n, alpha, A, 0,
                           lda, x, 0, incx, beta, y, 0, incy, 1, false);
}
hcblasStatus_t hcblasDgemv(hcblasHandle_t handle, hcblasOperation_t trans,
                           int m, int n, const double *alpha, const double *A,
                           int lda, const double *x, int incx,
                           const double *beta, double *y, int incy) {
  return gemv_entry<double>(handle, HCBLAS_COL_MAJOR, trans, m, n, alpha, A, 0,
                            lda, x, 0, incx, beta, y, 0, incy, 1, false);
}
hcblasStatus_t hcblasSgemvBatched(hcblasHandle_t handle,
                                  hcblasOperation_t trans, int m, int n,
                                  const float *alpha, const float *A, int lda,
                                  const float *x, int incx, const float *beta,
                                  float *y, int incy, int batchCount) {
  return gemv_entry<float>(handle, HCBLAS_COL_MAJOR, trans, m, n, alpha, A, 0,
                           lda, x, 0, incx, beta, y, 0, incy, batchCount, true);
}
hcblasStatus_t hcblasDgemvBatched(hcblasHandle_t handle,
                                  hcblasOperation_t trans, int m, int n,
                                  const double *alpha, const double *A,
                                  int lda, const double *x, int incx,
                                  const double *beta, double *y, int incy,
                                  int batchCount) {
  return gemv_entry<double>(handle, HCBLAS_COL_MAJOR, trans, m, n, alpha, A, 0,
                            lda, x, 0, incx, beta, y, 0, incy, batchCount,
                            true);
}
hcblasStatus_t hcblas_sgemv(hcblasHandle_t handle, hcblasOrder_t order,
                            hcblasOperation_t type, int M, int N,
                            const float *alpha, const float *A,
                            int64_t aOffset, int64_t lda, const float *X,
                            int64_t xOffset, int64_t incX, const float *beta,
                            float *Y, int64_t yOffset, int64_t incY) {
  return gemv_entry<float>(handle, order, type, M, N, alpha, A, aOffset, lda,
                           X, xOffset, incX, beta, Y, yOffset, incY, 1, false);
}
hcblasStatus_t hcblas_dgemv(hcblasHandle_t handle, hcblasOrder_t order,
                            hcblasOperation_t type, int M, int N,
                            const double *alpha, const double *A,
                            int64_t aOffset, int64_t lda, const double *X,
                            int64_t xOffset, int64_t incX, const double *beta,
                            double *Y, int64_t yOffset, int64_t incY) {
  return gemv_entry<double>(handle, order, type, M, N, alpha, A, aOffset, lda,
                            X, xOffset, incX, beta, Y, yOffset, incY, 1, false);
}

hcblasStatus_t hcblasSger(hcblasHandle_t handle, int m, int n,
                          const float *alpha, const float *x, int incx,
                          const float *y, int incy, float *A, int lda) {
  return ger_entry<float>(handle, HCBLAS_COL_MAJOR, m, n, alpha, x, 0, incx, y,
                          0, incy, A, 0, lda, 1);
}
hcblasStatus_t hcblasDger(hcblasHandle_t handle, int m, int n,
                          const double *alpha, const double *x, int incx,
                          const double *y, int incy, double *A, int lda) {
  return ger_entry<double>(handle, HCBLAS_COL_MAJOR, m, n, alpha, x, 0, incx, y,
                           0, incy, A, 0, lda, 1);
}
hcblasStatus_t hcblasSgerBatched(hcblasHandle_t handle, int m, int n,
                                 const float *alpha, const float *x, int incx,
                                 const float *y, int incy, float *A, int lda,
                                 int batchCount) {
  return ger_entry<float>(handle, HCBLAS_COL_MAJOR, m, n, alpha, x, 0, incx, y,
                          0, incy, A, 0, lda, batchCount);
}
hcblasStatus_t hcblasDgerBatched(hcblasHandle_t handle, int m, int n,
                                 const double *alpha, const double *x,
                                 int incx, const double *y, int incy,
                                 double *A, int lda, int batchCount) {
  return ger_entry<double>(handle, HCBLAS_COL_MAJOR, m, n, alpha, x, 0, incx,
                           y, 0, incy, A, 0, lda, batchCount);
}
hcblasStatus_t hcblas_sger(hcblasHandle_t handle, hcblasOrder_t order, int M,
                           int N, const float *alpha, const float *X,
                           int64_t xOffset, int64_t incX, const float *Y,
                           int64_t yOffset, int64_t incY, float *A,
                           int64_t aOffset, int64_t lda) {
  return ger_entry<float>(handle, order, M, N, alpha, X, xOffset, incX, Y,
                          yOffset, incY, A, aOffset, lda, 1);
}
hcblasStatus_t hcblas_dger(hcblasHandle_t handle, hcblasOrder_t order, int M,
                           int N, const double *alpha, const double *X,
                           int64_t xOffset, int64_t incX, const double *Y,
                           int64_t yOffset, int64_t incY, double *A,
                           int64_t aOffset, int64_t lda) {
  return ger_entry<double>(handle, order, M, N, alpha, X, xOffset, incX, Y,
                           yOffset, incY, A, aOffset, lda, 1);
}

hcblasStatus_t hcblas_sgemv_batched(
    hcblasHandle_t handle, hcblasOrder_t order, hcblasOperation_t type, int M,
    int N, const float *alpha, const float *A, int64_t aOffset,
    int64_t A_batchOffset, int64_t lda, const float *X, int64_t xOffset,
    int64_t X_batchOffset, int64_t incX, const float *beta, float *Y,
    int64_t yOffset, int64_t Y_batchOffset, int64_t incY, int batchSize) {
  return gemv_entry<float>(handle, order, type, M, N, alpha, A, aOffset, lda,
                           X, xOffset, incX, beta, Y, yOffset, incY, batchSize,
                           false, A_batchOffset, X_batchOffset, Y_batchOffset);
}
hcblasStatus_t hcblas_dgemv_batched(
    hcblasHandle_t handle, hcblasOrder_t order, hcblasOperation_t type, int M,
    int N, const double *alpha, const double *A, int64_t aOffset,
    int64_t A_batchOffset, int64_t lda, const double *X, int64_t xOffset,
    int64_t X_batchOffset, int64_t incX, const double *beta, double *Y,
    int64_t yOffset, int64_t Y_batchOffset, int64_t incY, int batchSize) {
  return gemv_entry<double>(handle, order, type, M, N, alpha, A, aOffset, lda,
                            X, xOffset, incX, beta, Y, yOffset, incY,
                            batchSize, false, A_batchOffset, X_batchOffset,
                            Y_batchOffset);
}
hcblasStatus_t hcblas_sger_batched(
    hcblasHandle_t handle, hcblasOrder_t order, int M, int N,
    const float *alpha, const float *X, int64_t xOffset,
    int64_t X_batchOffset, int64_t incX, const float *Y, int64_t yOffset,
    int64_t Y_batchOffset, int64_t incY, float *A, int64_t aOffset,
    int64_t A_batchOffset, int64_t lda, int batchSize) {
  return ger_entry<float>(handle, order, M, N, alpha, X, xOffset, incX, Y,
                          yOffset, incY, A, aOffset, lda, batchSize, false,
                          A_batchOffset, X_batchOffset, Y_batchOffset);
}
hcblasStatus_t hcblas_dger_batched(
    hcblasHandle_t handle, hcblasOrder_t order, int M, int N,
    const double *alpha, const double *X, int64_t xOffset,
    int64_t X_batchOffset, int64_t incX, const double *Y, int64_t yOffset,
    int64_t Y_batchOffset, int64_t incY, double *A, int64_t aOffset,
    int64_t A_batchOffset, int64_t lda, int batchSize) {
  return ger_entry<double>(handle, order, M, N, alpha, X, xOffset, incX, Y,
                           yOffset, incY, A, aOffset, lda, batchSize, false,
                           A_batchOffset, X_batchOffset, Y_batchOffset);
}

hcblasStatus_t hcblas_gemv_noalloc(hcblasHandle_t handle,
                                   hcblasDatatype_t dtype, hcblasOrder_t order,
                                   hcblasOperation_t type, int M, int N,
                                   const void *alpha, const void *A,
                                   int64_t aOffset, int64_t lda, const void *X,
                                   int64_t xOffset, int64_t incX,
                                   const void *beta, void *Y, int64_t yOffset,
                                   int64_t incY) {
  if (!handle_ok(handle)) return HCBLAS_STATUS_NOT_INITIALIZED;
  if (dtype == HCBLAS_R_32F)
    return gemv_entry<float>(
        handle, order, type, M, N, static_cast<const float *>(alpha),
        static_cast<const float *>(A), aOffset, lda,
        static_cast<const float *>(X), xOffset, incX,
        static_cast<const float *>(beta), static_cast<float *>(Y), yOffset,
        incY, 1, false, 0, 0, 0, true);
  if (dtype == HCBLAS_R_64F)
    return gemv_entry<double>(
        handle, order, type, M, N, static_cast<const double *>(alpha),
        static_cast<const double *>(A), aOffset, lda,
        static_cast<const double *>(X), xOffset, incX,
        static_cast<const double *>(beta), static_cast<double *>(Y), yOffset,
        incY, 1, false, 0, 0, 0, true);
  return HCBLAS_STATUS_INVALID_VALUE;
}

hcblasStatus_t hcblas_sger_out(hcblasHandle_t handle, hcblasOrder_t order,
                               int M, int N, const float *alpha,
                               const float *X, int64_t incX, const float *Y,
                               int64_t incY, const float *A, int64_t lda,
                               float *D, int64_t ldd) {
  return ger_out_entry<float>(handle, order, M, N, alpha, X, incX, Y, incY, A,
                              lda, D, ldd);
}
hcblasStatus_t hcblas_dger_out(hcblasHandle_t handle, hcblasOrder_t order,
                               int M, int N, const double *alpha,
                               const double *X, int64_t incX, const double *Y,
                               int64_t incY, const double *A, int64_t lda,
                               double *D, int64_t ldd) {
  return ger_out_entry<double>(handle, order, M, N, alpha, X, incX, Y, incY, A,
                               lda, D, ldd);
}

hcblasStatus_t hcblas_sger_backward(hcblasHandle_t handle,
                                    hcblasOrder_t order, int M, int N,
                                    const float *alpha, const float *X,
                                    int64_t incX, const float *Y, int64_t incY,
                                    const float *dA, int64_t ldda, float *dX,
                                    float *dY) {
  return ger_backward_entry<float>(handle, order, M, N, alpha, X, incX, Y,
                                   incY, dA, ldda, dX, dY);
}
hcblasStatus_t hcblas_dger_backward(hcblasHandle_t handle,
                                    hcblasOrder_t order, int M, int N,
                                    const double *alpha, const double *X,
                                    int64_t incX, const double *Y,
                                    int64_t incY, const double *dA,
                                    int64_t ldda, double *dX, double *dY) {
  return ger_backward_entry<double>(handle, order, M, N, alpha, X, incX, Y,
                                    incY, dA, ldda, dX, dY);
}

}  // extern "C"
