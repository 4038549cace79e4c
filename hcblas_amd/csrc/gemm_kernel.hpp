// Generic MFMA GEMM macro-tile kernel for gfx950.
//
// Replaces the VALU register-micro-tile kernels of the reference
// (e.g. sgemm_NN_kernels.cpp:1360-1469 MICRO_TS16XMTS2, :137
// Mini_Batch_M128_N128_K16_TS16XMTS4_MB2; dgemm/hgemm copies of the same).
//
// Problem (column-major storage, after the host has folded row-major order
// into an operand swap):  C[M x N] = alpha * A'[M x K] * B'[K x N] + beta * C
// where A' element (m,k) is A[k + m*lda] when A_K (k contiguous) and
// A[m + k*lda] otherwise; B' element (k,n) is B[k + n*ldb] when B_K and
// B[n + k*ldb] otherwise.
//
// Tiling:
//   - workgroup = 64*WM*WN threads (WM x WN waves), macro tile BM x BN,
//     K step BK; each wave owns a (BM/WM) x (BN/WN) sub-tile made of 16x16
//     MFMA blocks (v_mfma_*_16x16x{4,4,32,32,64}).
//   - LDS holds both operands k-contiguous ([rows][BK] + 16 bytes of padding
//     per row, which makes the 16-byte fragment reads of 16 rows
//     bank-conflict-free), double-buffered: global loads for tile k+1 are in
//     flight in registers while the MFMAs consume tile k, and one barrier per
//     K step separates the two buffers.
//   - a lane reads one 16-byte fragment per operand per chunk; the four lane
//     groups (lane/16) hold four disjoint k sub-ranges, and the same mapping is
//     used for A and B, so the MFMA sums exactly the products of the chunk.
//   - MFMA output layout (16x16, four values per lane): value r of lane l is
//     C(4*(l/16) + r, l%16) for the FP32/INT32-accumulating forms and
//     C(l/16 + 4*r, l%16) for v_mfma_f64_16x16x4f64 (out_row below).
//   - tile order: consecutive workgroup ids are spread over the 8 XCDs by the
//     dispatcher, so ids are remapped to give each XCD a contiguous slice of
//     a GROUP_M-grouped tile order (A and B panels stay in that XCD's L2).
#pragma once


#include <type_traits>

#include "common.hpp"
#include "gemm_tiles.hpp"

namespace hcb {

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));
typedef int intx4 __attribute__((ext_vector_type(4)));
typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

template <Elem E>
struct ElemT;
template <>
struct ElemT<Elem::F32> {
  using T = float;
  using Acc = float;
  using AccV = floatx4;
  static constexpr int VEC = 4;    // elements per 16-byte fragment
  static constexpr int STEPS = 4;  // MFMAs per fragment pair
};
template <>
struct ElemT<Elem::F64> {
  using T = double;
  using Acc = double;
  using AccV = doublex4;
  static constexpr int VEC = 2;
  static constexpr int STEPS = 2;
};
template <>
struct ElemT<Elem::F16> {
  using T = uint16_t;  // binary16 bits
  using Acc = float;
  using AccV = floatx4;
  static constexpr int VEC = 8;
  static constexpr int STEPS = 1;
};
template <>
struct ElemT<Elem::BF16> {
  using T = uint16_t;  // bfloat16 bits
  using Acc = float;
  using AccV = floatx4;
  static constexpr int VEC = 8;
  static constexpr int STEPS = 1;
};
template <>
struct ElemT<Elem::I8> {
  using T = int8_t;
  using Acc = int;
  using AccV = intx4;
  static constexpr int VEC = 16;
  static constexpr int STEPS = 1;
};

template <typename To, typename From>
__device__ __forceinline__ To bitcast(const From &f) {
  static_assert(sizeof(To) == sizeof(From), "bitcast size");
  To t;
  __builtin_memcpy(&t, &f, sizeof(To));
  return t;
}

typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef int intx16 __attribute__((ext_vector_type(16)));

// Accumulator of one MI x MI MFMA block (MI = 16 or 32).
// 16-byte fragment / staging register as a native vector (the HIP uint4
// struct defeats scalar replacement of the staging arrays).
typedef unsigned int vec4u __attribute__((ext_vector_type(4)));
typedef unsigned int vec2u __attribute__((ext_vector_type(2)));
// The same 16 bytes of global memory at an address that is only a multiple of
// the element size: gfx950 serves a global_load / store_dwordx4 at any
// address, so one kernel takes every base, offset and leading dimension. A
// wave's 1 KiB run off a cache line boundary touches one more line.
template <int ESIZE>
struct GlobalVecOf;
template <>
struct GlobalVecOf<1> { typedef vec4u type __attribute__((aligned(1))); };
template <>
struct GlobalVecOf<2> { typedef vec4u type __attribute__((aligned(2))); };
template <>
struct GlobalVecOf<4> { typedef vec4u type __attribute__((aligned(4))); };
template <>
struct GlobalVecOf<8> { typedef vec4u type __attribute__((aligned(8))); };
template <>
struct GlobalVecOf<16> { typedef vec4u type __attribute__((aligned(8))); };
template <typename T>
using GlobalVec = GlobalVecOf<(int)sizeof(T)>;

template <Elem E, int MI>
struct AccOf;
template <>
struct AccOf<Elem::F32, 16> { using type = floatx4; };
template <>
struct AccOf<Elem::F32, 32> { using type = floatx16; };
template <>
struct AccOf<Elem::F64, 16> { using type = doublex4; };
template <>
struct AccOf<Elem::F16, 16> { using type = floatx4; };
template <>
struct AccOf<Elem::F16, 32> { using type = floatx16; };
template <>
struct AccOf<Elem::BF16, 16> { using type = floatx4; };
template <>
struct AccOf<Elem::BF16, 32> { using type = floatx16; };
template <>
struct AccOf<Elem::I8, 16> { using type = intx4; };
template <>
struct AccOf<Elem::I8, 32> { using type = intx16; };

// MFMA step S of a fragment pair for MI x MI blocks:
//   FP32  v_mfma_f32_16x16x4f32 / v_mfma_f32_32x32x2f32 (one float per step)
//   FP64  v_mfma_f64_16x16x4f64                         (one double per step)
//   FP16  v_mfma_f32_16x16x32_f16 / v_mfma_f32_32x32x16_f16
//   BF16  v_mfma_f32_16x16x32_bf16 / v_mfma_f32_32x32x16_bf16
//   INT8  v_mfma_i32_16x16x64_i8 / v_mfma_i32_32x32x32_i8
template <Elem E, int MI, int S>
__device__ __forceinline__ void mfma_step(const vec4u &a, const vec4u &b,
                                          typename AccOf<E, MI>::type &c) {
  if constexpr (E == Elem::F32) {
    const uint32_t ua = S == 0 ? a.x : S == 1 ? a.y : S == 2 ? a.z : a.w;
    const uint32_t ub = S == 0 ? b.x : S == 1 ? b.y : S == 2 ? b.z : b.w;
    if constexpr (MI == 16)
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(ua),
                                               __uint_as_float(ub), c, 0, 0, 0);
    else
      c = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(ua),
                                               __uint_as_float(ub), c, 0, 0, 0);
  } else if constexpr (E == Elem::F64) {
    static_assert(MI == 16, "FP64 MFMA is 16x16 only");
    const double av =
        bitcast<double>(S == 0 ? a.xy : a.zw);
    const double bv =
        bitcast<double>(S == 0 ? b.xy : b.zw);
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, c, 0, 0, 0);
  } else if constexpr (E == Elem::F16) {
    if constexpr (MI == 16)
      c = __builtin_amdgcn_mfma_f32_16x16x32_f16(bitcast<halfx8>(a),
                                                 bitcast<halfx8>(b), c, 0, 0, 0);
    else
      c = __builtin_amdgcn_mfma_f32_32x32x16_f16(bitcast<halfx8>(a),
                                                 bitcast<halfx8>(b), c, 0, 0, 0);
  } else if constexpr (E == Elem::BF16) {
    if constexpr (MI == 16)
      c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(bitcast<bf16x8>(a),
                                                  bitcast<bf16x8>(b), c, 0, 0,
                                                  0);
    else
      c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(bitcast<bf16x8>(a),
                                                  bitcast<bf16x8>(b), c, 0, 0,
                                                  0);
  } else {
    if constexpr (MI == 16)
      c = __builtin_amdgcn_mfma_i32_16x16x64_i8(bitcast<intx4>(a),
                                                bitcast<intx4>(b), c, 0, 0, 0);
    else
      c = __builtin_amdgcn_mfma_i32_32x32x32_i8(bitcast<intx4>(a),
                                                bitcast<intx4>(b), c, 0, 0, 0);
  }
}

// ---------------------------------------------------------------------------
// Global -> register -> LDS tile loader for one operand.
// ROWS = tile extent in m (or n); the LDS tile is [ROWS][BK] k-contiguous.
// KCONT: the global operand is k-contiguous (element (r,k) at P[k + r*ld]).
//
// Every load is 16 bytes wide, whatever the operand's alignment, without
// branches and inside the operand:
//   - k-contiguous: a vector that reaches past K is read from k = K - VEC on
//     and moved down to its place (zeros behind it) before it goes to LDS;
//   - r-contiguous: of a row count R that is not a whole number of vectors,
//     the last vector is read from row R - VEC on and stays so: the tile rows
//     of that vector hold the rows `edge_shift` further down, which the
//     epilogue undoes (no other tile row is affected). Steps past K read the
//     last k and are zeroed before they go to LDS.
// Only an operand shorter than one vector is read by elements (load_narrow).
// Element-wise loads of unaligned operands cost 1.1-3 times the whole GEMM
// (529 x 192 x 1152 SGEMM NN 51.6 us, 2051 x 1777 x 1533 DGEMM NT 226 us).
// ---------------------------------------------------------------------------
template <typename T, int ROWS, int BK, bool KCONT, int NTH = 256>
struct TileLoader {
  static constexpr int VEC = 16 / (int)sizeof(T);
  using GV = typename GlobalVec<T>::type;
  static constexpr int NV = ROWS * BK / VEC;  // 16-byte vectors per tile
  static constexpr int PER_THREAD = (NV + NTH - 1) / NTH;
  static constexpr int ROWB = BK * (int)sizeof(T) + 16;  // LDS row stride
  // Transposing (r-contiguous) tiles: each group of 64 vectors covers
  // 8 r-vectors x 8 k, so a wave reads 128-byte runs of global memory and its
  // element-wise LDS stores spread over the banks (2-way instead of 8-way
  // conflicts for 32 r-vectors of one k).
  static constexpr bool BLOCKED = !KCONT && (ROWS / VEC) % 8 == 0 &&
                                  BK % 8 == 0 && NV % 64 == 0;
  // FP32 transposing tiles with four vectors per thread: each thread loads
  // the four k-lines of one 4-row x 4-k block and writes it with four
  // 16-byte LDS stores along k (a 4 x 4 transpose in its registers) instead
  // of sixteen 4-byte ones. The 16 lanes of a group take 4 consecutive
  // r-vectors x 4 consecutive k-quads, whose rows (4j + e) x ROWB + 16 kq
  // fall on 16 distinct 4-bank groups for both row strides used (528 and
  // 144 bytes); the four groups of a wave continue along r, so a load
  // instruction reads four k-lines in 256-byte runs.
  static constexpr bool TRANS4 =
      !KCONT && VEC == 4 && NV == 4 * NTH && ROWS % 16 == 0 && BK % 16 == 0 &&
      (ROWS / 16) * (BK / 16) * 16 == NTH;
  // 16-bit transposing tiles with four vectors per thread: each thread loads
  // the four k-lines of one 8-row vector and writes its 8 rows x 4 k with
  // eight 8-byte LDS stores along k (16-bit selects pair the k values) instead
  // of thirty-two 2-byte ones. Groups of 16 lanes take 16 k-quads of one
  // r-vector, neighbouring groups neighbouring r-vectors; the slots of a
  // half-wave, (8 jr + e) x ROWB + 8 kq, are 32 distinct 8-byte slots of 256
  // bytes, since 8 ROWB is 128 modulo 256 for every K step.
  static constexpr bool TRANS4H = !KCONT && VEC == 8 && NV == 4 * NTH &&
                                  BK % 64 == 0 && ROWS % 32 == 0;
  // The same with two vectors per thread: a thread loads two k-lines of one
  // r-vector and writes its rows with 8-byte (FP32) or 4-byte (16-bit) stores
  // along k. FP32: groups of 16 lanes take 16 k-pairs, and of four neighbouring
  // r-vectors the half-waves take {0, 2} and {1, 3} (row offsets 0 / 128 and
  // 64 / 192 of 256 bytes). 16-bit: half-waves take 32 k-pairs, so that a
  // wave's 4-byte slots of two r-vectors are all distinct (16 k-pairs of four
  // r-vectors collide in pairs).
  static constexpr bool TRANS2 = !KCONT && VEC == 4 && NV == 2 * NTH &&
                                 BK % 32 == 0 && ROWS % 16 == 0;
  static constexpr bool TRANS2H = !KCONT && VEC == 8 && NV == 2 * NTH &&
                                  BK % 32 == 0 && ROWS % 32 == 0;
  const int tid;  // thread of the workgroup
  vec4u reg[PER_THREAD];

  __device__ __forceinline__ explicit TileLoader(int t) : tid(t) {}

  // (r, k) of vector v of the tile (r, k are element indices).
  __device__ __forceinline__ static void vec_pos(int v, int &r, int &k) {
    if (KCONT) {
      r = v / (BK / VEC);
      k = (v % (BK / VEC)) * VEC;
    } else if (TRANS4) {
      const int t = v % NTH, i = v / NTH;
      const int g = t >> 4, jj = t & 3, kk = (t >> 2) & 3;
      constexpr int GJ = ROWS / 16;  // groups of 4 r-vectors along r
      r = (4 * (g % GJ) + jj) * 4;
      k = (4 * (g / GJ) + kk) * 4 + i;
    } else if (TRANS2 || TRANS2H || TRANS4H) {
      constexpr int NR = ROWS / VEC;       // r-vectors
      constexpr int KL = TRANS4H ? 4 : 2;  // k-lines per thread
      constexpr int GL = TRANS2H && BK % 64 == 0 ? 32 : 16;  // lanes per group
      // (unsigned: a group index that is always 0 costs no registers)
      const unsigned t = (unsigned)v % NTH, i = (unsigned)v / NTH, g = t / GL;
      unsigned j = g % NR;
      if (TRANS2) j = (j & ~3u) | ((j & 1) << 1) | ((j >> 1) & 1);
      r = j * VEC;
      k = ((g / NR) * GL + t % GL) * KL + i;
    } else if (BLOCKED) {
      constexpr int NRB = ROWS / VEC / 8;
      const int w = v >> 6, l = v & 63;
      r = ((w % NRB) * 8 + (l & 7)) * VEC;
      k = (w / NRB) * 8 + (l >> 3);
    } else {
      k = v / (ROWS / VEC);
      r = (v % (ROWS / VEC)) * VEC;
    }
  }

  // The contiguous dimension holds at least one vector.
  __device__ __forceinline__ static bool wide(int R, int K) {
    return (KCONT ? K : R) >= VEC;
  }

  // Tile rows of the last vector lie this far above the operand's rows.
  __device__ __forceinline__ static int edge_shift(int R) {
    return !KCONT && R >= VEC && R % VEC != 0 ? VEC - R % VEC : 0;
  }

  // First row of that vector (R if there is none).
  __device__ __forceinline__ static int edge_row(int R) {
    return edge_shift(R) ? R - R % VEC : R;
  }

  // A wide operand's step at k0: FULL if it lies entirely inside [0, K),
  // else mask() has to follow before the LDS store. Rows past R read row r0
  // (k-contiguous) or the last vector; they only feed outputs that are never
  // stored. The loaded registers are first consumed by the LDS store after
  // the MFMAs: the global latency stays hidden behind them.
  template <bool FULL>
  __device__ __forceinline__ void load_wide(const T *__restrict__ P,
                                            int64_t ld, int r0, int k0, int R,
                                            int K) {
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int v = tid + i * NTH;
      if (NV % NTH != 0 && v >= NV) continue;
      int r, k;
      vec_pos(v, r, k);
      const int last = KCONT ? K - VEC : K - 1;
      const int gr = r0 + r, gk = FULL || k0 + k < last ? k0 + k : last;
      const T *src = KCONT ? P + (int64_t)(gr < R ? gr : r0) * ld + gk
                           : P + (int64_t)gk * ld +
                                 (gr < R - VEC ? gr : R - VEC);
      reg[i] = *reinterpret_cast<const GV *>(src);
    }
  }

  // Zeros for k >= K in the registers of the (partial) step at k0.
  __device__ __forceinline__ void mask(int k0, int K) {
    // K - VEC of a moved vector lies this far below its place (0: none).
    const int shift = KCONT && K % VEC ? VEC - K % VEC : 0;
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      int r, k;
      vec_pos(tid + i * NTH, r, k);
      const int n = K - (k0 + k);  // k values of this vector inside K
      if (KCONT && n > 0 && n < VEC) reg[i] = down(reg[i], shift);
      if (n <= 0) reg[i] = vec4u{};
    }
  }

  // The vector moved down by n elements (0 < n < VEC), zeros behind it.
  __device__ __forceinline__ static vec4u down(vec4u w, int n) {
    const int b = n * (int)sizeof(T);
    if (b & 8) w = vec4u{w.z, w.w, 0, 0};
    if (b & 4) w = vec4u{w.y, w.z, w.w, 0};
    if (sizeof(T) < 4 && (b & 3)) {
      const int sh = 8 * (b & 3);
      w = vec4u{__builtin_amdgcn_alignbit(w.y, w.x, sh),
                __builtin_amdgcn_alignbit(w.z, w.y, sh),
                __builtin_amdgcn_alignbit(w.w, w.z, sh), w.w >> sh};
    }
    return w;
  }

  // An operand shorter than one vector, element by element. EACH: only the
  // elements inside it (most vectors of a narrow tile lie outside); otherwise
  // clamped loads, one vector's addresses at a time, for kernels whose registers
  // this path must not cost.
  template <bool EACH = false>
  __device__ __forceinline__ void load_narrow(const T *__restrict__ P,
                                              int64_t ld, int r0, int k0,
                                              int R, int K) {
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int v = tid + i * NTH;
      if (NV % NTH != 0 && v >= NV) continue;
      int r, k;
      vec_pos(v, r, k);
      T t[VEC];
#pragma unroll
      for (int e = 0; e < VEC; ++e) {
        const int gr = r0 + r + (KCONT ? 0 : e), gk = k0 + k + (KCONT ? e : 0);
        if constexpr (EACH) {
          t[e] = T{};
          if (gr < R && gk < K)
            t[e] = P[KCONT ? gr * ld + gk : gk * ld + gr];
        } else {
          const int64_t rr = gr < R ? gr : R - 1, kk = gk < K ? gk : K - 1;
          const T x = KCONT ? P[rr * ld + kk] : P[kk * ld + rr];
          t[e] = gk < K ? x : T(0);
        }
      }
      __builtin_memcpy(&reg[i], t, 16);
      if constexpr (!EACH) __builtin_amdgcn_sched_barrier(0);
    }
  }

  // Any step of any operand, ready for the LDS store.
  __device__ __forceinline__ void load_step(const T *__restrict__ P,
                                            int64_t ld, int r0, int k0, int R,
                                            int K, bool full) {
    if (full) {
      load_wide<true>(P, ld, r0, k0, R, K);
    } else if (wide(R, K)) {
      load_wide<false>(P, ld, r0, k0, R, K);
      mask(k0, K);
    } else {
      load_narrow(P, ld, r0, k0, R, K);
    }
  }

  __device__ __forceinline__ void store(char *lds) const {
    if constexpr (TRANS4) {
      int r, k;
      vec_pos(tid, r, k);  // reg[i] holds rows r..r+3 at k + i
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<vec4u *>(lds + (r + e) * ROWB + k * 4) =
            vec4u{reg[0][e], reg[1][e], reg[2][e], reg[3][e]};
      return;
    }
    if constexpr (TRANS2) {
      int r, k;
      vec_pos(tid, r, k);  // reg[i] holds rows r..r+3 at k + i
#pragma unroll
      for (int e = 0; e < 4; ++e)
        *reinterpret_cast<vec2u *>(lds + (r + e) * ROWB + k * 4) =
            vec2u{reg[0][e], reg[1][e]};
      return;
    }
    if constexpr (TRANS2H) {
      int r, k;
      vec_pos(tid, r, k);  // reg[i] holds rows r..r+7 at k + i
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        const int d = e >> 1;
        *reinterpret_cast<uint32_t *>(lds + (r + e) * ROWB + k * 2) =
            (e & 1) ? (reg[0][d] >> 16) | (reg[1][d] & 0xffff0000u)
                    : (reg[0][d] & 0xffffu) | (reg[1][d] << 16);
      }
      return;
    }
    if constexpr (TRANS4H) {
      int r, k;
      vec_pos(tid, r, k);  // reg[i] holds rows r..r+7 at k + i
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        // Row r + e is the low (e even) or high half of dword e / 2.
        const int d = e >> 1;
        const uint32_t lo =
            (e & 1) ? (reg[0][d] >> 16) | (reg[1][d] & 0xffff0000u)
                    : (reg[0][d] & 0xffffu) | (reg[1][d] << 16);
        const uint32_t hi =
            (e & 1) ? (reg[2][d] >> 16) | (reg[3][d] & 0xffff0000u)
                    : (reg[2][d] & 0xffffu) | (reg[3][d] << 16);
        *reinterpret_cast<vec2u *>(lds + (r + e) * ROWB + k * 2) =
            vec2u{lo, hi};
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < PER_THREAD; ++i) {
      const int v = tid + i * NTH;
      if (NV % NTH != 0 && v >= NV) continue;
      int r, k;
      vec_pos(v, r, k);
      if (KCONT) {
        *reinterpret_cast<vec4u *>(lds + r * ROWB + k * (int)sizeof(T)) =
            reg[i];
      } else {
        T t[VEC];
        __builtin_memcpy(t, &reg[i], 16);
#pragma unroll
        for (int e = 0; e < VEC; ++e)
          *reinterpret_cast<T *>(lds + (r + e) * ROWB + k * (int)sizeof(T)) =
              t[e];
      }
    }
  }
};

// Loader of a complex operand for the real embedding of a complex product. Its
// rows, k and step are those of the real operands,
//   EMBED (A'):  rows 2m, 2m + 1 of columns 2k, 2k + 1 hold (x, -y; y, x) with
//                x + iy = (ar + i ai) * a(m, k), the products rounded
//                separately;
//   else (B'):   row n of columns 2k, 2k + 1 holds re b(k, n), im b(k, n);
// a and b conjugated if asked. The operand is read in complex elements (the
// loader above, on 8- or 16-byte elements) and takes this form on its way into
// LDS. (Written to memory by a pass of its own, four reals for each complex
// element of A', it cost two launches and 6 MK + 4 KN complex elements of
// traffic: sixty-four 96^3 CGEMMs 22.9 us, now 10.9; 1024^3 NT 102 -> 95; 300^3
// ZGEMM NN 32 -> 13.)
typedef double doublex2 __attribute__((ext_vector_type(2)));
template <typename T>
using ComplexElem =
    typename std::conditional<sizeof(T) == 4, double, doublex2>::type;
template <typename T, int ROWS, int BK, bool KCONT, int NTH, bool EMBED>
struct ComplexLoader
    : TileLoader<ComplexElem<T>, EMBED ? ROWS / 2 : ROWS, BK / 2, KCONT, NTH> {
  using L =
      TileLoader<ComplexElem<T>, EMBED ? ROWS / 2 : ROWS, BK / 2, KCONT, NTH>;
  using CT = ComplexElem<T>;
  static constexpr int RD = EMBED ? 2 : 1;  // real rows per complex row
  static constexpr int ROWB = BK * (int)sizeof(T) + 16;
  const uint32_t flip;  // sign bit where the operand is conjugated
  const T ar, ai;
  int kv;  // k of the held step inside K (complex)

  __device__ __forceinline__ ComplexLoader(int t, bool conj, T r, T i)
      : L(t), flip(conj ? 0x80000000u : 0u), ar(r), ai(i) {}

  __device__ __forceinline__ static bool wide(int R, int K) {
    return L::wide(R / RD, K / 2);
  }
  __device__ __forceinline__ static int edge_shift(int R) {
    return RD * L::edge_shift(R / RD);
  }
  __device__ __forceinline__ static int edge_row(int R) {
    return RD * L::edge_row(R / RD);
  }
  template <bool FULL>
  __device__ __forceinline__ void load_wide(const T *P, int64_t ld, int r0,
                                            int k0, int R, int K) {
    kv = FULL ? BK / 2 : (K - k0) / 2;
    L::template load_wide<FULL>(reinterpret_cast<const CT *>(P), ld, r0 / RD,
                                k0 / 2, R / RD, K / 2);
  }
  template <bool EACH = false>
  __device__ __forceinline__ void load_narrow(const T *P, int64_t ld, int r0,
                                              int k0, int R, int K) {
    kv = (K - k0) / 2;
    L::template load_narrow<EACH>(reinterpret_cast<const CT *>(P), ld, r0 / RD, k0 / 2,
                   R / RD, K / 2);
  }
  __device__ __forceinline__ void mask(int k0, int K) { L::mask(k0 / 2, K / 2); }

  __device__ __forceinline__ void store(char *lds) const {
#pragma clang fp contract(off)
    constexpr int VC = L::VEC;  // complex elements per vector
#pragma unroll
    for (int i = 0; i < L::PER_THREAD; ++i) {
      const int v = this->tid + i * NTH;
      if (L::NV % NTH != 0 && v >= L::NV) continue;
      int r, k;
      L::vec_pos(v, r, k);
      char *p = lds + RD * r * ROWB + 2 * k * (int)sizeof(T);
      vec4u w = this->reg[i];
      if constexpr (VC == 2) w.y ^= flip;
      w.w ^= flip;
      if constexpr (EMBED) {
        T x[VC], y[VC], c[2 * VC];
        __builtin_memcpy(c, &w, 16);
#pragma unroll
        for (int e = 0; e < VC; ++e) {
          // (steps past K stay zero whatever alpha is)
          const bool in = k + (KCONT ? e : 0) < kv;
          const T sr = in ? ar : T(0), si = in ? ai : T(0);
          x[e] = sr * c[2 * e] - si * c[2 * e + 1];
          y[e] = sr * c[2 * e + 1] + si * c[2 * e];
        }
        if constexpr (VC == 2 && KCONT) {
          const T t0[4] = {x[0], -y[0], x[1], -y[1]};
          const T t1[4] = {y[0], x[0], y[1], x[1]};
          *reinterpret_cast<vec4u *>(p) = bitcast<vec4u>(t0);
          *reinterpret_cast<vec4u *>(p + ROWB) = bitcast<vec4u>(t1);
        } else {
          using W = typename std::conditional<VC == 2, vec2u, vec4u>::type;
#pragma unroll
          for (int e = 0; e < VC; ++e) {
            const T t0[2] = {x[e], -y[e]}, t1[2] = {y[e], x[e]};
            *reinterpret_cast<W *>(p + 2 * e * ROWB) = bitcast<W>(t0);
            *reinterpret_cast<W *>(p + (2 * e + 1) * ROWB) = bitcast<W>(t1);
          }
        }
      } else if constexpr (VC == 2 && !KCONT) {
        *reinterpret_cast<vec2u *>(p) = vec2u{w.x, w.y};
        *reinterpret_cast<vec2u *>(p + ROWB) = vec2u{w.z, w.w};
      } else {
        *reinterpret_cast<vec4u *>(p) = w;
      }
    }
  }
};

// alpha and the conjugations of a complex product.
struct ComplexArgs {
  double ar, ai;
  int conj_a, conj_b;
};

// The loader pair of a product: real operands, or (CX) a complex product's.
template <typename T, bool CX, bool A_K, bool B_K, int BM, int BN, int BK,
          int NTH>
struct Loaders {
  using A = typename std::conditional<
      CX, ComplexLoader<T, BM, BK, A_K, NTH, true>,
      TileLoader<T, BM, BK, A_K, NTH>>::type;
  using B = typename std::conditional<
      CX, ComplexLoader<T, BN, BK, B_K, NTH, false>,
      TileLoader<T, BN, BK, B_K, NTH>>::type;
  __device__ __forceinline__ static A a(int tid, const ComplexArgs &cx) {
    if constexpr (CX)
      return A(tid, cx.conj_a, (T)cx.ar, (T)cx.ai);
    else
      return A(tid);
  }
  __device__ __forceinline__ static B b(int tid, const ComplexArgs &cx) {
    if constexpr (CX)
      return B(tid, cx.conj_b, (T)cx.ar, (T)cx.ai);
    else
      return B(tid);
  }
};

// Batch member and tile of a workgroup of a (tiles, 1, batch) grid. Workgroups
// go to the 8 XCDs in turn, so in whole groups of 8 members each takes all its
// tiles on one XCD, whose L2 then holds the member's A and B once.
__device__ __forceinline__ void batch_tile(int tiles, int &z, int &pid) {
  constexpr int kXcd = 8;
  z = blockIdx.z;
  pid = blockIdx.x;
  if (z < (int)gridDim.z / kXcd * kXcd && tiles < 32768) {  // l < 2^31
    const unsigned l = (unsigned)z * tiles + pid, i = l / kXcd;
    z = i / tiles * kXcd + l % kXcd;
    pid = i % tiles;
  }
}

// Tile id -> (tile_m, tile_n): XCD-contiguous slices of a GROUP_M-grouped order
// (`spread`: consecutive ids are on different XCDs).
__device__ __forceinline__ void tile_coords(int pid, int tm, int tn,
                                            int &tile_m, int &tile_n,
                                            bool spread = true) {
  constexpr int kXcd = 8;
  constexpr int GROUP_M = 8;
  const int nt = tm * tn;
  if (spread && nt % kXcd == 0)
    pid = (pid % kXcd) * (nt / kXcd) + pid / kXcd;
  const int width = GROUP_M * tn;
  const int group = pid / width;
  const int first_m = group * GROUP_M;
  const int gsize = (tm - first_m) < GROUP_M ? (tm - first_m) : GROUP_M;
  const int in_group = pid % width;
  tile_m = first_m + in_group % gsize;
  tile_n = in_group / gsize;
}

// Row (within an MI x MI MFMA block) of accumulator value r of lane group g
// (g = lane / MI; the column is lane % MI):
//   16x16 FP32/INT32 accumulators: 4g + r;   16x16 FP64: g + 4r;
//   32x32 (16 values per lane):    8*(r/4) + 4g + r%4.
template <Elem E, int MI>
__device__ __forceinline__ int out_row(int g, int r) {
  if constexpr (MI == 32)
    return 8 * (r >> 2) + 4 * g + (r & 3);
  else if constexpr (E == Elem::F64)
    return g + 4 * r;
  else
    return 4 * g + r;
}

// Output conversion.
template <typename O, typename Acc>
__device__ __forceinline__ O to_out(Acc v) {
  return (O)v;
}
template <>
__device__ __forceinline__ uint16_t to_out<uint16_t, float>(float v) {
  return bitcast<uint16_t>((_Float16)v);
}
template <typename Acc, typename O>
__device__ __forceinline__ Acc from_out(O v) {
  return (Acc)v;
}
template <>
__device__ __forceinline__ float from_out<float, uint16_t>(uint16_t v) {
  return (float)bitcast<_Float16>(v);
}

__device__ __forceinline__ float fma_acc(float a, float b, float c) {
  return __builtin_fmaf(a, b, c);
}
__device__ __forceinline__ double fma_acc(double a, double b, double c) {
  return __builtin_fma(a, b, c);
}

struct GemmParams {
  int M, N, K;
  const void *A;
  int64_t lda, strideA;
  const void *B;
  int64_t ldb, strideB;
  void *C;
  int64_t ldc, strideC;
  // Pointer-array batches (device arrays); nullptr selects the strided form.
  const void *const *Aptrs;
  const void *const *Bptrs;
  void *const *Cptrs;
  int64_t aOff, bOff, cOff;
  double alpha, beta;
  int tiles_m, tiles_n;
  // A complex product's real embedding: M, N, K, offsets and strides are the
  // real form's, lda and ldb the complex operands'.
  // (Plain fields, read in the kernel only where needed: as a nested struct
  // they kept the compiler from seeing that the pointers are global ones, and
  // flat loads cost 3-5% of a GEMM.)
  double cx_ar, cx_ai;
  int conj_a, conj_b;
};

// LDS bytes used by one macro tile (two buffers of A and B).
template <Elem E, int BM, int BN, int BK>
constexpr int tile_lds_bytes() {
  return 2 * (BM + BN) * (BK * (int)sizeof(typename ElemT<E>::T) + 16);
}

// Wave sub-tile geometry of a BM x BN macro tile split over WM x WN waves.
template <Elem E, int BM, int BN, int WM, int WN, int MI>
struct WaveTile {
  static constexpr int WTM = BM / WM, WTN = BN / WN;
  static constexpr int FM = WTM / MI, FN = WTN / MI;
  static constexpr int NVAL = MI * MI / 64;  // accumulator values per block
  static_assert(FM * MI == WTM && FN * MI == WTN, "wave tile");
  using AccV = typename AccOf<E, MI>::type;
};

// Main loop of one BM x BN tile at (m0, n0): acc = A'(m0.., :) * B'(:, n0..)
// over the whole K range. Shared by the plain / batched kernel, the grouped
// kernel and the residue kernel, so all of them produce bit-identical sums
// on MFMA blocks of the same size MI (a block's lane groups hold different k of a
// chunk, so 16x16 and 32x32 blocks add in another order, and a size's last bits can
// change with its tile). CX: a complex product's operands (cx).
template <Elem E, bool A_K, bool B_K, int BM, int BN, int BK, int WM, int WN,
          int MI, bool NARROW, bool CX>
__device__ __forceinline__ void gemm_mainloop(
    const typename ElemT<E>::T *__restrict__ A, int64_t lda,
    const typename ElemT<E>::T *__restrict__ B, int64_t ldb, int M, int N,
    int K, int m0, int n0, int tid, char *lds, ComplexArgs cx,
    typename WaveTile<E, BM, BN, WM, WN, MI>::AccV (
        &acc)[WaveTile<E, BM, BN, WM, WN, MI>::FM]
             [WaveTile<E, BM, BN, WM, WN, MI>::FN]) {
  using Tr = ElemT<E>;
  using T = typename Tr::T;
  using WT = WaveTile<E, BM, BN, WM, WN, MI>;
  using AccV = typename WT::AccV;
  constexpr int VEC = Tr::VEC;
  constexpr int NG = 64 / MI;       // lane groups along k
  constexpr int CK = NG * VEC;      // k per fragment chunk
  static_assert(BK % CK == 0, "BK must be a multiple of the chunk");
  constexpr int NTH = 64 * WM * WN;  // workgroup size
  constexpr int WTM = WT::WTM, WTN = WT::WTN, FM = WT::FM, FN = WT::FN;

  using LP = Loaders<T, CX, A_K, B_K, BM, BN, BK, NTH>;
  using LA = typename LP::A;
  using LB = typename LP::B;
  constexpr int ROWB = LA::ROWB;
  constexpr int A_BYTES = BM * ROWB, B_BYTES = BN * ROWB;

  const int wave = tid >> 6, lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int lrow = lane % MI, lgrp = lane / MI;

#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = AccV{};

  LA la = LP::a(tid, cx);
  LB lb = LP::b(tid, cx);
  const int nk = (K + BK - 1) / BK;
  // (NARROW = false: the caller knows that both operands are wide)
  const bool wide_a = !NARROW || LA::wide(M, K);
  const bool wide_b = !NARROW || LB::wide(N, K);
  const int nfull = wide_a && wide_b ? K / BK : 0;  // steps without a tail

  // MFMAs over one LDS buffer. Small wave tiles (the 64 x 64 tiles of 8
  // waves, at most 2 fragments of each operand, and the 4-wave 64 x 64 FP64
  // tiles, 2 x 2 fragments) read chunk c + 1's fragments into a second
  // register set before chunk c's MFMAs, so the LDS latency is not paid
  // between chunks (1024^3 DGEMM 71.5 against 75.3 us); the larger tiles
  // have no registers to spare for it, and the 4-wave 128 x 128 16-bit tile
  // measured no faster with it.
  constexpr bool PIPE = (WM * WN == 8 && FM * FN <= 2) ||
                        (E == Elem::F64 && WM * WN == 4 && FM * FN == 4);
  // The large 8-wave tiles (256 x 256 and 256 x 128, two waves per SIMD)
  // issue the step's LDS writes and global loads among the first chunk's
  // MFMAs, behind that chunk's fragment reads, instead of before them: both
  // waves of a SIMD leave the barrier together, and the writes would
  // otherwise hold the MFMA pipe idle while they drain and the fragment
  // reads queue behind them (8192^3 SGEMM 3-7% faster over the four
  // transpose forms, DGEMM 6-11%, 3072^3 SGEMM on 256 x 128 tiles 10%).
  // The 4-wave 128 x 128 FP32 tile (64 x 64 per wave on 16 x 16 blocks, two
  // workgroups per CU) gains the same way (2048^3 SGEMM 166 against 187 us),
  // and so does the 8-wave 128 x 64 FP64 tile (2048^3 DGEMM 294 against
  // 344 us); the 4-wave 128 x 128 16-bit tile, with 4 MFMAs per chunk, was
  // 5-18% slower with it. The complex 64 x 64 FP32 tile of 4 waves, whose LDS
  // writes wait for the embedding's arithmetic, gains most: 1024^3 CGEMM NN 94.9
  // us with the writes before the MFMAs, 77.4 among them (and 93.4 for the
  // embedding written to memory first); 6144 x 160 x 3208 289, 232 (254).
  constexpr bool ILV =
      !PIPE && ((WM * WN == 8 && FM * FN >= 4) ||
                (WM * WN == 4 && MI == 16 && FM * FN >= (CX ? 4 : 8)));
  // 16-bit tiles have 8 MFMAs per chunk, too few to carry a whole step's
  // writes and loads: their four chunks take A's LDS writes, B's, A's loads
  // and B's loads in turn (8192^3 HGEMM 2-4% faster than all in chunk 0).
  constexpr bool SPREAD = ILV && BK / CK == 4 && FM * FN * Tr::STEPS < 16;
  // hook(c): the step's LDS writes and loads, or the part of them that
  // chunk c carries.
  auto compute = [&](const char *cur, auto hook) {
    const char *As = cur;
    const char *Bs = cur + A_BYTES;
    vec4u afp[PIPE ? 2 : 1][FM], bfp[PIPE ? 2 : 1][FN];
    auto frag = [&](int c, int set) {
      const int kbyte = (c * CK + lgrp * VEC) * (int)sizeof(T);
#pragma unroll
      for (int i = 0; i < FM; ++i)
        afp[set][i] = *reinterpret_cast<const vec4u *>(
            As + (wm * WTM + i * MI + lrow) * ROWB + kbyte);
#pragma unroll
      for (int j = 0; j < FN; ++j)
        bfp[set][j] = *reinterpret_cast<const vec4u *>(
            Bs + (wn * WTN + j * MI + lrow) * ROWB + kbyte);
    };
    if constexpr (PIPE) frag(0, 0);
#pragma unroll
    for (int c = 0; c < BK / CK; ++c) {
      const int set = PIPE ? (c & 1) : 0;
      if constexpr (PIPE) {
        if (c + 1 < BK / CK) frag(c + 1, (c + 1) & 1);
      } else {
        frag(c, 0);
      }
      if constexpr (ILV) {
        if (SPREAD || c == 0) hook(c);
      }
      const vec4u(&af)[FM] = afp[set];
      const vec4u(&bf)[FN] = bfp[set];
#pragma unroll
      for (int i = 0; i < FM; ++i)
#pragma unroll
        for (int j = 0; j < FN; ++j)
          mfma_step<E, MI, 0>(af[i], bf[j], acc[i][j]);
      if constexpr (Tr::STEPS > 1) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            mfma_step<E, MI, 1>(af[i], bf[j], acc[i][j]);
      }
      if constexpr (Tr::STEPS > 2) {
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            mfma_step<E, MI, 2>(af[i], bf[j], acc[i][j]);
#pragma unroll
        for (int i = 0; i < FM; ++i)
#pragma unroll
          for (int j = 0; j < FN; ++j)
            mfma_step<E, MI, 3>(af[i], bf[j], acc[i][j]);
      }
      if constexpr (PIPE) {
        // The next chunk's LDS reads go out behind the first MFMAs.
        constexpr int NMF = FM * FN * Tr::STEPS, NRD = FM + FN;
#pragma unroll
        for (int i = 0; i < NMF; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          if (i < NRD) __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if constexpr (SPREAD) {
        constexpr int NMF = FM * FN * Tr::STEPS, NRD = FM + FN;
        __builtin_amdgcn_sched_group_barrier(0x100, NRD, 0);  // DS read
#pragma unroll
        for (int i = 0; i < NMF; ++i) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
          if (c < 2)
            __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // DS write
          else
            __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM read
        }
        __builtin_amdgcn_sched_barrier(0);
      } else if constexpr (ILV) {
        if (c == 0) {
          constexpr int NMF = FM * FN * Tr::STEPS, NRD = FM + FN;
          __builtin_amdgcn_sched_group_barrier(0x100, NRD, 0);  // DS read
          // One LDS write, then one global load, every SP MFMAs (4, or
          // fewer where the chunk is short).
          constexpr int NWR = LA::PER_THREAD + LB::PER_THREAD;
          constexpr int SP = NMF >= 4 * NWR ? 4 : (NMF / NWR >= 2 ? 2 : 1);
#pragma unroll
          for (int i = 0; i < NMF; ++i) {
            __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // MFMA
            if (i % SP == 0)
              __builtin_amdgcn_sched_group_barrier(0x200, 1, 0);  // DS write
            if (i % SP == SP / 2)
              __builtin_amdgcn_sched_group_barrier(0x020, 1, 0);  // VMEM read
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
    }
  };
  auto none = [](int) {};
  auto buf = [&](int kt) { return lds + (kt & 1) * (A_BYTES + B_BYTES); };

  if (nk == 0) return;
  // Pipeline: the registers hold step kt+1 while step kt computes. At the
  // top of step kt they are written to the other LDS buffer (free: every
  // wave passed the previous barrier) and refilled with step kt+2, so the
  // LDS writes overlap this step's MFMAs and one barrier ends the step.
  auto load = [&](int k) {
    if (wide_a)
      la.template load_wide<false>(A, lda, m0, k * BK, M, K);
    else
      la.template load_narrow<true>(A, lda, m0, k * BK, M, K);
    if (wide_b)
      lb.template load_wide<false>(B, ldb, n0, k * BK, N, K);
    else
      lb.template load_narrow<true>(B, ldb, n0, k * BK, N, K);
  };
  auto store = [&](int k) {
    if ((k + 1) * BK > K) {
      if (wide_a) la.mask(k * BK, K);
      if (wide_b) lb.mask(k * BK, K);
    }
    la.store(buf(k));
    lb.store(buf(k) + A_BYTES);
  };
  load(0);
  store(0);
  if (nk > 1) load(1);
  __syncthreads();
  int kt = 0;
  for (; kt + 2 < nfull; ++kt) {
    auto step = [&](int c) {
      if constexpr (SPREAD) {
        if (c == 0) la.store(buf(kt + 1));
        if (c == 1) lb.store(buf(kt + 1) + A_BYTES);
        if (c == 2)
          la.template load_wide<true>(A, lda, m0, (kt + 2) * BK, M, K);
        if (c == 3)
          lb.template load_wide<true>(B, ldb, n0, (kt + 2) * BK, N, K);
      } else {
        la.store(buf(kt + 1));
        lb.store(buf(kt + 1) + A_BYTES);
        la.template load_wide<true>(A, lda, m0, (kt + 2) * BK, M, K);
        lb.template load_wide<true>(B, ldb, n0, (kt + 2) * BK, N, K);
      }
    };
    if constexpr (ILV) {
      compute(buf(kt), step);
    } else {
      step(0);
      __builtin_amdgcn_sched_barrier(0);
      compute(buf(kt), none);
    }
    __syncthreads();
  }
  for (; kt < nk; ++kt) {
    if (kt + 1 < nk) store(kt + 1);
    if (kt + 2 < nk) load(kt + 2);
    compute(buf(kt), none);
    __syncthreads();
  }
}

// Epilogue of a BM x BN tile through LDS. Stored straight from the
// accumulator layout, one store instruction writes one value per lane into
// 16 or 32 different columns, so the tile leaves in BM*BN/64 scattered store
// instructions; for short K loops (batched and grouped problems) that weighs
// as much as the main loop. Here the accumulators go to LDS as [n][m] (m
// contiguous, row stride BM plus 16 bytes), NC columns at a time (as many as
// the main loop's LDS holds), and each thread then blends and stores VE
// consecutive rows of one column with one 16-byte access, a column's BM rows
// by BM / VE consecutive lanes. The arithmetic is the direct form's
// (alpha * acc, then fma(beta, C, .)), so results are bit-identical to it.
// Accumulator layouts (value r of lane l, block row / column):
//   32x32 FP32/INT32: row 8 (r / 4) + 4 (l / 32) + r % 4, column l % 32;
//   16x16 FP32: row 4 (l / 16) + r, column l % 16;
//   16x16 FP64: row l / 16 + 4 r, column l % 16.
// edge_m / shift_m, edge_n / shift_n: the loaders' edge_row and edge_shift of
// either operand. Output row m >= edge_m lies in tile row m + shift_m (and
// columns alike). C is accessed 16 bytes at a time at any alignment; one by one
// leave the rows of a vector that reaches past M, or over edge_m (16-bit outputs
// of an FP32 operand, whose vectors are shorter). BOTH: below.
// Expects the LDS free on entry (the main loop ends with a barrier) and ends
// with a barrier.
template <Elem E, typename OutT, int BM, int BN, int WM, int WN, int MI,
          int LDS_BYTES, bool BOTH = true, typename AccArr>
__device__ __forceinline__ void store_tile_lds(const AccArr &acc, OutT *C,
                                               int64_t ldc, int M, int N,
                                               int m0, int n0, double alpha_d,
                                               double beta_d, int tid,
                                               char *lds, int edge_m,
                                               int shift_m, int edge_n,
                                               int shift_n) {
  using WT = WaveTile<E, BM, BN, WM, WN, MI>;
  using Acc = typename ElemT<E>::Acc;
  constexpr int LROW = BM + 16 / (int)sizeof(Acc);  // elements
  constexpr int NC_FIT = LDS_BYTES / (LROW * (int)sizeof(Acc));
  constexpr int NC = NC_FIT >= BN ? BN
                     : NC_FIT >= 128 ? 128
                     : NC_FIT >= 64  ? 64
                     : NC_FIT >= 32  ? 32
                                     : 16;
  static_assert(NC >= MI && BN % NC == 0 && NC * LROW * (int)sizeof(Acc) <= LDS_BYTES,
                "epilogue column chunk");
  constexpr int VE = 16 / (int)sizeof(OutT);
  constexpr int NTH = 64 * WM * WN;
  constexpr int TPC = BM / VE;  // threads per column
  static_assert(BM % VE == 0 && NTH % TPC == 0, "epilogue shape");
  Acc *t = reinterpret_cast<Acc *>(lds);
  const int wave = tid >> 6, lane = tid & 63;
  const int wm = wave / WN, wn = wave % WN;
  const int lrow = lane % MI, lgrp = lane / MI;
  const Acc alpha = (Acc)alpha_d, beta = (Acc)beta_d;
  using GV = typename GlobalVec<OutT>::type;
#pragma unroll
  for (int c0 = 0; c0 < BN; c0 += NC) {
#pragma unroll
    for (int j = 0; j < WT::FN; ++j) {
      const int cb = wn * WT::WTN + j * MI;  // wave-uniform
      if (cb < c0 || cb >= c0 + NC) continue;
      const int n = cb - c0 + lrow;
#pragma unroll
      for (int i = 0; i < WT::FM; ++i) {
        const int mb = wm * WT::WTM + i * MI;
        if constexpr (MI == 32) {
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            const auto &a = acc[i][j];
            floatx4 v = {(float)a[4 * q], (float)a[4 * q + 1],
                         (float)a[4 * q + 2], (float)a[4 * q + 3]};
            *reinterpret_cast<floatx4 *>(t + n * LROW + mb + 8 * q +
                                         4 * lgrp) = v;
          }
        } else if constexpr (sizeof(Acc) == 8) {
#pragma unroll
          for (int r = 0; r < 4; ++r)
            t[n * LROW + mb + lgrp + 4 * r] = acc[i][j][r];
        } else {
          *reinterpret_cast<floatx4 *>(t + n * LROW + mb + 4 * lgrp) =
              acc[i][j];
        }
      }
    }
    __syncthreads();
    // BOTH: two loops, one for tiles with moved rows, where a moved vector is read
    // from LDS by elements and stored whole (BF16 156 x 128x92x28 8.7 -> 6.3 us).
    // Without it one loop, in which moved rows leave one by one, for kernels of
    // many tile bodies (4096^3 among the grouped problems 371 -> 374 us in two
    // loops) or with no registers to spare (the adjoints, whose 256 x 256 tile
    // with an FP32 A spills one in two: 177 BF16 backward products of 31 x 214 x
    // 931 87 -> 99 us, one of 79 x 31 x 128 11.9 -> 12.6).
    const auto whole = [&](OutT *dst, const Acc *src) {
      OutT cin[VE], o[VE];
      if (beta != Acc(0)) {
        const vec4u w = *reinterpret_cast<const GV *>(dst);
        __builtin_memcpy(cin, &w, 16);
      }
#pragma unroll
      for (int e = 0; e < VE; ++e) {
        Acc v = alpha * src[e];
        if (beta != Acc(0)) v = fma_acc(beta, from_out<Acc>(cin[e]), v);
        o[e] = to_out<OutT>(v);
      }
      vec4u w;
      __builtin_memcpy(&w, o, 16);
      *reinterpret_cast<GV *>(dst) = w;
    };
    const auto columns = [&](auto moved) {
#pragma unroll
      for (int cc = 0; cc < NC; cc += NTH / TPC) {
        const int nl = cc + tid / TPC;
        const int ml = (tid % TPC) * VE;
        const int n = n0 + c0 + nl, m = m0 + ml;
        if (nl < NC && n < N && m < M) {
          OutT *dst = C + (int64_t)n * ldc + m;
          const Acc *src = t + (n < edge_n ? nl : nl + shift_n) * LROW + ml;
          const bool below = !decltype(moved)::value || m < edge_m;
          if (m + VE <= (decltype(moved)::value && below ? edge_m : M)) {
            whole(dst, below ? src : src + shift_m);
          } else {
            const int ne = M - m < VE ? M - m : VE;
#pragma unroll 1
            for (int e = 0; e < ne; ++e) {
              const int s =
                  decltype(moved)::value && m + e >= edge_m ? e + shift_m : e;
              Acc v = alpha * src[s];
              if (beta != Acc(0)) v = fma_acc(beta, from_out<Acc>(dst[e]), v);
              dst[e] = to_out<OutT>(v);
            }
          }
        }
      }
    };
    if constexpr (BOTH) {
      if (shift_m == 0 || m0 + BM <= edge_m)
        columns(std::false_type{});
      else
        columns(std::true_type{});
    } else {
#pragma unroll
      for (int cc = 0; cc < NC; cc += NTH / TPC) {
        const int nl = cc + tid / TPC;
        const int ml = (tid % TPC) * VE;
        const int n = n0 + c0 + nl, m = m0 + ml;
        if (nl < NC && n < N && m < M) {
          OutT *dst = C + (int64_t)n * ldc + m;
          const Acc *src = t + (n < edge_n ? nl : nl + shift_n) * LROW + ml;
          if (m + VE <= edge_m) {
            whole(dst, src);
          } else {
            const int ne = M - m < VE ? M - m : VE;
            for (int e = 0; e < ne; ++e) {
              Acc v = alpha * src[m + e < edge_m ? e : e + shift_m];
              if (beta != Acc(0)) v = fma_acc(beta, from_out<Acc>(dst[e]), v);
              dst[e] = to_out<OutT>(v);
            }
          }
        }
      }
    }
    __syncthreads();
  }
}

// One BM x BN output tile at (m0, n0) of C = alpha*A'*B' + beta*C, the whole
// K range; beta == 0 never reads C. LDS_BYTES: the LDS at `lds`.
template <Elem E, typename OutT, bool A_K, bool B_K, int BM, int BN, int BK,
          int WM, int WN, int MI, int LDS_BYTES, bool NARROW, bool CX = false,
          bool BOTH = true>
__device__ __forceinline__ void gemm_tile(
    const typename ElemT<E>::T *__restrict__ A, int64_t lda,
    const typename ElemT<E>::T *__restrict__ B, int64_t ldb, OutT *C,
    int64_t ldc, int M, int N, int K, double alpha_d, double beta_d, int m0,
    int n0, int tid, char *lds, ComplexArgs cx = {}) {
  using T = typename ElemT<E>::T;
  using WT = WaveTile<E, BM, BN, WM, WN, MI>;
  using LP = Loaders<T, CX, A_K, B_K, BM, BN, BK, 64 * WM * WN>;
  using LA = typename LP::A;
  using LB = typename LP::B;
  typename WT::AccV acc[WT::FM][WT::FN];
  gemm_mainloop<E, A_K, B_K, BM, BN, BK, WM, WN, MI, NARROW, CX>(
      A, lda, B, ldb, M, N, K, m0, n0, tid, lds, cx, acc);
  store_tile_lds<E, OutT, BM, BN, WM, WN, MI, LDS_BYTES, BOTH>(
      acc, C, ldc, M, N, m0, n0, alpha_d, beta_d, tid, lds,
      LA::edge_row(M), LA::edge_shift(M), LB::edge_row(N), LB::edge_shift(N));
}

// NARROW: an operand may be shorter than one vector along its contiguous
// dimension (the host knows; carrying the element-wise loads in every kernel cost
// 1-5%: SGEMM 1024^3 NN row-major 22.95 us against 22.55, HGEMM 1024^3 NN 9.24
// against 8.82, sixty-four 96^3 CGEMMs 10.7 against 10.3).
template <Elem E, typename OutT, bool A_K, bool B_K, int BM, int BN, int BK,
          int WM, int WN, int MI = 16, bool CX = false, bool NARROW = false>
__global__ __launch_bounds__(64 * WM * WN) void gemm_mfma_kernel(
    GemmParams p) {
  using T = typename ElemT<E>::T;
  constexpr int LDS_BYTES = tile_lds_bytes<E, BM, BN, BK>();
  __shared__ __attribute__((aligned(16))) char lds[LDS_BYTES];
  int z, pid;
  batch_tile(p.tiles_m * p.tiles_n, z, pid);
  const T *A;
  const T *B;
  OutT *C;
  if (p.Aptrs)
    A = static_cast<const T *>(p.Aptrs[z]) + p.aOff;
  else
    A = static_cast<const T *>(p.A) + p.aOff + (int64_t)z * p.strideA;
  if (p.Bptrs)
    B = static_cast<const T *>(p.Bptrs[z]) + p.bOff;
  else
    B = static_cast<const T *>(p.B) + p.bOff + (int64_t)z * p.strideB;
  if (p.Cptrs)
    C = static_cast<OutT *>(p.Cptrs[z]) + p.cOff;
  else
    C = static_cast<OutT *>(p.C) + p.cOff + (int64_t)z * p.strideC;
  int tile_m, tile_n;
  tile_coords(pid, p.tiles_m, p.tiles_n, tile_m, tile_n, gridDim.z < 8);
  gemm_tile<E, OutT, A_K, B_K, BM, BN, BK, WM, WN, MI, LDS_BYTES, NARROW, CX>(
      A, p.lda, B, p.ldb, C, p.ldc, p.M, p.N, p.K, p.alpha, p.beta,
      tile_m * BM, tile_n * BN, threadIdx.x, lds,
      CX ? ComplexArgs{p.cx_ar, p.cx_ai, p.conj_a, p.conj_b} : ComplexArgs{});
}

// Split-K partial tile: the K range [z ks, min(K, (z + 1) ks)) of one
// tile of a single (unbatched) problem, stored without alpha / beta into
// W + z M N (column-major, ld M). For problems with about as many tiles as
// CUs and a long K, splitting K gives every CU several workgroups to switch
// between; splitk_reduce_kernel then adds the partials in split order.
// (The last slice of K may be shorter than a vector: of a k-contiguous operand
// that is as wide as one, the vector then begins in the slice before.)
template <Elem E, bool A_K, bool B_K, int BM, int BN, int BK, int WM, int WN,
          int MI, bool CX = false, bool NARROW = false>
__global__ __launch_bounds__(64 * WM * WN) void gemm_splitk_kernel(
    GemmParams p, int ks, typename ElemT<E>::Acc *W) {
  using T = typename ElemT<E>::T;
  using Acc = typename ElemT<E>::Acc;
  constexpr int LDS_BYTES = tile_lds_bytes<E, BM, BN, BK>();
  __shared__ __attribute__((aligned(16))) char lds[LDS_BYTES];
  const int z = blockIdx.z;
  const int k0 = z * ks;
  const int kl = p.K - k0 < ks ? p.K - k0 : ks;
  // (k0 is even: of a complex operand, k0 / 2 lines of 2 lda reals)
  const T *A = static_cast<const T *>(p.A) + p.aOff +
               (A_K ? (int64_t)k0 : (int64_t)k0 * p.lda);
  const T *B = static_cast<const T *>(p.B) + p.bOff +
               (B_K ? (int64_t)k0 : (int64_t)k0 * p.ldb);
  int tile_m, tile_n;
  tile_coords(blockIdx.x, p.tiles_m, p.tiles_n, tile_m, tile_n);
  gemm_tile<E, Acc, A_K, B_K, BM, BN, BK, WM, WN, MI, LDS_BYTES, NARROW, CX>(
      A, p.lda, B, p.ldb, W + (int64_t)z * p.M * p.N, p.M, p.M, p.N, kl, 1.0,
      0.0, tile_m * BM, tile_n * BN, threadIdx.x, lds,
      CX ? ComplexArgs{p.cx_ar, p.cx_ai, p.conj_a, p.conj_b} : ComplexArgs{});
}

// C = alpha * sum_z W[z] + beta * C, the partials added in split order.
template <typename Acc, typename OutT>
__global__ __launch_bounds__(256) void splitk_reduce_kernel(
    int S, int M, int N, const Acc *__restrict__ W, OutT *C, int64_t ldc,
    Acc alpha, Acc beta) {
  const int64_t MN = (int64_t)M * N;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < MN;
       i += (int64_t)gridDim.x * 256) {
    Acc s = W[i];
    int z = 1;
    for (; z + 3 < S; z += 4) {  // four loads in flight, added in order
      Acc w[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) w[j] = W[(int64_t)(z + j) * MN + i];
#pragma unroll
      for (int j = 0; j < 4; ++j) s += w[j];
    }
    for (; z < S; ++z) s += W[(int64_t)z * MN + i];
    const int64_t n = i / M, m = i - n * M;
    OutT *dst = C + n * ldc + m;
    Acc v = alpha * s;
    if (beta != Acc(0)) v = fma_acc(beta, from_out<Acc>(*dst), v);
    *dst = to_out<OutT>(v);
  }
}

}  // namespace hcb
