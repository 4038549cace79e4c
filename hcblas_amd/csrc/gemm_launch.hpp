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

// Split-K form for one problem (no batch, no pointer arrays): partial tiles of
// the K slices into W (splits * M * N accumulators), then the reduction into C.
template <Elem E, typename OutT, bool CX = false>
hcblasStatus_t launch_gemm_splitk(hipStream_t stream, int num_cus,
                                  GemmParams p, bool a_k, bool b_k,
                                  const SplitK &sk,
                                  typename ElemT<E>::Acc *W);

}  // namespace hcb
