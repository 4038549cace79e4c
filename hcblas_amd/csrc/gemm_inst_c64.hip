// Template instances of the MFMA GEMM for one complex type.
#include "gemm_launch_impl.hpp"

namespace hcb {
template hcblasStatus_t launch_gemm<Elem::F32, float, true>(hipStream_t, int,
                                                         GemmParams, bool,
                                                         bool, int64_t);
template hcblasStatus_t launch_gemm_splitk<Elem::F32, float, true>(
    hipStream_t, int, GemmParams, bool, bool, const SplitK &,
    typename ElemT<Elem::F32>::Acc *);
}  // namespace hcb
