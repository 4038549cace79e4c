// Template instances of the MFMA GEMM for one complex type.
#include "gemm_launch_impl.hpp"

namespace hcb {
template hcblasStatus_t launch_gemm<Elem::F64, double, true>(hipStream_t, int,
                                                         GemmParams, bool,
                                                         bool, int64_t);
template hcblasStatus_t launch_gemm_splitk<Elem::F64, double, true>(
    hipStream_t, int, GemmParams, bool, bool, const SplitK &,
    typename ElemT<Elem::F64>::Acc *);
}  // namespace hcb
