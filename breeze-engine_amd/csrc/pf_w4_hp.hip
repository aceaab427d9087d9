// Prefill GEMM kernels for INT4 weights, two-pass INT16 activations.
#include "pf4_kernel.h"

namespace bq {
template hipError_t launch_pf4<true>(bool*, const Pf4Args&, bool, int, int, dim3, hipStream_t);
}  // namespace bq
