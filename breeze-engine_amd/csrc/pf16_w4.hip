// The INT4 GEMM for few output tiles (both activation modes: the records
// differ, not the kernel).
#include "pf16_kernel.h"

namespace bq {

hipError_t launch_pf16(const Pf4Args& p, bool zp, int ahead, int grid, hipStream_t st) {
    const int row_waves = (p.M + 15) / 16;
    const dim3 g((unsigned)grid), b(kPf16Waves * 64);
    if (zp && ahead == 4) pf16_kernel<true, 4><<<g, b, 0, st>>>(p, row_waves);
    else if (zp) pf16_kernel<true, 2><<<g, b, 0, st>>>(p, row_waves);
    else if (ahead == 4) pf16_kernel<false, 4><<<g, b, 0, st>>>(p, row_waves);
    else pf16_kernel<false, 2><<<g, b, 0, st>>>(p, row_waves);
    return hipGetLastError();
}

}  // namespace bq
