// The INT8 GEMM for few output tiles, both activation modes.
#include "pf16_w8_kernel.h"

namespace bq {

template <bool HP>
static void launch(const PfArgs& p, int scm, dim3 g, int row_waves, hipStream_t st) {
    const dim3 b(kPf16Waves * 64);
    if (scm == 0) pf16_w8_kernel<HP, 0><<<g, b, 0, st>>>(p, row_waves);
    else if (scm == 1) pf16_w8_kernel<HP, 1><<<g, b, 0, st>>>(p, row_waves);
    else pf16_w8_kernel<HP, 2><<<g, b, 0, st>>>(p, row_waves);
}

hipError_t launch_pf16_w8(const PfArgs& p, bool hp, int scm, int grid, hipStream_t st) {
    const int row_waves = (p.M + 15) / 16;
    if (hp) launch<true>(p, scm, dim3((unsigned)grid), row_waves, st);
    else launch<false>(p, scm, dim3((unsigned)grid), row_waves, st);
    return hipGetLastError();
}

}  // namespace bq
