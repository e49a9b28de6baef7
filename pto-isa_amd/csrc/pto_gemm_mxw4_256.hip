// The 256 x 256 MXFP8 / MXFP4 GEMM tile on four wavefronts (gemm_kernels_mxw4.hpp): a translation unit of its own, for the time it takes to compile.
#define PTO_WAVES_M 4
#define PTO_WAVES_N 1
#define PTO_MFMA_M 16
#include "gemm_kernels_mxw4.hpp"

namespace pto_amd {
int gemm_mx_w4_256(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                   int format, int c_fp32)
{
#define PTO_MXW4_CASE(FMT, FA, FB)                                                               \
    if (format == FMT)                                                                          \
        return c_fp32 ? launch_gemm_mxw4<FA, FB, float, 256>(st, c, a, b, sa, sb, m, n, k) :     \
                        launch_gemm_mxw4<FA, FB, bfloat16_t, 256>(st, c, a, b, sa, sb, m, n, k);
    PTO_MXW4_CASE(0, 0, 0)
    PTO_MXW4_CASE(1, 1, 1)
    PTO_MXW4_CASE(2, 0, 1)
    PTO_MXW4_CASE(3, 1, 0)
    PTO_MXW4_CASE(4, 4, 4)
#undef PTO_MXW4_CASE
    return PTO_ERR_UNSUPPORTED;
}
} // namespace pto_amd
