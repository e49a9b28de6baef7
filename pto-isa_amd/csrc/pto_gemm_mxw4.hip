// The MXFP8 / MXFP4 GEMM tile on four wavefronts (gemm_kernels_mxw4.hpp), wave grid 4 x 1.
#define PTO_WAVES_M 4
#define PTO_WAVES_N 1
#define PTO_MFMA_M 16
#include "gemm_kernels_mxw4.hpp"

namespace pto_amd {
// format: 0 = e4m3 x e4m3, 1 = e5m2 x e5m2, 2 = A e4m3 x B e5m2, 3 = A e5m2 x B e4m3, 4 = e2m1 x e2m1 (k then counts 4-bit
// elements, two per byte); width: 256, 192 or 128
int gemm_mx_w4(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                  int format, int c_fp32, int width)
{
    if (width == 256)
        return gemm_mx_w4_256(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
    if (format < 0 || format > 4 || (width != 192 && width != 128))
        return PTO_ERR_UNSUPPORTED;
#define PTO_MXW4_CASE(FMT, FA, FB)                                                                                         \
    if (format == FMT) {                                                                                                  \
        if (width == 192)                                                                                                 \
            return c_fp32 ? launch_gemm_mxw4<FA, FB, float, 192>(st, c, a, b, sa, sb, m, n, k) :                           \
                            launch_gemm_mxw4<FA, FB, bfloat16_t, 192>(st, c, a, b, sa, sb, m, n, k);                       \
        return c_fp32 ? launch_gemm_mxw4<FA, FB, float, 128>(st, c, a, b, sa, sb, m, n, k) :                               \
                        launch_gemm_mxw4<FA, FB, bfloat16_t, 128>(st, c, a, b, sa, sb, m, n, k);                           \
    }
    PTO_MXW4_CASE(0, 0, 0)
    PTO_MXW4_CASE(1, 1, 1)
    PTO_MXW4_CASE(2, 0, 1)
    PTO_MXW4_CASE(3, 1, 0)
    PTO_MXW4_CASE(4, 4, 4)
#undef PTO_MXW4_CASE
    return PTO_ERR_UNSUPPORTED;
}
} // namespace pto_amd
