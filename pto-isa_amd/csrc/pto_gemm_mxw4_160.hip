// The 256 x 160 MXFP8 / MXFP4 GEMM tile on four wavefronts (gemm_kernels_mxw4.hpp), wave grid 4 x 1: a translation unit a width, for the time they take to compile.
#define PTO_WAVES_M 4
#define PTO_WAVES_N 1
#define PTO_MFMA_M 16
#include "gemm_kernels_mxw4.hpp"

namespace pto_amd {
int gemm_mx_w4_160(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                   int format, int c_fp32)
{
    return launch_gemm_mxw4_format<160>(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
}
} // namespace pto_amd
