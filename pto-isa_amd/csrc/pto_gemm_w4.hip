// The 256 x BN and 192 x BN GEMM tiles on four wavefronts (gemm_kernels_w4.hpp), wave grid 4 x 1.
#define PTO_WAVES_M 4
#define PTO_WAVES_N 1
#define PTO_MFMA_M 16
#include "gemm_kernels_w4.hpp"

namespace pto_amd {
int gemm_f16f32_w4(hipStream_t st, float *c, const _Float16 *a, const _Float16 *b, int m, int n, int k, int shape)
{
    switch (shape) {
    case 0: return launch_gemm_w4<256>(st, c, a, b, m, n, k);
    case 1: return launch_gemm_w4<192>(st, c, a, b, m, n, k);
    case 2: return launch_gemm_w4<128>(st, c, a, b, m, n, k);
    case 3: return launch_gemm_w4<256, 3>(st, c, a, b, m, n, k);
    case 4: return launch_gemm_w4<192, 3>(st, c, a, b, m, n, k);
    case 5: return launch_gemm_w4<128, 3>(st, c, a, b, m, n, k);
    default: return PTO_ERR_UNSUPPORTED;
    }
}
} // namespace pto_amd

#if defined(PTO_ST_HOOKS)
// tile shape by number: 0 .. 2 = 256 rows x 256 / 192 / 128 columns, 3 .. 5 = 192 rows x the same widths
extern "C" int pto_gemm_f16f32_w4_variant(void *stream, float *c, const uint16_t *a, const uint16_t *b, int m, int n, int k, int variant)
{
    if (!c || !a || !b || m <= 0 || n <= 0 || k <= 0 || variant < 0 || variant > 5)
        return PTO_ERR_BAD_ARG;
    return pto_amd::gemm_f16f32_w4(static_cast<hipStream_t>(stream), c, reinterpret_cast<const _Float16 *>(a),
                                   reinterpret_cast<const _Float16 *>(b), m, n, k, variant);
}
#endif // PTO_ST_HOOKS
