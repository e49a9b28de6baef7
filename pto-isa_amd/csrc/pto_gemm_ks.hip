// The 32- to 256-row GEMM tiles with k split over two groups of wavefronts (gemm_kernels_ks.hpp).
#define PTO_WAVES_M 4
#define PTO_WAVES_N 1
#define PTO_MFMA_M 16
#include "gemm_kernels_ks.hpp"

namespace pto_amd {
int gemm_f16f32_ks(hipStream_t st, float *c, const _Float16 *a, const _Float16 *b, int m, int n, int k, int shape)
{
    switch (shape) {
    case 0: return launch_gemm_ks<32, 64, 5, 6>(st, c, a, b, m, n, k);
    case 1: return launch_gemm_ks<64, 64, 5, 4>(st, c, a, b, m, n, k);
    case 2: return launch_gemm_ks<64, 96, 4, 4>(st, c, a, b, m, n, k);
    case 3: return launch_gemm_ks<128, 64, 3, 4>(st, c, a, b, m, n, k);
    case 4: return launch_gemm_ks<128, 96, 5, 2>(st, c, a, b, m, n, k);
    case 5: return launch_gemm_ks<128, 128, 4, 2>(st, c, a, b, m, n, k);
    case 6: return launch_gemm_ks<192, 128, 4, 2>(st, c, a, b, m, n, k);
    case 7: return launch_gemm_ks<256, 128, 3, 2>(st, c, a, b, m, n, k);
    case 8: return launch_gemm_ks<192, 192, 3, 2>(st, c, a, b, m, n, k);
    case 9: return launch_gemm_ks<32, 32, 6, 4>(st, c, a, b, m, n, k);
    default: return PTO_ERR_UNSUPPORTED;
    }
}
} // namespace pto_amd

#if defined(PTO_ST_HOOKS)
// tile shape by number, as above
extern "C" int pto_gemm_f16f32_ks_variant(void *stream, float *c, const uint16_t *a, const uint16_t *b, int m, int n, int k, int variant)
{
    if (!c || !a || !b || m <= 0 || n <= 0 || k <= 0 || variant < 0 || variant > 9)
        return PTO_ERR_BAD_ARG;
    return pto_amd::gemm_f16f32_ks(static_cast<hipStream_t>(stream), c, reinterpret_cast<const _Float16 *>(a),
                                   reinterpret_cast<const _Float16 *>(b), m, n, k, variant);
}
#endif // PTO_ST_HOOKS
