// The 32- to 192-row MXFP8 / MXFP4 GEMM tiles with k split over two groups of wavefronts (gemm_kernels_mxks.hpp).
#define PTO_WAVES_M 4
#define PTO_WAVES_N 1
#define PTO_MFMA_M 16
#include "gemm_kernels_mxks.hpp"

namespace {
template <int FMT_A, int FMT_B, typename OutT>
int launch_shape(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k, int shape)
{
    switch (shape) {
    case 0: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 64, 64, 4, 4>(st, c, a, b, sa, sb, m, n, k);
    case 1: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 64, 128, 4, 2>(st, c, a, b, sa, sb, m, n, k);
    case 2: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 128, 64, 4, 2>(st, c, a, b, sa, sb, m, n, k);
    case 3: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 128, 128, 4, 2>(st, c, a, b, sa, sb, m, n, k);
    case 4: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 128, 192, 3, 2>(st, c, a, b, sa, sb, m, n, k);
    case 5: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 192, 128, 3, 2>(st, c, a, b, sa, sb, m, n, k);
    case 6: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 32, 32, 4, 2>(st, c, a, b, sa, sb, m, n, k);
    case 7: return launch_gemm_mxks<FMT_A, FMT_B, OutT, 32, 64, 4, 2>(st, c, a, b, sa, sb, m, n, k);
    default: return PTO_ERR_UNSUPPORTED;
    }
}
} // namespace

namespace pto_amd {
int gemm_mx_ks(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
               int format, int c_fp32, int shape)
{
#define PTO_MXKS_CASE(FMT, FA, FB)                                                               \
    if (format == FMT)                                                                          \
        return c_fp32 ? launch_shape<FA, FB, float>(st, c, a, b, sa, sb, m, n, k, shape) :       \
                        launch_shape<FA, FB, bfloat16_t>(st, c, a, b, sa, sb, m, n, k, shape);
    PTO_MXKS_CASE(0, 0, 0)
    PTO_MXKS_CASE(1, 1, 1)
    PTO_MXKS_CASE(2, 0, 1)
    PTO_MXKS_CASE(3, 1, 0)
    PTO_MXKS_CASE(4, 4, 4)
#undef PTO_MXKS_CASE
    return PTO_ERR_UNSUPPORTED;
}
} // namespace pto_amd
