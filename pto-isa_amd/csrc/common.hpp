// Shared host-side helpers of the C ABI translation units.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "pto_amd.h"
#if defined(PTO_ST_HOOKS)
#include "pto_amd_st.h" // test-only entry points (libpto_st.so)
#endif

namespace pto_amd {
extern thread_local int g_last_hip_error;

inline int check_launch()
{
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) {
        g_last_hip_error = static_cast<int>(e);
        return PTO_ERR_HIP;
    }
    return PTO_OK;
}

// compute units of the device that is current at the first call
inline int compute_units()
{
    static const int cus = [] {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n <= 0)
            n = 256;
        return n;
    }();
    return cus;
}

// Are the results of a launch to be stored past the L2 (write-through, system scope)?  A kernel ends with every L2 writing back what
// is dirty in it, after the last store and before the next kernel: 1.3 us behind 1 MB, 1.8 behind 4, 3.3 behind 12, 5.4 behind 33.
// Stored through, whole 64-byte pieces (what the kernels that ask write per row and instruction) are on their way at once:
// GEMM 256 x 3072 x 1024 6.12 -> 5.61 us, 1024 x 3072 x 1024 13.3 -> 11.9, 6144 x 3072 x 512 37.7 -> 31.7, 3072^3 50.6 -> 49.2.
// Pieces that straddle the 64 bytes are written by parts, which costs more (6144 x 3068 x 512 38.5 -> 50.6), and of a result much
// larger than the L2s (32 MB) most is written back while other tiles run (4096 x 6144 x 4096, 101 MB: 160.5 -> 157.9, 6144 x 6144 x 2048,
// 151 MB: 133 and 135).
inline bool store_through(const void *out, uint64_t rowBytes, uint64_t bytes)
{
    return (rowBytes | (uint64_t)(uintptr_t)out) % 64 == 0 && bytes <= (uint64_t)96 << 20;
}

// Dynamic LDS above 64 KiB has to be opted into per kernel.
template <typename K>
inline int allow_lds(K kernel, int bytes)
{
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void *>(kernel),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
    if (e != hipSuccess) {
        g_last_hip_error = static_cast<int>(e);
        return PTO_ERR_HIP;
    }
    return PTO_OK;
}

// defined in pto_gemm_w4.hip: tiles on four wavefronts, K-steps of 64; shape 0 .. 2 = 256 rows x 256 / 192 / 128 columns,
// 3 .. 5 = 192 rows x the same widths.  PTO_ERR_UNSUPPORTED unless m and n hold a tile, n % 4 == 0 and k % 128 == 0
int gemm_f16f32_w4(hipStream_t st, float *c, const _Float16 *a, const _Float16 *b, int m, int n, int k, int shape);
// defined in pto_gemm_ks.hip: tiles on eight wavefronts with k split over two groups of them; shape 0 .. 9 = 32 x 64, 64 x 64,
// 64 x 96, 128 x 64, 128 x 96, 128 x 128, 192 x 128, 256 x 128, 192 x 192, 32 x 32.  PTO_ERR_UNSUPPORTED unless n % 4 == 0 and k % 32 == 0
int gemm_f16f32_ks(hipStream_t st, float *c, const _Float16 *a, const _Float16 *b, int m, int n, int k, int shape);
// defined in pto_gemm_mxw4_<width>.hip (MXFP8 / MXFP4 on the four-wave engine: tiles of 256 x width);
// PTO_ERR_UNSUPPORTED unless m >= 256, n >= width, n % 4 == 0, k % 512 == 0 (fp4, format 4: k % 1024 == 0)
int gemm_mx_w4_96(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                  int format, int c_fp32);
int gemm_mx_w4_128(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                   int format, int c_fp32);
int gemm_mx_w4_160(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                   int format, int c_fp32);
int gemm_mx_w4_192(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                   int format, int c_fp32);
int gemm_mx_w4_224(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                   int format, int c_fp32);
int gemm_mx_w4_256(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                   int format, int c_fp32);
inline int gemm_mx_w4(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                      int format, int c_fp32, int width)
{
    switch (width) {
    case 96: return gemm_mx_w4_96(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
    case 128: return gemm_mx_w4_128(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
    case 160: return gemm_mx_w4_160(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
    case 192: return gemm_mx_w4_192(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
    case 224: return gemm_mx_w4_224(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
    case 256: return gemm_mx_w4_256(st, c, a, b, sa, sb, m, n, k, format, c_fp32);
    default: return PTO_ERR_UNSUPPORTED;
    }
}
// defined in pto_gemm_mxks.hip (MXFP8 / MXFP4 tiles with k split over two groups of wavefronts); shape 0 .. 5 = 64 x 64, 64 x 128,
// 128 x 64, 128 x 128, 128 x 192, 192 x 128 on eight wavefronts, 6 = 32 x 32 on two, 7 = 32 x 64 on four.  PTO_ERR_UNSUPPORTED unless
// n % 4 == 0 and k % 512 == 0
int gemm_mx_ks(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
               int format, int c_fp32, int shape);
// defined in pto_fa_w8.hip (head_dim 128, workgroups of eight wavefronts = 256 queries, two groups of four waves in
// opposite MFMA / softmax phases)
int fa_fwd_d128_w8(hipStream_t st, void *o, float *lse, const _Float16 *q, const _Float16 *k, const _Float16 *v, int batch, int heads,
                   int seqQ, int seqKv, bool causal, bool oFp32, int causalOff);
// defined in pto_fa_split.hip: the keys of a query block split over two, four or eight groups of a workgroup's eight wavefronts
int fa_fwd_split(hipStream_t st, void *o, float *lse, const _Float16 *q, const _Float16 *k, const _Float16 *v, int batch, int heads,
                 int seqQ, int seqKv, int headDim, bool causal, bool oFp32, int causalOff, int groups);
// defined in pto_fa_w8m16.hip: the schedule of fa_fwd_d128_w8 on v_mfma_f32_16x16x32_f16
int fa_fwd_d128_w8m16(hipStream_t st, void *o, float *lse, const _Float16 *q, const _Float16 *k, const _Float16 *v, int batch, int heads,
                      int seqQ, int seqKv, bool causal, bool oFp32, int causalOff);
} // namespace pto_amd
