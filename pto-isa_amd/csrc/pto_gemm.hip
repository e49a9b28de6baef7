// fp16 x fp16 -> fp32 GEMM for MI355X written with PTO tile instructions:
//   TLOAD (HBM -> LDS, async 16-byte copies)  ->  TEXTRACT (LDS -> MFMA operand fragments)
//   ->  TMATMUL / TMATMUL_ACC (v_mfma_f32_32x32x16_f16)  ->  TSTORE (accumulators -> HBM);
// and the entry point that picks among it and the kernels of pto_gemm_w4.hip and pto_gemm_ks.hip.
//
// Same decomposition as the reference's manual kernel
// (kernels/manual/a2a3/gemm_performance/gemm_performance_kernel.cpp:67-230): each "core" owns
// BM x BN blocks of C, walks K in steps of BK, double-buffers the staged A / B panels and
// synchronises the stages with set_flag / wait_flag.  Differences that the hardware asks for:
// the stages are software-pipelined in program order (one instruction stream per wavefront: the
// TLOAD of step i+1 is issued before the TEXTRACT / TMATMUL of step i), one workgroup per C block
// instead of a 24-core loop nest, and an XCD-aware block -> tile map.
#include "gemm_kernels.hpp"

#if defined(PTO_ST_HOOKS)
// Tuning hook (not part of the public header): the same GEMM with another tiling / pipeline depth.
extern "C" int pto_gemm_f16f32_variant(void *stream, float *c, const uint16_t *a, const uint16_t *b, int m, int n, int k,
                                       int variant)
{
    if (!c || !a || !b || m <= 0 || n <= 0 || k <= 0)
        return PTO_ERR_BAD_ARG;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const half *ha = reinterpret_cast<const half *>(a), *hb = reinterpret_cast<const half *>(b);
    switch (variant) {
    case 0: return launch_gemm<128, 256, 64, 2, 1, 8>(st, c, ha, hb, m, n, k);
    case 1: return launch_gemm<128, 256, 32, 2, 2, 8>(st, c, ha, hb, m, n, k);
    case 2: return launch_gemm<128, 256, 32, 3, 2, 8>(st, c, ha, hb, m, n, k);
    case 3: return launch_gemm<128, 256, 64, 3, 1, 8>(st, c, ha, hb, m, n, k);
    case 4: return launch_gemm<128, 256, 32, 4, 2, 8>(st, c, ha, hb, m, n, k);
    case 5: return launch_gemm<128, 256, 32, 3, 2, 4>(st, c, ha, hb, m, n, k);
    case 6: return launch_gemm<128, 256, 32, 3, 2, 16>(st, c, ha, hb, m, n, k);
    case 7: return launch_gemm<256, 256, 32, 4, 1, 8>(st, c, ha, hb, m, n, k);
    case 8: return launch_gemm<256, 256, 64, 2, 1, 8>(st, c, ha, hb, m, n, k);
    case 9: return launch_gemm<256, 256, 32, 3, 1, 8>(st, c, ha, hb, m, n, k);
    case 10: return launch_gemm<256, 256, 32, 4, 1, 4>(st, c, ha, hb, m, n, k);
    case 11: return launch_gemm<256, 256, 32, 2, 1, 8>(st, c, ha, hb, m, n, k);
    default: return PTO_ERR_BAD_ARG;
    }
}
#endif // PTO_ST_HOOKS

namespace {
// What a problem takes with one tile shape: tiles are dealt to the compute units, `rounds` of them to the busiest one, and
//   time = fixed + per_round (rounds - 1) + (k / 64) (step + step_round (rounds - 1)) + per_mb (megabytes of C)
// in microseconds, launch included.  The figures are least-squares fits to 150 problems between 128 x 128 x 256 and
// 6144 x 6144 x 6144, three operand sets in turn (root mean square of the relative error 4 .. 7 %); the choice they give was
// within 1 % of the best shape on average, and at worst the next best one.  What they say: a small tile's step is cheap and
// moves more bytes per flop (64 x 64: 0.16 us a step, 128 x 128: 0.34, the four-wave 256 x 192: 0.70), so it wins while it
// puts more compute units to work -- 512^3 8.9 us on six 192 x 128 tiles, 4.4 on 32 x 64 ones; 1024^3 13.7 and 6.8;
// 128 x 4096 x 4096 68 and 13; 768 x 768 x 6144 48 and 20 -- and the tiles of 192 and 256 rows win from about one whole round of
// them on (2048^3 24 against 21 on 128 x 128, 4096^3 106 against 142 on 192 x 128).
struct TileShape {
    enum Kernel { kW4, kKs, kBlock } kernel;
    int number, bm, bn;
    double fixed, perRound, step, stepRound, perMb;
};
constexpr TileShape kShapes[] = {
    {TileShape::kW4, 0, 256, 256, 8.53, 8.73, 0.918, 0.996, 0.152}, {TileShape::kW4, 1, 256, 192, 6.86, 1.26, 0.699, 0.982, 0.194},
    {TileShape::kW4, 2, 256, 128, 5.16, 1.36, 0.528, 0.701, 0.220}, {TileShape::kW4, 3, 192, 256, 6.82, 2.40, 0.709, 1.070, 0.179},
    {TileShape::kW4, 4, 192, 192, 5.90, 2.17, 0.542, 0.863, 0.177}, {TileShape::kW4, 5, 192, 128, 4.10, 0.00, 0.447, 0.630, 0.245},
    {TileShape::kKs, 0, 32, 64, 2.94, 0.29, 0.137, 0.142, 0.341},   {TileShape::kKs, 1, 64, 64, 2.89, 0.10, 0.165, 0.183, 0.284},
    {TileShape::kKs, 2, 64, 96, 3.04, 0.00, 0.229, 0.251, 0.286},   {TileShape::kKs, 3, 128, 64, 2.92, 0.00, 0.278, 0.260, 0.264},
    {TileShape::kKs, 4, 128, 96, 4.09, 0.65, 0.312, 0.391, 0.266},  {TileShape::kKs, 5, 128, 128, 4.47, 0.66, 0.342, 0.469, 0.242},
    {TileShape::kKs, 6, 192, 128, 5.61, 0.93, 0.450, 0.667, 0.237}, {TileShape::kKs, 7, 256, 128, 6.40, 2.29, 0.580, 0.751, 0.195},
    {TileShape::kKs, 8, 192, 192, 6.83, 2.62, 0.652, 0.852, 0.178},
    // the 128 x 256 block written with the tile instructions: 2048 x 6144 x 1056 38 us against 44 on 256 x 128
    {TileShape::kBlock, 0, 128, 256, 3.03, 0.00, 1.000, 0.750, 0.161},
};
} // namespace

extern "C" int pto_gemm_f16f32(void *stream, float *c, const uint16_t *a, const uint16_t *b, int m, int n, int k)
{
    if (!c || !a || !b || m <= 0 || n <= 0 || k <= 0)
        return PTO_ERR_BAD_ARG;
    const bool blocks = m % 128 == 0 && n % 256 == 0 && k % 32 == 0;
    if (!blocks && !(m >= 192 && n >= 128 && n % 4 == 0 && k % 128 == 0))
        return PTO_ERR_UNSUPPORTED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const half *ha = reinterpret_cast<const half *>(a), *hb = reinterpret_cast<const half *>(b);
    const int cus = compute_units();
    const TileShape *best = nullptr;
    double bestTime = 0.0;
    for (const TileShape &s : kShapes) {
        if ((s.kernel == TileShape::kW4 && (m < s.bm || n < s.bn || k % 128)) || (s.kernel == TileShape::kBlock && !blocks))
            continue;
        const long long tiles = (long long)((m + s.bm - 1) / s.bm) * ((n + s.bn - 1) / s.bn);
        const double more = (double)((tiles - 1) / cus), steps = (k + 63) / 64;
        const double time = s.fixed + s.perRound * more + steps * (s.step + s.stepRound * more) + s.perMb * (4e-6 * m * n);
        if (best == nullptr || time < bestTime) {
            best = &s;
            bestTime = time;
        }
    }
    switch (best->kernel) {
    case TileShape::kW4: return pto_amd::gemm_f16f32_w4(st, c, ha, hb, m, n, k, best->number);
    case TileShape::kKs: return pto_amd::gemm_f16f32_ks(st, c, ha, hb, m, n, k, best->number);
    default: return launch_gemm<128, 256, 32, 3, 2, 8>(st, c, ha, hb, m, n, k);
    }
}
