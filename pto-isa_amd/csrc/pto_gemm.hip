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
//   time = fixed + per_round more + (k / 64) (step + step_round more + step_share share) + per_mb (megabytes of C),
// more = rounds - 1, share of the units busy in the last round, in microseconds, launch included.  The figures are
// least-squares fits to 330 problems between 128 x 128 x 256 and 6144 x 6144 x 6144, three operand sets in turn (root mean
// square of the relative error 4 .. 6 %).  The k-split shapes are taken 6 % dearer than fitted: where the two kinds come out
// even, the four-wave tiles stay (without it 5768 x 500 x 256 ran 8 % and 3 of 330 problems over 2 % longer than on four-wave
// tiles alone, with it 1 of 330); so chosen, a problem is 0.1 % from its best shape on average.  What the figures say: a small
// tile's step is cheap and moves more bytes per flop (64 x 64: 0.17 us a step, 128 x 128: 0.34, the four-wave 256 x 192: 0.67),
// so it wins while it puts more compute units to work -- 512^3 8.9 us on six 192 x 128 tiles, 4.1 on 32 x 64 ones; 1024^3 13.7
// and 6.8; 128 x 4096 x 4096 68 and 13; 768 x 768 x 6144 48 and 20 -- and the tiles of 192 and 256 rows win from about one
// whole round of them on (2048^3 24 against 21 on 128 x 128, 4096^3 106 against 142 on 192 x 128).
struct TileShape {
    enum Kernel { kW4, kKs, kBlock } kernel;
    int number, bm, bn;
    double fixed, perRound, step, stepRound, perMb, stepShare;
};
constexpr TileShape kShapes[] = {
    {TileShape::kW4, 0, 256, 256, 8.66, 3.98, 0.888, 1.402, 0.112, 0.336}, {TileShape::kW4, 1, 256, 192, 6.82, 2.09, 0.672, 1.070, 0.126, 0.286},
    {TileShape::kW4, 2, 256, 128, 4.99, 1.25, 0.520, 0.744, 0.171, 0.103}, {TileShape::kW4, 3, 192, 256, 7.05, 2.80, 0.674, 1.078, 0.114, 0.302},
    {TileShape::kW4, 4, 192, 192, 5.77, 2.47, 0.524, 0.818, 0.135, 0.197}, {TileShape::kW4, 5, 192, 128, 4.04, 0.99, 0.434, 0.611, 0.180, 0.103},
    {TileShape::kKs, 0, 32, 64, 2.70, 0.69, 0.134, 0.139, 0.194, 0.022},   {TileShape::kKs, 1, 64, 64, 2.67, 0.59, 0.166, 0.169, 0.189, 0.030},
    {TileShape::kKs, 2, 64, 96, 2.91, 0.52, 0.224, 0.239, 0.207, 0.031},   {TileShape::kKs, 3, 128, 64, 2.63, 0.01, 0.286, 0.259, 0.252, 0.028},
    {TileShape::kKs, 4, 128, 96, 4.00, 1.67, 0.315, 0.372, 0.202, 0.038},  {TileShape::kKs, 5, 128, 128, 4.38, 1.62, 0.340, 0.441, 0.186, 0.066},
    {TileShape::kKs, 6, 192, 128, 5.58, 2.65, 0.441, 0.622, 0.159, 0.118}, {TileShape::kKs, 7, 256, 128, 6.25, 2.69, 0.572, 0.788, 0.153, 0.128},
    {TileShape::kKs, 8, 192, 192, 6.74, 3.26, 0.642, 0.863, 0.144, 0.139},
    // the 128 x 256 block written with the tile instructions: 2048 x 6144 x 1056 38 us against 44 on 256 x 128
    {TileShape::kBlock, 0, 128, 256, 3.03, 0.00, 1.000, 0.750, 0.161, 0.000},
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
        const double more = (double)((tiles - 1) / cus), share = (double)((tiles - 1) % cus + 1) / cus, steps = (k + 63) / 64;
        const double time = (s.fixed + s.perRound * more + steps * (s.step + s.stepRound * more + s.stepShare * share) + s.perMb * (4e-6 * m * n)) *
                            (s.kernel == TileShape::kKs ? 1.06 : 1.0);
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
