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
// more = rounds - 1, share of the units busy in the last round, in microseconds, launch included; the k-split tiles take 6 %
// longer where k ends in half a step.  The figures are least-squares fits to 2293 problems (128 x 128 x 128 .. 6144^3 ragged,
// .. 16384 x 8192 x 8192 in whole tiles, three operand sets in turn) in which those near a shape's best use count most (root
// mean square of the relative error there 3 .. 6 %).  The k-split shapes are taken 3 %, the 128 x 256 block 2 % dearer than
// fitted: where they and the four-wave tiles come out even, the latter stay.  So chosen, a problem is 0.15 % from its best
// shape on average (21 % at worst) and 12 of the 2293 are over 2 % slower than with four-wave tiles (k a multiple of 128)
// or blocks alone, the worst 7.6 % (with a fit to 330 problems that counted every one alike: 24 of 1893, and 12.4 %).  What the figures say: a
// small tile's step is cheap and moves more bytes per flop (64 x 64: 0.2 us a step, 128 x 128: 0.45, the four-wave 256 x 192:
// 1.1), so it wins while it puts more compute units to work -- 512^3 8.9 us on twelve 192 x 128 tiles, 3.8 on 32 x 64 ones, 3.3 on 32 x 32;
// 1024^3 13.7 and 6.8; 128 x 4096 x 4096 68 and 12; 768 x 768 x 6144 48 and 20 -- and the tiles of 192 and 256 rows win from
// about one whole round of them on (2048^3 22.7 against 21.0 on 128 x 128, 4096^3 104 against 137 on 192 x 128).
struct TileShape {
    enum Kernel { kW4, kKs, kBlock } kernel;
    int number, bm, bn;
    double fixed, perRound, step, stepRound, perMb, stepShare;
};
// (small tiles first: for a small problem, whose call the host bounds, the choice is then the first shape's time and lower bounds of the others)
constexpr TileShape kShapes[] = {
    // 32 x 32, fitted to 400 problems of up to 900 such tiles: it is the shortest where they are one round, and by 8 to 29 % (from a graph 512^3 3.76 -> 3.29 us,
    // 512 x 512 x 2048 7.4 -> 6.0, 256 x 256 x 6144 15.8 -> 11.5, 300 x 700 x 1024 4.70 -> 4.14), and never where they are two (640 x 512 x 1024 4.8 / 5.4)
    {TileShape::kKs, 9, 32, 32, 2.487, 0.411, 0.091, 0.076, 0.159, 0.017},
    {TileShape::kKs, 0, 32, 64, 2.670, 0.853, 0.135, 0.136, 0.178, 0.026},   {TileShape::kKs, 1, 64, 64, 2.822, 0.902, 0.152, 0.165, 0.175, 0.044},
    {TileShape::kKs, 2, 64, 96, 3.214, 0.965, 0.207, 0.240, 0.183, 0.052},   {TileShape::kKs, 3, 128, 64, 3.221, 0.868, 0.249, 0.258, 0.180, 0.080},
    {TileShape::kKs, 4, 128, 96, 4.595, 2.050, 0.258, 0.411, 0.162, 0.127},  {TileShape::kKs, 5, 128, 128, 5.026, 2.036, 0.293, 0.488, 0.140, 0.156},
    {TileShape::kKs, 6, 192, 128, 6.565, 2.833, 0.384, 0.682, 0.109, 0.218}, {TileShape::kKs, 7, 256, 128, 7.789, 4.862, 0.468, 0.875, 0.072, 0.314},
    {TileShape::kKs, 8, 192, 192, 8.656, 5.901, 0.502, 0.952, 0.058, 0.342},
    {TileShape::kW4, 0, 256, 256, 9.263, 7.420, 0.770, 1.429, 0.085, 0.610}, {TileShape::kW4, 1, 256, 192, 8.193, 6.015, 0.543, 1.115, 0.070, 0.533},
    {TileShape::kW4, 2, 256, 128, 6.567, 3.898, 0.379, 0.817, 0.083, 0.373}, {TileShape::kW4, 3, 192, 256, 7.814, 4.941, 0.581, 1.150, 0.084, 0.490},
    {TileShape::kW4, 4, 192, 192, 7.134, 4.643, 0.393, 0.916, 0.072, 0.451}, {TileShape::kW4, 5, 192, 128, 4.741, 1.197, 0.337, 0.658, 0.159, 0.242},
    // the 128 x 256 block written with the tile instructions: 2048 x 6144 x 1056 37 us against 44 on 256 x 128
    {TileShape::kBlock, 0, 128, 256, 3.292, 0.364, 0.919, 0.820, 0.114, 0.161},
};
struct GemmChoice {
    int m, n, k, cus;
    bool blocks;
    double steps = (k + 63) / 64, megabytes = 4e-6 * m * n, ksFactor = k % 64 ? 1.03 * 1.06 : 1.03;
    bool Takes(const TileShape &s) const { return s.kernel == TileShape::kKs || (s.kernel == TileShape::kW4 ? m >= s.bm && n >= s.bn && k % 128 == 0 : blocks); }
    double Factor(const TileShape &s) const { return s.kernel == TileShape::kW4 ? 1.0 : s.kernel == TileShape::kKs ? ksFactor : 1.02; }
    double AtLeast(const TileShape &s) const { return (s.fixed + steps * s.step) * Factor(s); } // (every figure of a shape is positive)
    double Time(const TileShape &s) const
    {
        const long long tiles = (long long)((m + s.bm - 1) / s.bm) * ((n + s.bn - 1) / s.bn);
        const double more = (double)((tiles - 1) / cus), share = (double)((tiles - 1) % cus + 1) / cus;
        return (s.fixed + s.perRound * more + steps * (s.step + s.stepRound * more + s.stepShare * share) + s.perMb * megabytes) * Factor(s);
    }
    // (a shape is passed over that could not win in one round of full speed: 512^3 37 ns of the call's 3.9 us instead of 113, 1000 x 3000 x 2048 92, 6144^3 145)
    const TileShape &Best() const
    {
        const TileShape *best = &kShapes[0]; // (a k-split one: any problem)
        double bestTime = Time(*best);
        for (const TileShape &s : kShapes) {
            if (&s == &kShapes[0] || !Takes(s) || AtLeast(s) >= bestTime)
                continue;
            const double time = Time(s);
            if (time < bestTime) {
                best = &s;
                bestTime = time;
            }
        }
        return *best;
    }
};
static_assert(kShapes[0].kernel == TileShape::kKs, "the first shape takes any problem");
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
    const TileShape &best = GemmChoice{m, n, k, pto_amd::compute_units(), blocks}.Best();
    switch (best.kernel) {
    case TileShape::kW4: return pto_amd::gemm_f16f32_w4(st, c, ha, hb, m, n, k, best.number);
    case TileShape::kKs: return pto_amd::gemm_f16f32_ks(st, c, ha, hb, m, n, k, best.number);
    default: return launch_gemm<128, 256, 32, 3, 2, 8>(st, c, ha, hb, m, n, k);
    }
}

#if defined(PTO_ST_HOOKS)
// The choice among the shapes without a launch (needs no device): the number of the shape that the entry point takes on `units` compute units; expected: the
// time of each shape, an infinity where it does not take the problem.  PTO_ERR_UNSUPPORTED as the entry point.
extern "C" int pto_gemm_f16f32_choice(int m, int n, int k, int units, double *expected)
{
    const bool blocks = m % 128 == 0 && n % 256 == 0 && k % 32 == 0;
    if (m <= 0 || n <= 0 || k <= 0 || units <= 0)
        return PTO_ERR_BAD_ARG;
    if (!blocks && !(m >= 192 && n >= 128 && n % 4 == 0 && k % 128 == 0))
        return PTO_ERR_UNSUPPORTED;
    const GemmChoice choice{m, n, k, units, blocks};
    for (const TileShape &s : kShapes)
        if (expected != nullptr)
            expected[&s - kShapes] = choice.Takes(s) ? choice.Time(s) : __builtin_inf();
    return (int)(&choice.Best() - kShapes);
}
#endif
