// MXFP8 / MXFP4 GEMM tiles of 32 .. 192 rows for problems that the 256-row tiles of gemm_kernels_mxw4.hpp leave compute units
// idle on: the kernel of gemm_kernels_ks.hpp (eight wavefronts in a 2 x 2 x 2 grid, rows x columns x k) on MX operands.  A
// K-step is again 128 bytes of every row; group g multiplies bytes 64 g .. 64 g + 63 of them: one v_mfma_scale_f32_32x32x64
// (fp8: 64 k, 16 passes) or two (fp4: 128 k, 8 passes each) per 32 x 32 block.  Copies, stages and the meeting of the two
// partial sums are those of the fp16 kernel.
//
// 32 x 32 tiles are two wavefronts, one for each half of k, and 32 x 64 ones four: a unit's copies bound a step, so products of few tiles gain by
// smaller ones on more units.  To bf16, launched from a graph, the same operands each time; thirty sets of them in turn: 64 x 64 -> 32 x 32, 512^3 fp8 3.60 -> 2.86 us; 4.0 -> 3.2,
// fp4 3.40 -> 2.78; 3.6 -> 2.95, 256 x 256 x 6144 8.8 -> 6.3; 13.0 -> 9.3, fp4 7.5 -> 5.7; 9.0 -> 6.6; 64 x 64 -> 32 x 64, 256 x 1536 x 2048 5.1 -> 4.2; 6.4 -> 5.5, fp4
// 4.6 -> 3.9; 5.3 -> 4.4.  (Called one by one 512^3 takes 4.1 on either: the host.)  Six and eight stages for them: 512 x 512 x 2048 fp8 4.51 -> 5.03 and 5.16, only from k = 4096 on up to 11 % faster.
//
// Scales.  32 bytes of a row's scales last P = 8 steps (fp8) or 4 (fp4); they come into one of two LDS buffers with one or two
// copy instructions per wave and period (two lanes per row), a period ahead.  A lane's MFMA operand needs the scale of its own
// 32 k: every Q = P / 2 steps it reads 16 bytes of its row's scales with the fragments and shifts the byte (fp4, whose chunks are
// dealt so that they are neighbours: the two bytes) of the step down.  A row's two 16-byte halves change places every eight
// rows, so that these reads touch every bank once.  (One ds_read_u8 per block and step instead: eight clocks each, rows 32 bytes
// apart meet in four of the 32 banks that a 4-byte read sees; 128 x 128 tiles 25 % slower.)
//
// What bounds a step: the copies, as in the fp16 kernel.  One 64 x 64 tile takes 0.16 us a step, 64 x 128 0.24, 128 x 128 0.37,
// 128 x 192 0.52: 79 to 102 bytes per ns and compute unit, where its MFMAs take 0.05, 0.11, 0.21, 0.32.
// fp8 to fp32, the same operands each time, 256 x 128 tiles on four wavefronts / the best of these: 512^3 9.4 / 2.9 us, 256 x 256 x 6144 29.8 / 6.3,
// 2048^3 15.1 / 11.7 (128 x 128); 3072^3 stays on 256 x 192 tiles (31 against 40).
//
// The way out: bf16 by the hardware conversion (the integer form was 7 instructions an element), 16 bytes a lane, 64 bytes of a row to a
// store instruction, past the L2 where that pays (store_through): 2048 x 2048 x 1024 to bf16 11.1 -> 8.6 us in fp8, 9.1 -> 6.7 in
// fp4, to fp32 11.8 -> 9.6 and 9.9 -> 7.7.
#pragma once
#include "gemm_kernels_ks.hpp"

#include <type_traits>

PTO_DEVICE_CODE_BEGIN
namespace {

// the reads into a set of fragments (and of scales) are over (as KsArrived)
template <int MB, int NB>
PTO_DEV void MxKsArrived(ks_f16x8 (&a)[MB][2], ks_f16x8 (&b)[NB][2], ks_f16x8 (&scales)[MB + NB])
{
    KsWaitLds();
#pragma unroll
    for (int i = 0; i < NB; ++i)
        asm volatile("" : "+v"(b[i][0]), "+v"(b[i][1]));
#pragma unroll
    for (int i = 0; i < MB; ++i)
        asm volatile("" : "+v"(a[i][0]), "+v"(a[i][1]));
#pragma unroll
    for (int i = 0; i < MB + NB; ++i)
        asm volatile("" : "+v"(scales[i]));
}

template <int BM, int BN, int S>
constexpr int MxKsLdsBytes() // S stages of 128-byte rows, two buffers of 32 scale bytes per row; the partial sums afterwards
{
    constexpr int stages = S * (BM + BN) * 128 + 2 * (BM + BN) * 32, sums = BM * BN * (int)sizeof(float);
    return stages > sums ? stages : sums;
}

// wavefronts of a tile: at most two by two of 32 rows and columns and more, times two groups of k
constexpr int MxKsGrid(int extent) { return extent < 64 ? 1 : 2; }
constexpr int MxKsWaves(int bm, int bn) { return 2 * MxKsGrid(bm) * MxKsGrid(bn); }

// FMT: 0 = e4m3, 1 = e5m2, 4 = e2m1 (both operands then); ld = bytes of a row of A and B, ldScale = of their scales
template <int FMT_A, int FMT_B, typename OutT, int BM, int BN, int S, int MIN_WAVES, int GROUP_M>
__global__ __launch_bounds__(64 * MxKsWaves(BM, BN), MIN_WAVES) AICORE
    void GemmMxKs(__gm__ OutT *out, __gm__ const uint8_t *src0, __gm__ const uint8_t *src1, __gm__ const uint8_t *scale0,
                  __gm__ const uint8_t *scale1, int m, int n, uint32_t ld, uint32_t ldScale, int through)
{
    constexpr bool FP4 = FMT_A == 4;
    static_assert((FMT_A == 4) == (FMT_B == 4), "fp4 with fp4");
    constexpr int WM = MxKsGrid(BM), WN = MxKsGrid(BN), kWaves = MxKsWaves(BM, BN);
    constexpr int MB = BM / WM / 32, NB = BN / WN / 32;                           // 32 x 32 blocks of a wave
    constexpr int kInst = (BM + BN) / 8, kCopies = (kInst + kWaves - 1) / kWaves; // copy instructions of 8 rows a step; per wave
    constexpr int kScaleInst = (BM + BN) / 32, kScaleCopies = (kScaleInst + kWaves - 1) / kWaves; // of 32 rows' scales a period; per wave
    constexpr int kStepScales = FP4 ? 8 : 4, P = 32 / kStepScales;  // scale bytes of a row and step; steps of a period
    constexpr uint32_t kStage = (BM + BN) * 128, kRing = S * kStage, kScaleBuf = (BM + BN) * 32;
    // (S <= P: the wait for step it + P at the top of step it + P - 1 then covers the scales issued in step it)
    static_assert(BM % (32 * WM) == 0 && BN % (32 * WN) == 0 && S >= 3 && S <= P, "tile shape");

    int tm, tn;
    TileOfBlock<GROUP_M>((int)blockIdx.x, (m + BM - 1) / BM, (n + BN - 1) / BN, tm, tn);
    const int row0 = tm * BM, col0 = tn * BN;
    const int wave = hw::wave(), group = wave / (WM * WN), wm = wave / WN % WM, wn = wave % WN;
    const uint32_t lane = (uint32_t)hw::lane();
    const uint32_t ldsBase = (uint32_t)(uintptr_t)hw::lds_base();
    const int steps = (int)(ld / 128); // a multiple of Q

    // the copies of a step: as in gemm_kernels_ks.hpp (rows past m, columns past n repeat the last one)
    const char *base[kCopies];
    uint32_t off[kCopies], lds[kCopies];
#pragma unroll
    for (int j = 0; j < kCopies; ++j) {
        const int i = kWaves * j + wave < kInst ? kWaves * j + wave : kInst - 1;
        const bool isA = i < BM / 8;
        const int first = isA ? row0 + 8 * i : col0 + 8 * (i - BM / 8), last = (isA ? m : n) - 1;
        const int row = first + (int)(lane / 8) < last ? first + (int)(lane / 8) : last;
        const int origin = first < last ? first : last;
        const uint32_t chunk = (lane % 8) ^ ((4u * (uint32_t)i + lane / 16) % 8);
        base[j] = detail::uniform_ptr(reinterpret_cast<const char *>(isA ? src0 : src1) + (int64_t)origin * ld);
        off[j] = (uint32_t)(row - origin) * ld + chunk * 16u;
        lds[j] = ldsBase + (uint32_t)i * 1024u;
    }
    auto copyOne = [&](int j, int step, uint32_t stageOff) __attribute__((always_inline)) {
        const int s = step < steps ? step : steps - 1; // (past the end: the last step again, into a stage nobody reads)
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds[j] + stageOff), "v"(off[j]), "s"(base[j] + (int64_t)s * 128) : "memory");
    };
    // Scales of a period: instruction i covers 32 rows, lane l the 16 bytes (l % 2) ^ (l / 16) % 2 of row l / 2 (past the end of
    // the row, whose scales are a multiple of 16 bytes: its last 16, which nobody uses).
    const char *scaleBase[kScaleCopies];
    uint32_t scaleOff[kScaleCopies], scaleLds[kScaleCopies];
    const uint32_t scaleChunk = ((lane % 2) ^ (lane / 16 % 2)) * 16u;
#pragma unroll
    for (int j = 0; j < kScaleCopies; ++j) {
        const int i = (kWaves * j + wave) % kScaleInst;
        const bool isA = i < BM / 32;
        const int first = isA ? row0 + 32 * i : col0 + 32 * (i - BM / 32), last = (isA ? m : n) - 1;
        const int row = first + (int)(lane / 2) < last ? first + (int)(lane / 2) : last;
        const int origin = first < last ? first : last;
        scaleBase[j] = detail::uniform_ptr(reinterpret_cast<const char *>(isA ? scale0 : scale1) + (int64_t)origin * ldScale);
        scaleOff[j] = (uint32_t)(row - origin) * ldScale;
        scaleLds[j] = ldsBase + kRing + (uint32_t)i * 1024u;
    }
    auto copyScales = [&](int period) __attribute__((always_inline)) {
        const uint32_t at = (uint32_t)period * 32u + scaleChunk, atIn = at < ldScale - 16u ? at : ldScale - 16u;
#pragma unroll
        for (int j = 0; j < kScaleCopies; ++j)
            asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(scaleLds[j] + (uint32_t)(period & 1) * kScaleBuf), "v"(scaleOff[j] + atIn),
                         "s"(scaleBase[j])
                         : "memory");
    };

    // Fragment reads: lane l holds row l % 32 of a block; its half h = l / 32 holds, of the group's 64 bytes, the 16-byte chunks
    // h and 2 + h (fp8: the operand of one MFMA, k block h of its two), or 2 h and 2 h + 1 (fp4: the operands of two MFMAs).
    const uint32_t r32 = lane % 32, h = lane / 32;
    uint32_t aAddr[2], bAddr[2];
#pragma unroll
    for (int q = 0; q < 2; ++q) {
        const uint32_t chunk = (uint32_t)group * 4u + (FP4 ? 2u * h + (uint32_t)q : h + 2u * (uint32_t)q);
        const uint32_t fragOff = r32 * 128u + ((chunk ^ ((r32 / 2) % 8)) * 16u);
        aAddr[q] = ldsBase + (uint32_t)(wm * (BM / WM)) * 128u + fragOff;
        bAddr[q] = ldsBase + (uint32_t)(BM + wn * (BN / WN)) * 128u + fragOff;
    }
    // The 16 scale bytes of a row that last Q steps (4 of fp8, 2 of fp4) come into registers with one read per block; those of
    // step t among them are bytes 4 t + 2 group + h (fp8), 8 t + 4 group + 2 h and the next (fp4).
    constexpr int Q = P / 2;
    const uint32_t scaleLane = r32 * 32u + ((r32 / 8) % 2) * 16u;
    const uint32_t scaleShift = FP4 ? 32u * (uint32_t)group + 16u * h : 16u * (uint32_t)group + 8u * h;

    ks_f16x8 a[2][MB][2], b[2][NB][2], scales[MB + NB];
    uint32_t sa[MB], sb[NB];
    auto readStep = [&](auto setTag, uint32_t stageOff) __attribute__((always_inline)) {
        constexpr int set = decltype(setTag)::value;
        StaticFor<0, NB>([&](auto i) __attribute__((always_inline)) {
            constexpr int I = decltype(i)::value;
            b[set][I][0] = KsLdsRead16<I * 4096>(bAddr[0] + stageOff);
            b[set][I][1] = KsLdsRead16<I * 4096>(bAddr[1] + stageOff);
        });
        StaticFor<0, MB>([&](auto i) __attribute__((always_inline)) {
            constexpr int I = decltype(i)::value;
            a[set][I][0] = KsLdsRead16<I * 4096>(aAddr[0] + stageOff);
            a[set][I][1] = KsLdsRead16<I * 4096>(aAddr[1] + stageOff);
        });
    };
    auto readScales = [&](int it) __attribute__((always_inline)) { // of steps it .. it + Q - 1
        const uint32_t addr = (scaleLane ^ (uint32_t)((it / Q % 2) * 16)) + ldsBase + kRing + (uint32_t)((it / P) & 1) * kScaleBuf;
        const uint32_t saAddr = addr + (uint32_t)(wm * (BM / WM)) * 32u, sbAddr = addr + (uint32_t)(BM + wn * (BN / WN)) * 32u;
        StaticFor<0, NB>([&](auto i) __attribute__((always_inline)) { scales[MB + decltype(i)::value] = KsLdsRead16<decltype(i)::value * 1024>(sbAddr); });
        StaticFor<0, MB>([&](auto i) __attribute__((always_inline)) { scales[decltype(i)::value] = KsLdsRead16<decltype(i)::value * 1024>(saAddr); });
    };
    auto pick = [&](auto tTag, const ks_f16x8 &s) __attribute__((always_inline)) { // this lane's scales of step t, from byte 0
        constexpr int t = decltype(tTag)::value;
        const u32x4 w = __builtin_bit_cast(u32x4, s);
        if constexpr (FP4)
            return (uint32_t)((((uint64_t)w[2 * t + 1] << 32) | w[2 * t]) >> scaleShift);
        else
            return w[t] >> scaleShift;
    };
    auto whole = [](const ks_f16x8 (&p)[2]) __attribute__((always_inline)) {
        const u32x4 lo = __builtin_bit_cast(u32x4, p[0]), hi = __builtin_bit_cast(u32x4, p[1]);
        return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    };
    typedef float f32x16_ks __attribute__((ext_vector_type(16)));
    f32x16_ks acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
            for (int v = 0; v < 16; ++v)
                acc[i][j][v] = 0.0f;

    uint32_t readOff = kStage, copyOff = 0; // of step it + 1, of step it (and it + S)
    copyScales(0);
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int j = 0; j < kCopies; ++j)
            copyOne(j, s, s * kStage);
    hw::wait_vm<(S - 1) * kCopies>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory"); // (the barrier alone does not hold loads back from moving ahead of it)
    readStep(std::integral_constant<int, 0>(), 0u);
    readScales(0);
    MxKsArrived(a[0], b[0], scales);

    auto step = [&](auto tTag, int it) __attribute__((always_inline)) { // t = it % Q
        constexpr int t = decltype(tTag)::value, set = t % 2;
#pragma unroll
        for (int i = 0; i < MB; ++i)
            sa[i] = pick(tTag, scales[i]);
#pragma unroll
        for (int j = 0; j < NB; ++j)
            sb[j] = pick(tTag, scales[MB + j]);
        // this wave has read all of step it, its copies of step it + 1 have landed; behind the barrier that is so of every wave
        // (scale copies among the younger ones only make the wait stricter)
        hw::wait_vm<(S - 2) * kCopies>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        readStep(std::integral_constant<int, 1 - set>(), readOff);
        if constexpr (t == Q - 1)
            readScales(it + 1);
        if (t == 0 && it % P == 0) // the next period's, into the buffer of the one before
            copyScales(it / P + 1);
        __builtin_amdgcn_sched_barrier(0);
        StaticFor<0, MB * NB>([&](auto qTag) __attribute__((always_inline)) {
            constexpr int q = decltype(qTag)::value, i = q / NB, j = q % NB;
            if constexpr (FP4) {
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(detail::mx_operand(__builtin_bit_cast(u32x4, b[set][j][0])),
                                                                            detail::mx_operand(__builtin_bit_cast(u32x4, a[set][i][0])), acc[i][j],
                                                                            FMT_B, FMT_A, 0, (int)sb[j], 0, (int)sa[i]);
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(detail::mx_operand(__builtin_bit_cast(u32x4, b[set][j][1])),
                                                                            detail::mx_operand(__builtin_bit_cast(u32x4, a[set][i][1])), acc[i][j],
                                                                            FMT_B, FMT_A, 1, (int)sb[j], 1, (int)sa[i]);
            } else {
                acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(whole(b[set][j]), whole(a[set][i]), acc[i][j], FMT_B, FMT_A, 0,
                                                                            (int)sb[j], 0, (int)sa[i]);
            }
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int c = q * kCopies / (MB * NB); c < (q + 1) * kCopies / (MB * NB); ++c)
                copyOne(c, it + S, copyOff);
        });
        copyOff = readOff;
        readOff = readOff + kStage == kRing ? 0u : readOff + kStage;
        __builtin_amdgcn_sched_barrier(0);
        MxKsArrived(a[1 - set], b[1 - set], scales);
    };
    for (int it = 0; it < steps; it += Q)
        StaticFor<0, Q>([&](auto tTag) __attribute__((always_inline)) { step(tTag, it + decltype(tTag)::value); });

    // Partial sums: a group keeps half of its wave's blocks (of a single block half its registers), gives the rest to its partner
    // (same rows and columns, other k) and stores the sums of what it keeps.  In quads of four registers: quad u of block
    // half h is columns 8 u + 4 h .. + 3 of row r32.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the copies past the end
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    char *sums = hw::lds_base();
    const int pair = wave % (WM * WN);
    constexpr int kQuads = MB * NB * 4, kKept = kQuads / 2;
    auto quad = [&](auto qTag) __attribute__((always_inline)) {
        constexpr int idx = decltype(qTag)::value / 4, r = 4 * (decltype(qTag)::value % 4);
        const f32x16_ks &v = acc[idx / NB][idx % NB];
        return ks_f32x4{v[r], v[r + 1], v[r + 2], v[r + 3]};
    };
    StaticFor<0, 2>([&](auto gTag) __attribute__((always_inline)) {
        constexpr int g = decltype(gTag)::value;
        if (group != g) {
            StaticFor<g * kKept, (g + 1) * kKept>([&](auto qTag) __attribute__((always_inline)) {
                *reinterpret_cast<ks_f32x4 *>(sums + ((uint32_t)(pair * kQuads + decltype(qTag)::value) * 64u + lane) * 16u) = quad(qTag);
            });
        }
    });
    __syncthreads();
    auto summed = [&](auto qTag) __attribute__((always_inline)) {
        return quad(qTag) + *reinterpret_cast<const ks_f32x4 *>(sums + ((uint32_t)(pair * kQuads + decltype(qTag)::value) * 64u + lane) * 16u);
    };
    // Two quads side by side change lanes: then a store instruction writes 64 bytes of fp32 of each of 16 rows, or 32 of bf16 (eight columns
    // a lane) of 32 rows, and with the block's other two quads 64 of bf16 of 16 rows.
    const int rowLane = row0 + wm * (BM / WM), colLane = col0 + wn * (BN / WN);
    auto words = [](const ks_f32x4 &v) __attribute__((always_inline)) { return __builtin_bit_cast(Words4, v); };
    StaticFor<0, 2>([&](auto gTag) __attribute__((always_inline)) {
        constexpr int g = decltype(gTag)::value;
        if (group != g)
            return;
        if constexpr (std::is_same_v<OutT, float>) {
            // (one block, past no cache: quads as they lie, 32 bytes of a row; 256 x 256 x 6144 12.2 us, 12.3 with the exchange.  Larger tiles:
            // 2048 x 2044 x 1024 in fp8 12.2 as they lie, 11.6 with it)
            if (kKept == 2 && !through) {
                StaticFor<g * kKept, (g + 1) * kKept>([&](auto qTag) __attribute__((always_inline)) {
                    constexpr int q = decltype(qTag)::value, idx = q / 4;
                    const ks_f32x4 v = summed(qTag);
                    const int row = rowLane + 32 * (idx / NB) + (int)r32, col = colLane + 32 * (idx % NB) + 8 * (q % 4) + 4 * (int)h;
                    if (row < m && col < n) // n % 4 == 0: four columns are inside together
                        StoreFour(out + (int64_t)row * n + col, v, 0);
                });
                return;
            }
            StaticFor<0, kKept / 2>([&](auto tag) __attribute__((always_inline)) {
                constexpr int q = g * kKept + 2 * decltype(tag)::value, idx = q / 4;
                Words4 x = words(summed(std::integral_constant<int, q>())), y = words(summed(std::integral_constant<int, q + 1>()));
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    uint32_t xi = x[i], yi = y[i];
                    SwapRows(xi, yi);
                    x[i] = xi;
                    y[i] = yi;
                }
                const int row = rowLane + 32 * (idx / NB) + (int)(lane % 16), col = colLane + 32 * (idx % NB) + 8 * (q % 4 + (int)(lane / 16 % 2)) + 4 * (int)h;
                if (col < n) {
                    if (row < m)
                        StoreFour(out + (int64_t)row * n + col, __builtin_bit_cast(Four, x), through);
                    if (row + 16 < m)
                        StoreFour(out + (int64_t)(row + 16) * n + col, __builtin_bit_cast(Four, y), through);
                }
            });
        } else {
            auto eight = [&](auto qTag) __attribute__((always_inline)) { // columns 8 (q + h) .. + 7 of the block
                const ks_f32x4 x = summed(qTag), y = summed(std::integral_constant<int, decltype(qTag)::value + 1>());
                uint32_t x0 = Bf16Pair(x[0], x[1]), x1 = Bf16Pair(x[2], x[3]), y0 = Bf16Pair(y[0], y[1]), y1 = Bf16Pair(y[2], y[3]);
                SwapHalves(x0, y0);
                SwapHalves(x1, y1);
                return Words4{x0, x1, y0, y1};
            };
            if constexpr (kKept % 4 == 0) {
                StaticFor<0, kKept / 4>([&](auto tag) __attribute__((always_inline)) {
                    constexpr int q = g * kKept + 4 * decltype(tag)::value, idx = q / 4;
                    Words4 x = eight(std::integral_constant<int, q>()), y = eight(std::integral_constant<int, q + 2>());
#pragma unroll
                    for (int i = 0; i < 4; ++i) {
                        uint32_t xi = x[i], yi = y[i];
                        SwapRows(xi, yi);
                        x[i] = xi;
                        y[i] = yi;
                    }
                    const int row = rowLane + 32 * (idx / NB) + (int)(lane % 16), col = colLane + 32 * (idx % NB) + 16 * (int)(lane / 16 % 2) + 8 * (int)h;
                    if (col < n) {
                        if (row < m)
                            StoreEight(out + (int64_t)row * n + col, x, col + 4 < n, through);
                        if (row + 16 < m)
                            StoreEight(out + (int64_t)(row + 16) * n + col, y, col + 4 < n, through);
                    }
                });
            } else {
                static_assert(kKept == 2, "whole blocks, or half of the only one");
                constexpr int q = g * kKept;
                const Words4 x = eight(std::integral_constant<int, q>());
                const int row = rowLane + (int)r32, col = colLane + 8 * (q + (int)h);
                if (row < m && col < n)
                    StoreEight(out + (int64_t)row * n + col, x, col + 4 < n, 0);
            }
        }
    });
}

} // namespace
PTO_DEVICE_CODE_END

namespace {
template <int FMT_A, int FMT_B, typename OutT, int BM, int BN, int S, int MIN_WAVES>
int launch_gemm_mxks(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k)
{
    if (m <= 0 || n <= 0 || k <= 0 || n % 4 || k % 512) // (512 k: 16 scale bytes of a row, an even number of steps)
        return PTO_ERR_UNSUPPORTED;
    constexpr int lds = MxKsLdsBytes<BM, BN, S>();
    static_assert(lds <= 160 * 1024, "stages fit the LDS");
    auto kernel = GemmMxKs<FMT_A, FMT_B, OutT, BM, BN, S, MIN_WAVES, 4>;
    static const int attr = lds <= 64 * 1024 ? PTO_OK : pto_amd::allow_lds(kernel, lds);
    if (attr != PTO_OK)
        return attr;
    const long long tiles = (long long)((m + BM - 1) / BM) * ((n + BN - 1) / BN);
    if (tiles > 0x7fffffffll)
        return PTO_ERR_UNSUPPORTED;
    kernel<<<dim3((unsigned)tiles), dim3(64 * MxKsWaves(BM, BN)), lds, st>>>(reinterpret_cast<OutT *>(c), a, b, sa, sb, m, n, (uint32_t)(FMT_A == 4 ? k / 2 : k),
                                                          (uint32_t)(k / 32), pto_amd::store_through(c, sizeof(OutT) * (uint64_t)n, sizeof(OutT) * (uint64_t)m * n));
    return pto_amd::check_launch();
}
} // namespace
