// MXFP8 GEMM tile of 256 x BN (BN = 96, 128 .. 256 in steps of 32) on four wavefronts: the four-wave fp16 kernel of gemm_kernels_w4.hpp with
// 8-bit operands.  A K-step is the same 128 bytes per operand row (128 k instead of 64), so copies, LDS images and fragment
// reads are byte for byte those of the fp16 kernel; what differs:
//   * one v_mfma_scale_f32_16x16x128_f8f6f4 (8 passes) per 16 x 16 block and step instead of two v_mfma_f32_16x16x32_f16
//     (4 passes each).  Its operand registers hold, for lane group g = lane / 16, bytes 16 g .. + 15 of the row's first 64
//     k and bytes 64 + 16 g .. + 15 of its second 64 k: exactly the two reads of the fp16 kernel;
//   * the block scales (one e8m0 byte per row and 32 k = per lane and MFMA exactly one byte).  The MFMAs of four steps
//     (512 k = 16 scale bytes of a row) take theirs from one register per block row / column: byte j = the scale of the
//     lane's k block g in step j (op_sel selects j).  These registers are made for 16 steps (64 scale bytes of a row) at
//     once: lane group g loads bytes 16 g .. + 15 of the 64 straight from memory (one instruction and one cache line per
//     row for 16 steps), transposes its 4 x 4 bytes (register u = byte u of each k-block quadruple: what lane group u
//     needs) and the four lane groups exchange register u of group g with register g of group u (two
//     v_permlane32_swap, two v_permlane16_swap).  One block row / column per step: load at the start of the step,
//     permutes and swaps behind its barrier, into the set of the next 16 steps;
//   * four B stages (96 + 64 KiB = the whole LDS at BN = 192), which makes the step's second barrier unnecessary: a
//     stage is overwritten two steps after its last read, with the barrier of the step in between.
// Steps come in groups of four (B stage, A slot and scale byte repeat): k % 512 == 0.
// BN = 224 and 256: up to all 256 accumulation registers, a seventh fewer copies and a sixteenth fewer fragment reads per MFMA at 256 than at 192.  Three B stages fit, so a step has a
// second barrier again, ahead of its first copy of B, and as three stages and eight (sixteen) steps of a scale period do not go together, they take
// turns at run time.  Two sets of scale registers do not fit: rows are loaded over their own first three quarters when the last one has been moved
// aside, and spread in place.  What the time goes into (2040 x 8100 x 8192 fp4 on 256 x 128 tiles, 72.8 us; one part taken out): copies 8.8, reads of B 5.3 and of
// A 3.0, scales 3.9; with none of them 53.3, the MFMAs at the clock they hold.  With 256 x 256 tiles 66.0; fp8 121 -> 104.  The widths between are for products whose rounds they fill:
// 1000 x 6144 x 4096 fp8 on 256 x 96 tiles 27.6 -> 25.7 us, fp4 19.0 -> 17.4.
// MXFP4 (format 4, two e2m1 per byte): a K-step of 128 bytes is 256 k = two MFMAs (4 passes each, 16-byte operands: lane group
// g holds bytes 16 g .. + 15 of the MFMA's 64) and eight scale blocks per row, so a scale register lasts two steps (the MFMA of
// step j % 2 and half kk selects byte 2 (j % 2) + kk), the 64 scale bytes of a row eight steps, and two block rows / columns
// are loaded per step: k % 1024 == 0.
#pragma once
#include "gemm_kernels_w4.hpp"

PTO_DEVICE_CODE_BEGIN
namespace {

// acc block BLK += first x second (both 16 rows x 128 k bytes) with their scales, scale byte SEL of either register
template <int BLK, int SEL, int FMT_FIRST, int FMT_SECOND>
PTO_DEV void MxW4Mfma(i32x8 first, i32x8 second, uint32_t scaleFirst, uint32_t scaleSecond)
{
#define X(b, r0, r1, r2, r3)                                                                                                          \
    if constexpr (BLK == b)                                                                                                           \
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 a[" #r0 ":" #r3 "], %0, %1, a[" #r0 ":" #r3 "], %2, %3 op_sel:[%4,%4,0] "       \
                     "op_sel_hi:[%5,%5,0] cbsz:%6 blgp:%7" ::"v"(first),                                                              \
                     "v"(second), "v"(scaleFirst), "v"(scaleSecond), "n"(SEL & 1), "n"(SEL >> 1), "n"(FMT_FIRST), "n"(FMT_SECOND)    \
                     : "a" #r0, "a" #r1, "a" #r2, "a" #r3);
    PTO_W4_ACC_BLOCKS(X)
#undef X
}

// the same with 4-bit operands: 16 rows x 128 k = 64 bytes per row, 16 per lane
template <int BLK, int SEL>
PTO_DEV void MxW4MfmaFp4(u32x4 first, u32x4 second, uint32_t scaleFirst, uint32_t scaleSecond)
{
#define X(b, r0, r1, r2, r3)                                                                                                          \
    if constexpr (BLK == b)                                                                                                           \
        asm volatile("v_mfma_scale_f32_16x16x128_f8f6f4 a[" #r0 ":" #r3 "], %0, %1, a[" #r0 ":" #r3 "], %2, %3 op_sel:[%4,%4,0] "       \
                     "op_sel_hi:[%5,%5,0] cbsz:4 blgp:4" ::"v"(first),                                                                \
                     "v"(second), "v"(scaleFirst), "v"(scaleSecond), "n"(SEL & 1), "n"(SEL >> 1)                                      \
                     : "a" #r0, "a" #r1, "a" #r2, "a" #r3);
    PTO_W4_ACC_BLOCKS(X)
#undef X
}

// 16 bytes per lane from memory as assembly (counted by the kernel's own waits); use the result only behind such a wait
PTO_DEV u32x4 MxW4Load16(const char *base, uint32_t voff)
{
    u32x4 r;
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(r) : "v"(voff), "s"(base) : "memory");
    return r;
}

// (the compiler does not see that the load above is still on its way: a value is used only behind one of these)
PTO_DEV void MxW4Pin(u32x4 &x) { asm volatile("" : "+v"(x)); }
PTO_DEV void MxW4WaitLoads(u32x4 &x) { asm volatile("s_waitcnt vmcnt(0)" : "+v"(x)::"memory"); }

// w = the 16 scale bytes that this lane's group g loaded (bytes 16 g .. + 15 of the 64 of its row) -> out[u] = bytes g, 4 + g,
// 8 + g, 12 + g of the 16 bytes that group u loaded: the scales of the lane's k block in the four MFMA rounds of quarter u
// In four parts, each a few instructions between two MFMAs; w is worked on in place and holds out[0 .. 3] after part 3.
template <int PART>
PTO_DEV void MxW4ScaleSpreadPart(u32x4 &w)
{
    if constexpr (PART == 0) { // bytes transposed within the lane: register u = byte u of w[0], w[1], w[2], w[3], in two rounds
        const uint32_t t0 = __builtin_amdgcn_perm(w[1], w[0], 0x05010400u), t1 = __builtin_amdgcn_perm(w[1], w[0], 0x07030602u);
        const uint32_t t2 = __builtin_amdgcn_perm(w[3], w[2], 0x05010400u), t3 = __builtin_amdgcn_perm(w[3], w[2], 0x07030602u);
        w = u32x4{t0, t1, t2, t3};
    } else if constexpr (PART == 1) {
        const uint32_t p0 = __builtin_amdgcn_perm(w[2], w[0], 0x05040100u), p1 = __builtin_amdgcn_perm(w[2], w[0], 0x07060302u);
        const uint32_t p2 = __builtin_amdgcn_perm(w[3], w[1], 0x05040100u), p3 = __builtin_amdgcn_perm(w[3], w[1], 0x07060302u);
        w = u32x4{p0, p1, p2, p3};
    } else if constexpr (PART == 2) { // registers transposed against lane groups: (register u of group g) <-> (register g of group u)
        const auto a = __builtin_amdgcn_permlane32_swap(w[0], w[2], false, false), b = __builtin_amdgcn_permlane32_swap(w[1], w[3], false, false);
        w = u32x4{a[0], b[0], a[1], b[1]};
    } else {
        const auto c = __builtin_amdgcn_permlane16_swap(w[0], w[1], false, false), d = __builtin_amdgcn_permlane16_swap(w[2], w[3], false, false);
        w = u32x4{c[0], c[1], d[0], d[1]};
    }
}

PTO_DEV void MxW4ScaleSpread(u32x4 w, uint32_t (&out)[4])
{
    MxW4ScaleSpreadPart<0>(w);
    MxW4ScaleSpreadPart<1>(w);
    MxW4ScaleSpreadPart<2>(w);
    MxW4ScaleSpreadPart<3>(w);
    out[0] = w[0];
    out[1] = w[1];
    out[2] = w[2];
    out[3] = w[3];
}

// Issue slots of a K-step: slot = 4 nb + mb (nb: 16-column block, outer; mb: 16-row block of the wave's 64 rows).
template <int NNB, int NCOPY>
struct MxW4Sched {
    static constexpr int kPD = 2, kSlots = 4 * NNB, kBarrier = 4 * (NNB - kPD) - 1;
    // the eight A reads of the next step
    static constexpr int aReadSlot(int q) { return NNB >= 10 ? 4 * (q + 1) + 3 : 4 * (q / 2 + 1) + 2 + q % 2; }
    static constexpr int copySlot(int j) { return 2 + j * (kSlots - 6) / NCOPY; }
    static constexpr int aReadAt(int idx)
    {
        for (int q = 0; q < 8; ++q)
            if (aReadSlot(q) == idx)
                return q;
        return -1;
    }
    static constexpr int copyAt(int idx)
    {
        for (int j = 0; j < NCOPY; ++j)
            if (copySlot(j) == idx)
                return j;
        return -1;
    }
    static constexpr int aReadsIn(int lo, int hi) // A reads at slots in [lo, hi]
    {
        int n = 0;
        for (int q = 0; q < 8; ++q)
            if (aReadSlot(q) >= lo && aReadSlot(q) <= hi)
                ++n;
        return n;
    }
    static constexpr int copiesBefore(int idx) // copies of this step issued at slots < idx
    {
        int n = 0;
        for (int j = 0; j < NCOPY; ++j)
            if (copySlot(j) < idx)
                ++n;
        return n;
    }
    static constexpr bool distinct()
    {
        for (int q = 1; q < 8; ++q)
            if (aReadSlot(q) <= aReadSlot(q - 1))
                return false;
        for (int j = 1; j < NCOPY; ++j)
            if (copySlot(j) <= copySlot(j - 1)) // the LDS address of copy j is set one slot before it, behind a copy there
                return false;
        return true;
    }
    // (A is read ahead of the block column behind which the next step waits for nothing older)
    static_assert(aReadSlot(7) < 4 * (NNB - 1) && copySlot(NCOPY - 1) < kSlots && copySlot(0) >= 2 && distinct(), "order of the step");
    static_assert(kBarrier + 8 < kSlots, "two scale rows are spread in the slots behind the barrier");
};

// accumulators = (A .* scales)[row0 .. + 256, :] x (B .* scales)[col0 .. + BN, :]^T over the whole K extent (k elements, four
// K-steps of 128 bytes per row at a time); block (mb, nb) of this wave's 64 rows in accumulator block (BN / 16) mb + nb.
// FMT: 0 = e4m3, 1 = e5m2, 4 = e2m1 (both operands then).
template <int FMT_A, int FMT_B, int BN>
AICORE inline __attribute__((always_inline)) void MxW4TileCompute(__gm__ const uint8_t *src0, __gm__ const uint8_t *src1,
                                                                  __gm__ const uint8_t *scale0, __gm__ const uint8_t *scale1, int k,
                                                                  int row0, int col0)
{
    constexpr bool WIDE = BN > 192;
    constexpr int NMB = 4, NNB = BN / 16, NBUF = 4, BSTAGES = WIDE ? 3 : 4, NA = 8, NCB = BN / 32, NCOPY = NA + NCB;
    using S = MxW4Sched<NNB, NCOPY>;
    constexpr bool FP4 = FMT_A == 4;
    static_assert((FMT_A == 4) == (FMT_B == 4), "fp4 with fp4");
    // steps that a scale register (16 scale bytes of a row) lasts, steps that the 64 bytes loaded at once last, and block rows /
    // columns loaded in each of these
    constexpr int PD = S::kPD, kScales = NMB + NNB, kGroupSteps = FP4 ? 2 : 4, kSuperSteps = 4 * kGroupSteps;
    constexpr int kScaleLoads = (kScales + kSuperSteps - 1) / kSuperSteps;
    constexpr uint32_t kStepBytes = 128, kBBytes = kStepBytes * BN, kASlot = 64 * kStepBytes, kABase = BSTAGES * kBBytes;
    static_assert(BN % 32 == 0 && kABase + 8 * kASlot <= 160 * 1024, "tile width");
    using std::integral_constant;

    const int wave = hw::wave();
    const uint32_t lane = (uint32_t)hw::lane();
    const uint32_t ldsBase = (uint32_t)(uintptr_t)hw::lds_base();
    const int64_t ld = FP4 ? k / 2 : k; // bytes between rows of A and between columns of B
    const int kLoop = (int)(ld / 128), supers = (kLoop + kSuperSteps - 1) / kSuperSteps;
    const char *aWave = reinterpret_cast<const char *>(src0) + ((int64_t)row0 + 64 * wave) * ld;
    const char *bPanel = reinterpret_cast<const char *>(src1) + (int64_t)col0 * ld;
    auto chunkOf = [](uint32_t q) { return q; };
    const uint32_t posEven = (lane % 8) ^ (lane / 16);
    const uint32_t aCopyOff[2] = {(lane / 8) * (uint32_t)ld + chunkOf(posEven) * 16u, (lane / 8) * (uint32_t)ld + chunkOf(posEven ^ 4u) * 16u};
    const uint32_t bCopyOff = (uint32_t)(8 * wave + lane / 8) * (uint32_t)ld + chunkOf((lane % 8) ^ ((4 * wave + lane / 16) % 8)) * 16u;
    const uint32_t aLdsWave = ldsBase + kABase + (uint32_t)wave * (2 * kASlot), bLdsWave = ldsBase + (uint32_t)wave * 1024u;
    uint32_t aAddr[2][2], bAddr[2][BSTAGES];
    {
        const uint32_t r = lane % 16, pos = (lane / 16) ^ detail::mat_swz<128>(r);
        const uint32_t off = r * 128u + pos * 16u;
#pragma unroll
        for (int s = 0; s < 2; ++s) {
            aAddr[0][s] = aLdsWave + s * kASlot + off;
            aAddr[1][s] = aAddr[0][s] ^ 64u;
        }
#pragma unroll
        for (int s = 0; s < BSTAGES; ++s) {
            bAddr[0][s] = ldsBase + s * kBBytes + off;
            bAddr[1][s] = bAddr[0][s] ^ 64u;
        }
    }
    const char *aBase[NA], *bBase[NCB];
#pragma unroll
    for (int t = 0; t < NA; ++t)
        aBase[t] = detail::uniform_ptr(aWave + (int64_t)(8 * t) * ld);
#pragma unroll
    for (int t = 0; t < NCB; ++t)
        bBase[t] = detail::uniform_ptr(bPanel + (int64_t)(32 * t) * ld);
    // scales: scale row i < NMB is block row i of this wave (row 16 i + lane % 16), i >= NMB block column i - NMB of the tile;
    // k / 32 bytes between rows, 64 bytes per kSuperSteps steps of which lane group g loads bytes 16 g .. + 15 (the last 16 of
    // the row where that is past its end: scales of steps beyond K)
    const uint32_t ldScale = (uint32_t)(k / 32);
    const char *saWave = detail::uniform_ptr(reinterpret_cast<const char *>(scale0) + ((int64_t)row0 + 64 * wave) * ldScale);
    const char *sbPanel = detail::uniform_ptr(reinterpret_cast<const char *>(scale1) + (int64_t)col0 * ldScale);
    const uint32_t scaleRowOff = (lane % 16) * ldScale;
    auto scaleLoad = [&](auto iTag, int super) __attribute__((always_inline)) {
        constexpr int i = decltype(iTag)::value;
        const uint32_t chunk = (uint32_t)super * 64u + (lane / 16) * 16u;
        const uint32_t voff = scaleRowOff + (uint32_t)((i < NMB ? i : i - NMB) * 16) * ldScale + (chunk < ldScale - 16u ? chunk : ldScale - 16u);
        return MxW4Load16(i < NMB ? saWave : sbPanel, voff);
    };

    // WIDE: three B stages take turns at run time: of step it, of it + 1 and of the copies for it + 2
    uint32_t bNow[2] = {bAddr[0][0], bAddr[1][0]}, bThen[2] = {bAddr[0][1], bAddr[1][1]};
    uint32_t stageNow = 0, stageThen = kBBytes, stageCopy = 2 * kBBytes;
    uint32_t voffA[2], voffB;
    auto setLds = [&](uint32_t waveBase, auto immTag) __attribute__((always_inline)) {
        asm volatile("s_add_u32 m0, %0, %1" ::"s"(waveBase), "n"(decltype(immTag)::value) : "memory", "scc");
    };
    auto copyAsm = [&](uint32_t voff, const char *base) __attribute__((always_inline)) {
        asm volatile("global_load_lds_dwordx4 %0, %1" ::"v"(voff), "s"(base) : "memory");
    };
    struct Pair { // the two 16-byte halves of a 32-byte operand
        f16x8 h[2];
    };
    Pair aF[2][NMB], bF[NBUF];
    // scales of the current kSuperSteps steps and of the next, a register per quarter.  WIDE: one set.  In the last quarter, which then stands apart
    // (scLast), the rows' new ones are loaded over the others
    uint32_t sc[kScales][4], scNext[WIDE ? 1 : kScales][4] = {};
    u32x4 raw[kScaleLoads], rows[WIDE ? kScales : 1];
    uint32_t scLast[WIDE ? kScales : 1];
    constexpr int kLastQuarter = 3 * kGroupSteps;
    auto readA = [&](auto setTag, auto qTag) __attribute__((always_inline)) {
        constexpr int set = decltype(setTag)::value, q = decltype(qTag)::value, mb = q / 2, kk = q % 2;
        aF[set][mb].h[kk] = W4LdsRead16<mb * 2048>(aAddr[kk][set]);
    };
    // (bufTag: the block column counted on through the steps, so that the buffers take turns whatever their number in a step)
    auto readB = [&](auto stageTag, auto nbTag, auto kkTag, auto bufTag) __attribute__((always_inline)) {
        constexpr int stage = decltype(stageTag)::value, nb = decltype(nbTag)::value, kk = decltype(kkTag)::value, buf = decltype(bufTag)::value % NBUF;
        if constexpr (WIDE)
            bF[buf].h[kk] = W4LdsRead16<nb * 2048>(stage == 0 ? bNow[kk] : bThen[kk]);
        else
            bF[buf].h[kk] = W4LdsRead16<nb * 2048>(bAddr[kk][stage]);
    };
    static_assert(2 * NNB % NBUF == 0, "the same turn every second step");
    auto operand = [](const Pair &p) {
        const u32x4 lo = __builtin_bit_cast(u32x4, p.h[0]), hi = __builtin_bit_cast(u32x4, p.h[1]);
        return i32x8{(int)lo[0], (int)lo[1], (int)lo[2], (int)lo[3], (int)hi[0], (int)hi[1], (int)hi[2], (int)hi[3]};
    };
    auto clampStep = [&](int s) { return s < kLoop ? s : kLoop - 1; };

    // ---- prologue: the scales of the first four steps, A and B of steps 0 and 1 ----
    __builtin_amdgcn_s_barrier(); // every wave is done with the LDS of the tile before
    u32x4 first[kScales]; // all in flight at once, picked apart behind the wait for step 0 below
    W4For<0, kScales>([&](auto iTag) __attribute__((always_inline)) { first[decltype(iTag)::value] = scaleLoad(iTag, 0); });
    W4For<0, 2>([&](auto sTag) __attribute__((always_inline)) {
        constexpr int s = decltype(sTag)::value;
        const uint32_t kOff = (uint32_t)clampStep(s) * kStepBytes;
        W4For<0, NCOPY>([&](auto jTag) __attribute__((always_inline)) {
            constexpr int j = decltype(jTag)::value;
            if constexpr (j < NA)
                setLds(aLdsWave, integral_constant<int, s * kASlot + j * 1024>());
            else
                setLds(bLdsWave, integral_constant<int, s * kBBytes + (j - NA) * 4096>());
            asm volatile("s_nop 0" ::: "memory");
            if constexpr (j < NA)
                copyAsm(aCopyOff[j % 2] + kOff, aBase[j]);
            else
                copyAsm(bCopyOff + kOff, bBase[j - NA]);
        });
    });
    hw::wait_vm<NCOPY>();
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
    W4For<0, kScales>([&](auto iTag) __attribute__((always_inline)) {
        constexpr int i = decltype(iTag)::value;
        MxW4Pin(first[i]); // (older than the copies waited for above)
        if constexpr (WIDE) {
            rows[i] = first[i];
            W4For<0, 4>([&](auto partTag) __attribute__((always_inline)) { MxW4ScaleSpreadPart<decltype(partTag)::value>(rows[i]); });
        } else {
            MxW4ScaleSpread(first[i], sc[i]);
        }
    });
    __builtin_amdgcn_sched_barrier(0);
    W4For<0, NA>([&](auto qTag) __attribute__((always_inline)) { readA(integral_constant<int, 0>(), qTag); });
    W4For<0, 2 * PD>([&](auto fTag) __attribute__((always_inline)) {
        constexpr int f = decltype(fTag)::value;
        readB(integral_constant<int, 0>(), integral_constant<int, f / 2>(), integral_constant<int, f % 2>(), integral_constant<int, f / 2>());
    });

    // ---- K-step `it`, number t = it % kSuperSteps of its scale period: B stage t % 4, A register set and LDS slot t % 2, scale
    // register t / kGroupSteps, byte t % kGroupSteps (fp4: two bytes).  The copies of A of step it + 2 go to this step's A slot,
    // those of B to the stage of step it - 2; scale rows kScaleLoads t .. of the next period are loaded at the start of the step
    // and spread over the lane groups behind its barrier.
    // WIDE: three B stages in turn (stageNow, stageThen, stageCopy), the copies of B of step it + 2 to the stage of step it - 1, behind a barrier of their
    // own; all scale rows of the next period are loaded and spread in the last quarter of a period, over the three quarters that are used up.
    auto step = [&](auto tTag, int it, int super) __attribute__((always_inline)) {
        constexpr int t = decltype(tTag)::value, j = t % 4, par = j % 2;
        constexpr int s = WIDE ? 0 : j, sNext = WIDE ? 1 : (j + 1) % BSTAGES, sCopy = (j + 2) % BSTAGES;
        constexpr int quarter = t / kGroupSteps, jj = t % kGroupSteps, left = kScales - kScaleLoads * t;
        constexpr int nLoads = WIDE ? 0 : left < 0 ? 0 : (left < kScaleLoads ? left : kScaleLoads);
        const uint32_t kOff = (uint32_t)clampStep(it + 2) * kStepBytes;
        const int nextSuper = super + 1 < supers ? super + 1 : supers - 1;
        W4For<0, S::kSlots>([&](auto idxTag) __attribute__((always_inline)) {
            constexpr int idx = decltype(idxTag)::value, nb = idx / NMB, mb = idx % NMB;
            if constexpr (idx == 0) { // (older than every copy of this step)
                W4For<0, nLoads>([&](auto uTag) __attribute__((always_inline)) {
                    constexpr int u = decltype(uTag)::value;
                    raw[u] = scaleLoad(integral_constant<int, kScaleLoads * t + u>(), nextSuper);
                });
            }
            if constexpr (idx == 1) {
                voffA[0] = aCopyOff[0] + kOff;
                voffA[1] = aCopyOff[1] + kOff;
                voffB = bCopyOff + kOff;
            }
            if constexpr (WIDE) {
                // the last quarter's scales out of the way; the next rows loaded, a slot each; their parts from kSpread slots on, a slot each
                constexpr int since = (t - kLastQuarter) * S::kSlots + idx;
                if constexpr (t == kLastQuarter - 1 && idx < kScales)
                    asm volatile("v_mov_b32 %0, %1" : "=v"(scLast[idx]) : "v"(rows[idx][3]));
                if constexpr (since >= 0 && since < kScales)
                    rows[since] = scaleLoad(integral_constant<int, since>(), nextSuper);
                constexpr int kSpread = 2 * S::kSlots - 4 * kScales;
                static_assert(kSpread >= kScales, "all loaded before the first is spread");
                if constexpr (since == kSpread) // (the copies issued since the last of the loads may be under way)
                    hw::wait_vm<S::copiesBefore(kSpread) - S::copiesBefore(kScales)>();
                if constexpr (since >= kSpread && since < kSpread + 4 * kScales) {
                    constexpr int row = (since - kSpread) / 4, part = (since - kSpread) % 4;
                    if constexpr (part == 0)
                        MxW4Pin(rows[row]);
                    MxW4ScaleSpreadPart<part>(rows[row]);
                }
                if constexpr (idx == S::copySlot(NA) - 2) { // every wave has read all of the step before, whose B stage the copies go to
                    __builtin_amdgcn_s_barrier();
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if constexpr (idx == S::kBarrier) {
                // this wave's copies of the step before have landed (and this step's scale rows, which are older than its copies)
                // (WIDE: the scale rows of a step, some of them behind its first copies, are older than its last ones as well)
                hw::wait_vm<S::copiesBefore(S::kBarrier)>();
                __builtin_amdgcn_s_barrier();
                __builtin_amdgcn_sched_barrier(0);
            }
            if constexpr (idx > S::kBarrier && idx <= S::kBarrier + 4 * nLoads) { // a part of the spreading of a loaded scale row
                constexpr int u = (idx - S::kBarrier - 1) / 4, part = (idx - S::kBarrier - 1) % 4;
                if constexpr (part == 0)
                    MxW4Pin(raw[u]); // (not before the wait above)
                MxW4ScaleSpreadPart<part>(raw[u]);
                if constexpr (part == 3) {
                    scNext[kScaleLoads * t + u][0] = raw[u][0];
                    scNext[kScaleLoads * t + u][1] = raw[u][1];
                    scNext[kScaleLoads * t + u][2] = raw[u][2];
                    scNext[kScaleLoads * t + u][3] = raw[u][3];
                }
            }
            if constexpr (mb < 2) { // half mb of the B operand of block column nb + PD
                constexpr int g = nb + PD;
                if constexpr (g < NNB)
                    readB(integral_constant<int, s>(), integral_constant<int, g>(), integral_constant<int, mb>(), integral_constant<int, g + NNB * par>());
                else
                    readB(integral_constant<int, sNext>(), integral_constant<int, g - NNB>(), integral_constant<int, mb>(), integral_constant<int, g + NNB * par>());
            }
            if constexpr (S::aReadAt(idx) >= 0) {
                if constexpr (S::aReadAt(idx) == 0) // this wave's A copies of the step before have landed
                    hw::wait_vm<NCB + nLoads + S::copiesBefore(idx) + (WIDE && t == kLastQuarter ? idx + 1 : 0)>();
                readA(integral_constant<int, par ^ 1>(), integral_constant<int, S::aReadAt(idx)>());
            }
            if constexpr (S::copyAt(idx) >= 0) {
                constexpr int c = S::copyAt(idx);
                if constexpr (c < NA)
                    copyAsm(voffA[c % 2], aBase[c]);
                else
                    copyAsm(voffB, bBase[c - NA]);
            }
            if constexpr (S::copyAt(idx + 1) >= 0) {
                constexpr int c = S::copyAt(idx + 1);
                if constexpr (c < NA)
                    setLds(aLdsWave, integral_constant<int, par * kASlot + c * 1024>());
                else if constexpr (WIDE)
                    setLds(bLdsWave + stageCopy, integral_constant<int, (c - NA) * 4096>());
                else
                    setLds(bLdsWave, integral_constant<int, sCopy * kBBytes + (c - NA) * 4096>());
            }
            if constexpr (mb == 0) { // both halves of block column nb have arrived; what was read after them may be under way
                constexpr int lo = 4 * (nb - PD) + 1;
                asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(2 * (PD - 1) + 1 + (lo > 0 ? S::aReadsIn(lo, idx) : 0)) : "memory");
            }
            auto scaleOf = [&](auto rowTag) __attribute__((always_inline)) {
                constexpr int row = decltype(rowTag)::value;
                if constexpr (!WIDE)
                    return sc[row][quarter];
                else if constexpr (quarter == 3)
                    return scLast[row];
                else
                    return (uint32_t)rows[row][quarter];
            };
            if constexpr (FP4) {
                // (the second half right behind the first: with the halves of two blocks in turn 2 % slower)
                MxW4MfmaFp4<mb * NNB + nb, 2 * jj>(__builtin_bit_cast(u32x4, bF[(nb + NNB * par) % NBUF].h[0]), __builtin_bit_cast(u32x4, aF[par][mb].h[0]),
                                                   scaleOf(integral_constant<int, NMB + nb>()), scaleOf(integral_constant<int, mb>()));
                MxW4MfmaFp4<mb * NNB + nb, 2 * jj + 1>(__builtin_bit_cast(u32x4, bF[(nb + NNB * par) % NBUF].h[1]), __builtin_bit_cast(u32x4, aF[par][mb].h[1]),
                                                       scaleOf(integral_constant<int, NMB + nb>()), scaleOf(integral_constant<int, mb>()));
            } else {
                MxW4Mfma<mb * NNB + nb, jj, FMT_B, FMT_A>(operand(bF[(nb + NNB * par) % NBUF]), operand(aF[par][mb]), scaleOf(integral_constant<int, NMB + nb>()),
                                                          scaleOf(integral_constant<int, mb>()));
            }
            __builtin_amdgcn_sched_barrier(0);
        });
        if constexpr (WIDE) {
            const uint32_t done = stageNow;
            stageNow = stageThen;
            stageThen = stageCopy;
            stageCopy = done;
#pragma unroll
            for (int kk = 0; kk < 2; ++kk) {
                bNow[kk] = bThen[kk];
                bThen[kk] = bAddr[kk][0] + stageThen;
            }
        }
    };
    for (int super = 0; super < supers; ++super) {
        const int it0 = super * kSuperSteps;
        W4For<0, kSuperSteps / 4>([&](auto qTag) __attribute__((always_inline)) {
            constexpr int q = decltype(qTag)::value;
            if (it0 + 4 * q < kLoop) { // (K is whole groups of four steps, not whole scale periods)
                step(integral_constant<int, 4 * q>(), it0 + 4 * q, super);
                step(integral_constant<int, 4 * q + 1>(), it0 + 4 * q + 1, super);
                step(integral_constant<int, 4 * q + 2>(), it0 + 4 * q + 2, super);
                step(integral_constant<int, 4 * q + 3>(), it0 + 4 * q + 3, super);
            }
        });
        if constexpr (!WIDE) {
#pragma unroll
            for (int i = 0; i < kScales; ++i)
#pragma unroll
                for (int u = 0; u < 4; ++u)
                    sc[i][u] = scNext[i][u];
        }
    }
    hw::wait_vm0(); // the copies issued past the end of K
    // the last MFMAs have written their accumulators
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_nop 15\n\ts_nop 15" ::: "memory");
}

// This wave's accumulator blocks to C (row-major, n elements between rows; fp32, or bf16 rounded to nearest even).  bf16: a lane has
// four columns of a row, 8 bytes; two blocks side by side change lanes so that it has eight of one of them, and a store
// instruction writes 64 bytes of each of its sixteen rows, as with fp32 (and the hardware conversion: 6144^3 182 -> 175 us in fp8, 121 -> 112
// in fp4, 1000 x 6144 x 4096 in fp8 31.5 -> 28.3, of which 1.3 by storing past the L2).
template <typename OutT, int BN>
AICORE inline __attribute__((always_inline)) void MxW4StoreTile(OutT *out, int64_t n, int row0, int col0, int through)
{
    constexpr int NNB = BN / 16;
    static_assert(NNB % 2 == 0, "blocks in pairs");
    const uint32_t lane = (uint32_t)hw::lane();
    if constexpr (std::is_same_v<OutT, float>) {
        OutT *cWave = out + ((int64_t)row0 + 64 * hw::wave() + lane % 16) * n + col0 + 4 * (lane / 16);
        W4For<0, 4 * NNB>([&](auto idxTag) __attribute__((always_inline)) {
            constexpr int idx = decltype(idxTag)::value, mb = idx / NNB, nb = idx % NNB;
            StoreFour(cWave + (int64_t)(16 * mb) * n + 16 * nb, W4ReadAcc<idx>(), through);
        });
    } else {
        // (lane groups 0 .. 3 of a pair: columns 0, 16, 8, 24 onwards)
        OutT *cWave = out + ((int64_t)row0 + 64 * hw::wave() + lane % 16) * n + col0 + 16 * (lane / 16 % 2) + 8 * (lane / 32);
        W4For<0, 2 * NNB>([&](auto idxTag) __attribute__((always_inline)) {
            constexpr int idx = 2 * decltype(idxTag)::value, mb = idx / NNB, nb = idx % NNB;
            const detail::AccFrag x = W4ReadAcc<idx>(), y = W4ReadAcc<idx + 1>();
            uint32_t x0 = Bf16Pair(x.x, x.y), x1 = Bf16Pair(x.z, x.w), y0 = Bf16Pair(y.x, y.y), y1 = Bf16Pair(y.z, y.w);
            SwapRows(x0, y0);
            SwapRows(x1, y1);
            StoreEight(cWave + (int64_t)(16 * mb) * n + 16 * nb, Words4{x0, x1, y0, y1}, true, through);
        });
    }
}

// One 256 x BN tile of C per workgroup; the last tile row / column is moved back to end with the matrix.
template <int FMT_A, int FMT_B, typename OutT, int BN, int GROUP_M>
__global__ __launch_bounds__(kBlockThreads, 1) AICORE
    void GemmMxW4(__gm__ OutT *out, __gm__ const uint8_t *src0, __gm__ const uint8_t *src1, __gm__ const uint8_t *scale0,
                  __gm__ const uint8_t *scale1, int m, int n, int k, int through)
{
    constexpr int TM = 256;
    const int tilesM = (m + TM - 1) / TM, tilesN = (n + BN - 1) / BN;
    int tm, tn;
    TileOfId<GROUP_M>(RegroupXcd((int)get_block_idx(), tilesM * tilesN), tilesM, tilesN, tm, tn);
    const int r = tm * TM, c = tn * BN;
    const int row0 = __builtin_amdgcn_readfirstlane(r + TM <= m ? r : m - TM);
    const int col0 = __builtin_amdgcn_readfirstlane(c + BN <= n ? c : n - BN);
    W4ZeroAcc<4 * BN / 16>();
    MxW4TileCompute<FMT_A, FMT_B, BN>(src0, src1, scale0, scale1, k, row0, col0);
    MxW4StoreTile<OutT, BN>(out, n, row0, col0, through);
}

} // namespace
PTO_DEVICE_CODE_END

namespace {
template <int FMT_A, int FMT_B, typename OutT, int BN>
int launch_gemm_mxw4(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k)
{
    // (n % 4: four consecutive elements of a row are inside or outside together)
    if (m < 256 || n < BN || n % 4 || k % (FMT_A == 4 ? 1024 : 512) || k <= 0)
        return PTO_ERR_UNSUPPORTED;
    constexpr int lds = (BN > 192 ? 3 : 4) * 128 * BN + 4 * 2 * 64 * 128; // four (three) B stages + two A slots per wave
    auto kernel = GemmMxW4<FMT_A, FMT_B, OutT, BN, 4>;
    static const int attr = pto_amd::allow_lds(kernel, lds);
    if (attr != PTO_OK)
        return attr;
    const int tiles = ((m + 255) / 256) * ((n + BN - 1) / BN);
    kernel<<<dim3((unsigned)tiles), dim3(kBlockThreads), lds, st>>>(reinterpret_cast<OutT *>(c), a, b, sa, sb, m, n, k,
                                                               pto_amd::store_through(c, sizeof(OutT) * (uint64_t)n, sizeof(OutT) * (uint64_t)m * n));
    return pto_amd::check_launch();
}
// format: 0 = e4m3 x e4m3, 1 = e5m2 x e5m2, 2 = A e4m3 x B e5m2, 3 = A e5m2 x B e4m3, 4 = e2m1 x e2m1 (k then counts 4-bit
// elements, two per byte)
template <int BN>
int launch_gemm_mxw4_format(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                            int format, int c_fp32)
{
#define PTO_MXW4_CASE(FMT, FA, FB)                                                              \
    if (format == FMT)                                                                         \
        return c_fp32 ? launch_gemm_mxw4<FA, FB, float, BN>(st, c, a, b, sa, sb, m, n, k) :     \
                        launch_gemm_mxw4<FA, FB, bfloat16_t, BN>(st, c, a, b, sa, sb, m, n, k);
    PTO_MXW4_CASE(0, 0, 0)
    PTO_MXW4_CASE(1, 1, 1)
    PTO_MXW4_CASE(2, 0, 1)
    PTO_MXW4_CASE(3, 1, 0)
    PTO_MXW4_CASE(4, 4, 4)
#undef PTO_MXW4_CASE
    return PTO_ERR_UNSUPPORTED;
}
} // namespace
