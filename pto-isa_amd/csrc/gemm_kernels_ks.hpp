// fp16 x fp16 -> fp32 GEMM tiles of 32 .. 256 rows for problems that the 256- and 192-row tiles of gemm_kernels_w4.hpp leave
// most of the chip idle on, and for K extents that are no multiple of 128: BM x BN of C per workgroup of eight wavefronts in
// a 2 x 2 x 2 grid (rows x columns x k).  Both k groups work on the same tile: of a K-step of 64, staged as 128-byte rows,
// group g multiplies k 32 g .. 32 g + 31, so every SIMD has two waves whatever the number of workgroups, at the LDS traffic
// of four waves; the two partial sums meet in the LDS at the end.
//
// A K-step of a wave is (BM + BN) / 32 fragment reads and BM BN / 1024 MFMAs of 16 x 16 x 32.  The fragments of step i + 1
// are read while the MFMAs of step i run (two register sets), the copies of step i + S go to the stage that the barrier of
// step i has freed, S - 1 steps ahead of their first read.
//
// What bounds a step: the copies.  A compute unit takes in 53 bytes per clock of L2-resident lines (measured with all of
// them loading), so the (BM + BN) 128 bytes of a 128 x 128 step are 620 clocks against 512 of its MFMAs; with one part
// taken out a step of 0.46 us (1024 x 3072 x 8192) runs 0.43 without the fragment reads, 0.36 with copies alone and 0.33
// with MFMAs alone.  The place of the copies in the step, raised wave priority and deeper rings changed nothing (1 %; a 32 x 64 step, 12 KiB in
// 0.13 us: rings of 6 to 13 stages 0 to 20 % slower, two steps from one barrier to the next 0 to 10 %).  So where units are idle the tile gets
// smaller: 32 x 32, 0.09 us a step, on twice as many of them (from a graph 512^3 3.76 -> 3.29 us, called one by one 3.87 -> 3.67 or what the host takes; 256 x 256 x 6144 15.8 -> 11.5; four stages 14.8, five 12.0, eight 11.5).
// (1000 x 3000 x 2048 on 128 x 96 tiles runs 0.4 us a step: 28 KiB of copies, from beyond the L2.)
// Small tiles lose there what they win in compute units at work: 512^3 8.96 -> 3.3 us (from a graph), 1000 x 3000 x 2048 21.1 -> 18.0,
// 128 x 4096 x 4096 68 -> 12.  C past the L2 where that pays (store_through): 1000 x 3072 x 2048 18.5 -> 17.0.
//
// Rows past m and columns past n repeat the last one on the way in (their memory may not exist) and are not stored.
#pragma once
#include "gemm_kernels.hpp"

PTO_DEVICE_CODE_BEGIN
namespace {

typedef _Float16 ks_f16x8 __attribute__((ext_vector_type(8)));
typedef float ks_f32x4 __attribute__((ext_vector_type(4)));
typedef float ks_c4 __attribute__((ext_vector_type(4), aligned(4))); // four elements of C, whose rows need no more alignment than these

// 16 bytes per lane from the LDS.  A load that the compiler knows: the registers of one in flight may be spilled or moved, behind
// a wait that it then places (as assembly it stored them with the read still outstanding where a tile had too few registers).
template <int IMM>
PTO_DEV ks_f16x8 KsLdsRead16(uint32_t addr)
{
    const auto *p = (const __attribute__((address_space(3))) char *)(uintptr_t)addr;
    const ks_f16x8 r = *(const __attribute__((address_space(3))) ks_f16x8 *)(p + IMM);
    __builtin_amdgcn_sched_barrier(0); // (in the order written)
    return r;
}

// lgkmcnt(0), the other counters left alone: the builtin, which the compiler counts with (behind one in assembly it would add
// a wait of its own for every fragment)
PTO_DEV void KsWaitLds() { __builtin_amdgcn_s_waitcnt(0xc07f); }

// the reads into a set of fragments are over; keeps them where they were issued, ahead of the MFMAs
template <int MB, int NB>
PTO_DEV void KsArrived(ks_f16x8 (&a)[MB], ks_f16x8 (&b)[NB])
{
    KsWaitLds();
#pragma unroll
    for (int i = 0; i < NB; ++i)
        asm volatile("" : "+v"(b[i]));
#pragma unroll
    for (int i = 0; i < MB; ++i)
        asm volatile("" : "+v"(a[i]));
}

template <int BM, int BN, int S>
constexpr int KsLdsBytes() // S stages of 128-byte rows; the partial sums of half the blocks of either k group afterwards
{
    constexpr int stages = S * (BM + BN) * 128, sums = BM * BN * (int)sizeof(float);
    return stages > sums ? stages : sums;
}

// HALF: k % 64 == 32, the last step is one of 32 (group 1 has no part in it)
template <int BM, int BN, int S, int MIN_WAVES, bool HALF, int GROUP_M>
__global__ __launch_bounds__(512, MIN_WAVES) AICORE void GemmF16F32Ks(float *out, const half *src0, const half *src1, int m, int n, int k, int through)
{
    constexpr int MB = BM / 32, NB = BN / 32;                  // 16 x 16 blocks of a wave
    constexpr int kInst = (BM + BN) / 8, kCopies = (kInst + 7) / 8; // copy instructions of 8 rows a step; per wave
    constexpr uint32_t kStage = (BM + BN) * 128, kRing = S * kStage;
    static_assert(BM % 32 == 0 && BN % 32 == 0 && S >= 3 && ((MB * NB) % 2 == 0 || MB * NB == 1), "tile shape");

    int tm, tn;
    TileOfBlock<GROUP_M>((int)blockIdx.x, (m + BM - 1) / BM, (n + BN - 1) / BN, tm, tn);
    const int row0 = tm * BM, col0 = tn * BN;
    const int wave = hw::wave(), group = wave >> 2, wm = (wave >> 1) & 1, wn = wave & 1;
    const uint32_t lane = (uint32_t)hw::lane();
    const uint32_t ldsBase = (uint32_t)(uintptr_t)hw::lds_base();
    const uint32_t ld = (uint32_t)k * 2u;
    const int steps = (k + 63) / 64;

    // Copy j of a wave is instruction 8 j + wave of the step: eight rows of the stage's image, A's rows first, then B's.
    // Lane l copies the 16-byte chunk (l % 8) ^ swz(row) of row 8 i + l / 8 to position l % 8 of that row's image, swz(r) =
    // (r / 2) % 8 (no bank conflicts in the fragment reads).  Past the last instruction the wave repeats the last one
    // (same bytes to the same place), so that every wave counts kCopies outstanding copies a step.
    const char *base[kCopies];
    uint32_t off[kCopies], lds[kCopies], offHalf[HALF ? kCopies : 1];
#pragma unroll
    for (int j = 0; j < kCopies; ++j) {
        const int i = 8 * j + wave < kInst ? 8 * j + wave : kInst - 1;
        const bool isA = i < BM / 8;
        const int first = isA ? row0 + 8 * i : col0 + 8 * (i - BM / 8), last = (isA ? m : n) - 1;
        const int row = first + (int)(lane / 8) < last ? first + (int)(lane / 8) : last;
        const int origin = first < last ? first : last;
        const uint32_t chunk = (lane % 8) ^ ((4u * (uint32_t)i + lane / 16) % 8);
        base[j] = detail::uniform_ptr(reinterpret_cast<const char *>(isA ? src0 : src1) + (int64_t)origin * ld);
        off[j] = (uint32_t)(row - origin) * ld + chunk * 16u;
        if constexpr (HALF)
            offHalf[j] = (uint32_t)(row - origin) * ld + (chunk & 3u) * 16u; // the upper 64 bytes are not there (and not used)
        lds[j] = ldsBase + (uint32_t)i * 1024u;
    }
    // the LDS address of a copy goes through M0 (one wait state before its use)
    auto copyOne = [&](int j, int step, uint32_t stageOff) __attribute__((always_inline)) {
        const int s = step < steps ? step : steps - 1; // (past the end: the last step again, into a stage nobody reads)
        const uint32_t o = HALF && s == steps - 1 ? offHalf[HALF ? j : 0] : off[j];
        asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, %2" ::"s"(lds[j] + stageOff), "v"(o), "s"(base[j] + (int64_t)s * 128) : "memory");
    };

    // fragment reads: lane l holds row l % 16 of a block and the k group l / 16 of this wave's 32
    const uint32_t r16 = lane % 16, fragOff = r16 * 128u + ((((uint32_t)group * 4u + lane / 16) ^ ((r16 / 2) % 8)) * 16u);
    const uint32_t aAddr = ldsBase + (uint32_t)(wm * (BM / 2)) * 128u + fragOff;
    const uint32_t bAddr = ldsBase + (uint32_t)(BM + wn * (BN / 2)) * 128u + fragOff;
    ks_f16x8 a[2][MB], b[2][NB];
    auto readStep = [&](auto setTag, uint32_t stageOff) __attribute__((always_inline)) {
        constexpr int set = decltype(setTag)::value;
        StaticFor<0, NB>([&](auto i) __attribute__((always_inline)) { b[set][i] = KsLdsRead16<decltype(i)::value * 2048>(bAddr + stageOff); });
        StaticFor<0, MB>([&](auto i) __attribute__((always_inline)) { a[set][i] = KsLdsRead16<decltype(i)::value * 2048>(aAddr + stageOff); });
    };
    ks_f32x4 acc[MB][NB];
#pragma unroll
    for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j)
            acc[i][j] = ks_f32x4{0.f, 0.f, 0.f, 0.f};

    uint32_t readOff = kStage, copyOff = 0; // of step it + 1, of step it (and it + S)
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int j = 0; j < kCopies; ++j)
            copyOne(j, s, s * kStage);
    hw::wait_vm<(S - 1) * kCopies>();
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory"); // (the barrier alone does not hold loads back from moving ahead of it)
    readStep(std::integral_constant<int, 0>(), 0u);
    KsArrived(a[0], b[0]);

    auto step = [&](auto setTag, auto readTag, int it) __attribute__((always_inline)) {
        constexpr int set = decltype(setTag)::value;
        constexpr bool read = decltype(readTag)::value; // the fragments of step it + 1
        // this wave has read all of step it, its copies of step it + 1 have landed; behind the barrier that is so of every wave
        hw::wait_vm<(S - 2) * kCopies>();
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (read)
            readStep(std::integral_constant<int, 1 - set>(), readOff);
        __builtin_amdgcn_sched_barrier(0);
        const bool mine = !HALF || group == 0 || it < steps - 1;
#pragma unroll
        for (int i = 0; i < MB || i < kCopies; ++i) {
            if (i < MB && mine) {
#pragma unroll
                for (int j = 0; j < NB; ++j)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(b[set][j], a[set][i], acc[i][j], 0, 0, 0);
            }
            __builtin_amdgcn_sched_barrier(0);
            if (i < kCopies)
                copyOne(i, it + S, copyOff);
        }
        copyOff = readOff;
        readOff = readOff + kStage == kRing ? 0u : readOff + kStage;
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (read)
            KsArrived(a[1 - set], b[1 - set]);
    };
    int it = 0;
    for (; it + 2 <= steps; it += 2) { // (past the end it reads fragments that nobody uses)
        step(std::integral_constant<int, 0>(), std::true_type(), it);
        step(std::integral_constant<int, 1>(), std::true_type(), it + 1);
    }
    if (it < steps)
        step(std::integral_constant<int, 0>(), std::false_type(), it);

    // Partial sums: each group keeps half of its wave's blocks (of one block the second group keeps it), gives the other half to its partner (same rows and
    // columns, other k) and stores the sums of the half it keeps.
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory"); // the copies past the end
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    constexpr int kHalfBlocks = MB * NB / 2;
    char *sums = hw::lds_base();
    const int pair = wave & 3;
    StaticFor<0, MB * NB>([&](auto idxTag) __attribute__((always_inline)) {
        constexpr int idx = decltype(idxTag)::value;
        if ((idx < kHalfBlocks) != (group == 0)) // the half that the partner keeps
            *reinterpret_cast<ks_f32x4 *>(sums + ((uint32_t)(pair * MB * NB + idx) * 64u + lane) * 16u) = acc[idx / NB][idx % NB];
    });
    __syncthreads();
    const int rowLane = row0 + wm * (BM / 2) + (int)(lane % 16), colLane = col0 + wn * (BN / 2) + 4 * (int)(lane / 16);
    StaticFor<0, MB * NB>([&](auto idxTag) __attribute__((always_inline)) {
        constexpr int idx = decltype(idxTag)::value, i = idx / NB, j = idx % NB;
        if ((idx < kHalfBlocks) == (group == 0)) {
            const ks_f32x4 v = acc[i][j] + *reinterpret_cast<const ks_f32x4 *>(sums + ((uint32_t)(pair * MB * NB + idx) * 64u + lane) * 16u);
            const int row = rowLane + 16 * i, col = colLane + 16 * j;
            if (row < m && col < n) // n % 4 == 0: four columns are inside together
                StoreFour(out + (int64_t)row * n + col, v, through);
        }
    });
}

} // namespace
PTO_DEVICE_CODE_END

namespace {
template <int BM, int BN, int S, int MIN_WAVES>
int launch_gemm_ks(hipStream_t st, float *c, const half *a, const half *b, int m, int n, int k)
{
    if (n % 4 || k % 32)
        return PTO_ERR_UNSUPPORTED;
    constexpr int lds = KsLdsBytes<BM, BN, S>();
    static_assert(lds <= 160 * 1024, "stages fit the LDS");
    auto whole = GemmF16F32Ks<BM, BN, S, MIN_WAVES, false, 4>;
    auto half64 = GemmF16F32Ks<BM, BN, S, MIN_WAVES, true, 4>;
    static const int attr = lds <= 64 * 1024 ? PTO_OK : (pto_amd::allow_lds(whole, lds) | pto_amd::allow_lds(half64, lds));
    if (attr != PTO_OK)
        return PTO_ERR_HIP;
    const long long tiles = (long long)((m + BM - 1) / BM) * ((n + BN - 1) / BN);
    if (tiles > 0x7fffffffll)
        return PTO_ERR_UNSUPPORTED;
    // (half pieces past the L2 pay while C is small and k short: 1000 x 3000 x 1024 12.5 -> 12.0 us, with a conversion of C behind it 19.5 -> 18.5;
    // 503 x 6088 x 1024 12.0 -> 11.6, 19.8 -> 18.3.  With more to read before, the product gains little and the reader of C loses more: 1000 x 3000 x 1536 15.5 -> 14.3,
    // 20.2 -> 20.9; x 2048 18.4 -> 18.3, 22.5 -> 23.6; 503 x 6088 x 3072 24.2 -> 24.1, 28.4 -> 29.7.  1024 x 6136 x 1024, 25 MB of C, 18.8 and 19.8)
    const uint64_t bytes = 4ull * m * n;
    const int through = pto_amd::store_through(c, 4ull * n, bytes) || (bytes <= 12u << 20 && k <= 1280 && (n * 4ull | (uintptr_t)c) % 32 == 0);
    (k % 64 ? half64 : whole)<<<dim3((unsigned)tiles), dim3(512), lds, st>>>(c, a, b, m, n, k, through);
    return pto_amd::check_launch();
}
} // namespace
