// Row-wise top-k for MI355X: per row, the (score, index) pairs in descending order of score, equal scores in ascending
// order of index, first k of them written as scores and as indices.
//
// Mirrors the reference kernel kernels/manual/a2a3/topk/topk_kernel.cpp:282-345 (launchTopk: TLOAD -> TSORT32 on groups of
// 32 -> TMRGSORT merges of 4 lists -> TGATHER splits scores and indices -> TSTORE) and its golden
// (scripts/gen_data.py:55-64: np.lexsort((idx, -row))[:topk]); the order is the comparator of TSORT32 / TMRGSORT
// (include/pto/cpu/TSort32.hpp:32-41: score descending, then index ascending, -0 == +0).
//
// The reference builds the order from 32-element hardware sorts and 4-way merges in its unified buffer, re-viewing one
// buffer through differently shaped tiles.  On a CDNA4 compute unit the natural form is a bitonic network in registers:
// one wave per row of up to 1024 columns with 2 .. 16 keys per lane, two or four waves for 2048 and 4096.
// * Indices that increase with the column (the reference passes 0, 1, 2, ...): the order is that of (score, -column), 32 +
//   12 bits, which fit the mantissa of a double: key = 1.order(score).(4095 - column).x, always a normal number between 1
//   and 2.  A compare-exchange of two keys in a lane is then v_max_f64 + v_min_f64, two instructions instead of a 64-bit
//   compare and four selects (measured, four waves per SIMD: 1.8 ns each on one SIMD, like v_cndmask and v_cmp_u64).
// * Across lanes the sign does the choosing: before a stage a lane that is to keep the smaller key of a pair negates its
//   key (one v_xor on the upper word); the pair then holds k and -k', and max(own, -received) is right for both lanes.
// * The lanes of a row of 16 are numbered so that the partners of the four lowest lane strides are lane ^ 1, ^ 2, ^ 7, ^ 8:
//   one DPP move for the upper word, and for the lower word another, or the LDS pipe (ds_swizzle), which the network leaves idle
//   otherwise (LOW_DPP, at the dispatch); partners 16 and 32 lanes away come over the LDS pipe whole (v_permlane*_swap: 3.5 ns a word, 4.2 us of the
//   kernel's time for three stages of 55); strides across waves go through LDS memory.
// * topk of an eighth of the padded row length or less: once the sorted runs are as long as topk (rounded up to keys per lane times a power of
//   two), a merge of two runs keeps their larger halves only, in both runs' lanes, and its sort passes no longer cover the
//   dropped half.
// * Any other index vector: the same network sorts the (index, column) pairs first, once per workgroup (the rows share their
//   indices); the rank of a column in that order then stands in the scores' keys for the column.  4800 x 1024 whole: 42 us (127
//   with keys in the LDS and a pass over it per stage); 1000 x 256: 6.6 (15).
// What bounds it: vector instructions, 2520 per row of 1024 (3850 in the integer network this replaced), behind a phase of
// loads and before one of stores that all waves share: of 23.2 us (4800 x 1024, top 1000, 58 MB = 9 us at 6.5 TB/s) 10 are
// launch, loads and stores (five waves on a SIMD instead of four, at 96 registers of 106: 28.0 and 28.2 us on one card).  Persistent waves that load the next row while they sort one, and wave priorities that let
// some run ahead, do not hide them (32 us and no change).
#include <hip/hip_runtime.h>

#include "common.hpp"

namespace {

constexpr int kTopkThreads = 256, kTopkWaves = 4;

__device__ inline uint32_t ScoreOrder(uint32_t bits) { return bits ^ ((uint32_t)((int32_t)bits >> 31) | 0x80000000u); }
__device__ inline uint32_t ScoreBits(uint32_t ord) { return ord ^ ((uint32_t)(~(int32_t)ord >> 31) | 0x80000000u); }

template <int FIRST, int LAST, typename F>
__device__ inline void StaticFor(F &&f)
{
    if constexpr (FIRST < LAST) {
        f(std::integral_constant<int, FIRST>());
        StaticFor<FIRST + 1, LAST>(f);
    }
}

constexpr uint32_t kSign = 0x80000000u;

__device__ inline uint32_t High(double k) { return (uint32_t)(__builtin_bit_cast(uint64_t, k) >> 32); }
__device__ inline uint32_t Low(double k) { return (uint32_t)__builtin_bit_cast(uint64_t, k); }
__device__ inline double Key(uint32_t high, uint32_t low) { return __builtin_bit_cast(double, ((uint64_t)high << 32) | low); }

// (as assembly: the compiler would add instructions that quieten signalling NaNs, and no key is one)
__device__ inline double Max(double a, double b)
{
    double r;
    asm("v_max_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ inline double Min(double a, double b)
{
    double r;
    asm("v_min_f64 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
__device__ inline double MaxOfNegated(double a, double b) // max(a, -b)
{
    double r;
    asm("v_max_f64 %0, %1, -%2" : "=v"(r) : "v"(a), "v"(b));
    return r;
}
// Between instructions written as assembly and lane moves of their results: the compiler does not know that the former
// are vector instructions, so the wait states that a lane move asks for are placed here.
__device__ inline void StageEdge()
{
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_nop 1");
    __builtin_amdgcn_sched_barrier(0);
}

// A word of the partner at lane stride J (of the numbering by LaneRank: lane ^ 1, ^ 2, ^ 7, ^ 8, ^ 16, ^ 32), moved by the
// vector pipe or by the LDS pipe
template <int J>
__device__ inline uint32_t LaneMove(uint32_t v)
{
    static_assert(J < 4, "inside a row of 16 lanes");
    constexpr int kCtrl = J == 0 ? 0xB1 : J == 1 ? 0x4E : J == 2 ? 0x141 : 0x128; // quad_perm twice, row_half_mirror, row_ror:8
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, kCtrl, 0xf, 0xf, true);
}
template <int J>
__device__ inline uint32_t ThroughLds(uint32_t v)
{
    if constexpr (J < 5) {
        constexpr int kXor = J == 0 ? 1 : J == 1 ? 2 : J == 2 ? 7 : J == 3 ? 8 : 16;
        return (uint32_t)__builtin_amdgcn_ds_swizzle((int)v, (kXor << 10) | 0x1f);
    } else {
        return (uint32_t)__builtin_amdgcn_ds_bpermute((int)((threadIdx.x ^ 32u) << 2), (int)v);
    }
}
// the words go through the LDS pipe where the vector pipe would need two moves; else the upper one never, the lower one as the
// launch has it
template <int J>
constexpr bool kFarLane = J >= 4;

// lane = c0 ^ 2 c1 ^ 7 c2 ^ 8 c3 ^ 16 c4 ^ 32 c5  ->  c0 + 2 c1 + 4 c2 + ...
__device__ inline uint32_t LaneRank(uint32_t lane) { return (lane & 4u) ? lane ^ 3u : lane; }

// Sorting of the 64 E W keys of a row, descending; key e of the lane with number q = 64 (wave of the row) + LaneRank(lane) is of
// rank q E + e in the end.  keepBits: the ranks below E << keepBits are wanted.  A key is kept negated where `form` has its
// sign bit set.  xchg: E x 64 keys per wave (W > 1).
template <int E, int W, bool LOW_DPP>
struct RowSort {
    static constexpr int kLaneBits = 6 + (W == 4 ? 2 : W == 2 ? 1 : 0);
    double k[E];
    uint32_t form, q;
    uint64_t *xchg;

    __device__ inline void SetForm(uint32_t f)
    {
        uint32_t d = form ^ f;
        asm("" : "+v"(d)); // (one xor per key: left to itself the compiler applies both terms to every key)
#pragma unroll
        for (int e = 0; e < E; ++e)
            k[e] = Key(High(k[e]) ^ d, Low(k[e]));
        form = f;
    }
    __device__ inline uint32_t Bit(int b) const { return (q >> b & 1u) ? kSign : 0u; }
    // compare-exchange inside the lane: the larger key to the lower register
    __device__ inline void Exchange(double &hi, double &lo)
    {
        const double a = Max(hi, lo), b = Min(hi, lo);
        hi = a;
        lo = b;
    }
    __device__ inline void SortLane() // all E keys, descending in the present form (Batcher's odd-even merge sort: 63 exchanges of 16 keys)
    {
#pragma unroll
        for (int run = 1; run < E; run <<= 1)
#pragma unroll
            for (int j = run; j > 0; j >>= 1)
#pragma unroll
                for (int e = j % run; e + j < E; e += 2 * j)
#pragma unroll
                    for (int i = 0; i < j; ++i)
                        if (e + i + j < E && (e + i) / (2 * run) == (e + i + j) / (2 * run))
                            Exchange(k[e + i], k[e + i + j]);
    }
    __device__ inline void MergeLane() // a bitonic sequence of E keys
    {
#pragma unroll
        for (int j = E >> 1; j > 0; j >>= 1)
#pragma unroll
            for (int e = 0; e < E; ++e)
                if ((e & j) == 0)
                    Exchange(k[e], k[e | j]);
    }
    // partners at lane stride J: the lane whose bit is clear keeps the larger key where dir is 0.  BOTH: either keeps the larger
    template <int J, bool BOTH>
    __device__ inline void Stage(uint32_t dir)
    {
        if constexpr (J < 6) {
            SetForm(BOTH ? 0u : dir ^ Bit(J));
            StageEdge();
            uint32_t low[E], high[E];
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if constexpr (kFarLane<J> || !LOW_DPP)
                    low[e] = ThroughLds<J>(Low(k[e]));
                if constexpr (kFarLane<J>)
                    high[e] = ThroughLds<J>(High(k[e]));
            }
#pragma unroll
            for (int e = 0; e < E; ++e) {
                if constexpr (!kFarLane<J>)
                    high[e] = LaneMove<J>(High(k[e]));
                if constexpr (!kFarLane<J> && LOW_DPP)
                    low[e] = LaneMove<J>(Low(k[e]));
                const double o = Key(high[e], low[e]);
                k[e] = BOTH ? Max(k[e], o) : MaxOfNegated(k[e], o);
            }
        } else if constexpr (J < kLaneBits) { // another wave of the row
            SetForm(BOTH ? 0u : dir ^ Bit(J));
            const uint32_t wave = threadIdx.x / 64, lane = threadIdx.x % 64, other = wave ^ (1u << (J - 6));
            __syncthreads(); // everyone is done with the exchange before
#pragma unroll
            for (int e = 0; e < E; ++e)
                xchg[(wave * E + e) * 64 + lane] = __builtin_bit_cast(uint64_t, k[e]);
            __syncthreads();
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const double o = __builtin_bit_cast(double, xchg[(other * E + e) * 64 + lane]);
                k[e] = BOTH ? Max(k[e], o) : MaxOfNegated(k[e], o);
            }
        }
        StageEdge();
    }
    // MOST: the largest keepBits there is; kLaneBits for a whole sort, whose code then holds no branch
    template <int MOST>
    __device__ inline __attribute__((always_inline)) void Sort(int keepBits)
    {
        SetForm(Bit(0));
        StageEdge();
        SortLane();
        StageEdge();
        // (straight-line code: one copy for all runs branches around its stages, 8 to 15 % of the time at 8 and 16 keys per lane
        // where topk is small, 2 to 6 % of a whole sort)
        StaticFor<1, kLaneBits + 1>([&](auto run) { Merge<decltype(run)::value, MOST>(MOST == kLaneBits ? kLaneBits : keepBits); });
    }
    // runs of E << RUN keys out of two of half the length, descending and ascending in turn (the last: descending)
    template <int RUN, int MOST>
    __device__ inline __attribute__((always_inline)) void Merge(int keepBits)
    {
        const uint32_t dir = RUN == kLaneBits ? 0u : Bit(RUN);
        int strides = RUN;
        if (RUN > MOST || RUN > keepBits) {
            strides = keepBits;
            Stage<RUN - 1, true>(dir);
        }
        StaticFor<0, RUN>([&](auto below) {
            constexpr int j = RUN - 1 - decltype(below)::value;
            if (j < MOST && strides > j)
                Stage<j, false>(dir);
        });
        SetForm(dir);
        StageEdge();
        MergeLane();
        StageEdge();
    }
};

// E keys per lane, W waves per row (the row is padded to 64 E W keys; padding keys lie below every real one), 4 / W rows per
// workgroup.  WHOLE: a whole sort, otherwise keepBits is below the row's by more than kWholeBits.  Where more than an eighth of
// the row is wanted the merges save less than their branches cost (cut to keepBits / whole sort: 1024 columns, 600 rows, top 256
// 7.4 / 7.2 us, 4800 rows 21.6 / 21.6; 128 x 256, top 64 3.7 / 3.3, top 256 4.0 / 3.6; 4800 x 1024, top 1024 26.0 / 25.5).
constexpr int kWholeBits = 2;
// one key per lane and four waves per row: for few rows of which more than 16 are wanted, where the whole sort is the shorter one
template <int E, int W>
constexpr bool kOnlyWhole = E == 1 && W == 4;
template <int E, int W, bool LOW_DPP, bool WHOLE>
__global__ __launch_bounds__(kTopkThreads) void TopkRows(float *outScore, uint32_t *outIndex, const float *src, const uint32_t *inIdx,
                                                         int rows, int validCols, int ld, int topk, int keepBits, int through)
{
    constexpr int N = 64 * E * W, kRows = kTopkWaves / W, kBits = RowSort<E, W, LOW_DPP>::kLaneBits;
    constexpr int kStaged = 64 * E + 4 * E; // words of a wave's results, one of padding behind every 16
    constexpr int kStages = E <= 8 ? 2 : 1;  // scores and columns side by side, or one after the other (LDS for four workgroups more)
    // exchanges, then results (or, between two sorts, the ranks of the columns); behind them the columns in the order of their indices
    constexpr size_t kExchange = W > 1 ? (size_t)kTopkWaves * E * 64 * 8 : 0, kStage = (size_t)kTopkWaves * kStaged * 4 * kStages;
    constexpr size_t kWork = kExchange > kStage ? kExchange : kStage;
    static_assert(kWork >= (size_t)N * 2, "the ranks fit");
    __shared__ __attribute__((aligned(16))) char lds[kWork + (size_t)N * 2];
    uint16_t *rankOf = reinterpret_cast<uint16_t *>(lds), *columnOf = reinterpret_cast<uint16_t *>(lds + kWork);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int waveOfRow = wave % W, row0 = (int)blockIdx.x * kRows, row = row0 + wave / W < rows ? row0 + wave / W : rows - 1;
    uint32_t i0 = (uint32_t)(waveOfRow * E * 64 + lane); // this lane's first column; then every 64th

    // A lane past the last column looks at the last one: loads without branches are all in flight at once (16 of them one
    // behind the other were half of the kernel's time).  Up to four keys and few waves: always so, the branch around
    // it takes longer (1 x 200, top 16: 3.29 / 3.18 us; with many waves 8192 x 256, top 8: 6.4 / 6.7)
    constexpr bool kClamp = E <= 4 && LOW_DPP;
    auto load = [&](const uint32_t *from, uint32_t (&to)[E]) __attribute__((always_inline)) {
        if (!kClamp && validCols == N) {
#pragma unroll
            for (int e = 0; e < E; ++e)
                to[e] = from[i0 + e * 64];
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e)
                to[e] = from[i0 + e * 64 < (uint32_t)validCols ? i0 + e * 64 : (uint32_t)validCols - 1u];
        }
    };
    uint32_t bits[E], ids[E];
    const uint32_t *scores = reinterpret_cast<const uint32_t *>(src) + (size_t)row * (size_t)ld;
    load(scores, bits);
    load(inIdx, ids);

    // are the indices first, first + 1, ... or at least increasing with the column?  (then the column decides among equal
    // scores, as the index would; the same answer in every wave of the workgroup)
    const uint32_t first = inIdx[0];
    uint32_t wrong = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t at = i0 + e * 64 < (uint32_t)validCols ? i0 + e * 64 : (uint32_t)validCols - 1u;
        wrong |= (ids[e] - first) ^ at;
    }
    auto everyone = [&](bool v) { return W > 1 ? __syncthreads_and(v) != 0 : __builtin_amdgcn_ballot_w64(!v) == 0; };
    const bool consecutive = everyone(wrong == 0 && first <= 0xffffffffu - (uint32_t)validCols);
    bool increasing = consecutive;
    if (__builtin_expect(!consecutive, 0)) {
        bool ok = true;
        for (int e = 0; e < E; ++e) {
            const int i = (int)i0 + e * 64;
            if (i + 1 < validCols)
                ok = ok && inIdx[i] < inIdx[i + 1];
        }
        increasing = everyone(ok);
    }
    RowSort<E, W, LOW_DPP> s;
    s.q = (uint32_t)waveOfRow * 64u + LaneRank((uint32_t)lane);
    s.xchg = reinterpret_cast<uint64_t *>(lds);
    // the ranks of a wave go in order through its piece of LDS, so that its stores cover consecutive addresses
    uint32_t *staged = reinterpret_cast<uint32_t *>(lds) + wave * (kStaged * kStages), *stagedColumn = staged + (kStages - 1) * kStaged;
    const int firstRank = waveOfRow * 64 * E, laneRank = (int)LaneRank((uint32_t)lane) * E, count = topk - firstRank;
    auto ordered = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
    const uint32_t columnBits = (4095u - i0) << 8;
    if (__builtin_expect(!increasing, 0)) { // the columns in the order of their indices; rows of one wave: the first wave does it for all four
        if (W > 1 || wave == 0) {
            s.form = 0;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const uint32_t order = ~ids[e];
                s.k[e] = Key(__builtin_amdgcn_alignbit(0x3ffu, order, 12), (order << 20) | (columnBits - (uint32_t)(e * 64 << 8)));
                if (i0 + e * 64 >= (uint32_t)validCols)
                    s.k[e] = 1.0;
            }
            s.template Sort<kBits>(kBits);
            asm volatile("" : "+v"(i0), "+v"(s.q)); // (nothing that depends on them is kept in registers across the sort)
            if (W > 1)
                __syncthreads(); // (the exchanges are over)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const uint32_t rank = s.q * E + e, column = 4095u - ((Low(s.k[e]) >> 8) & 0xfffu);
                if (wave < W && rank < (uint32_t)validCols) {
                    rankOf[column] = (uint16_t)rank;
                    columnOf[rank] = (uint16_t)column;
                }
            }
        }
        load(scores, bits);
    }
    s.form = 0;
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const bool negZero = bits[e] == kSign; // compares equal to +0: same key, remembered below the column bits
        const uint32_t order = ScoreOrder(negZero ? 0u : bits[e]);
        s.k[e] = Key(__builtin_amdgcn_alignbit(0x3ffu, order, 12), (order << 20) | (columnBits - (uint32_t)(e * 64 << 8) + (negZero ? 1u : 0u)));
    }
    if (__builtin_expect(!increasing, 0)) {
        __syncthreads(); // the ranks are there
#pragma unroll
        for (int e = 0; e < E; ++e)
            s.k[e] = Key(High(s.k[e]), (Low(s.k[e]) & 0xfff000ffu) | (4095u - rankOf[i0 + e * 64]) << 8); // (past the row's end: overwritten below)
        __syncthreads(); // and read, before their memory is used for something else
    }
    if (kClamp || validCols != N) {
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (i0 + e * 64 >= (uint32_t)validCols)
                s.k[e] = 1.0;
    }
    s.template Sort<WHOLE ? kBits : kBits - kWholeBits - 1>(keepBits);

    if (W > 1)
        __syncthreads(); // (the exchanges are over)
    if (row0 + wave / W >= rows || count <= 0)
        return;
    uint32_t *toScore = reinterpret_cast<uint32_t *>(outScore) + (size_t)row * (size_t)topk + firstRank;
    uint32_t *toIndex = outIndex + (size_t)row * (size_t)topk + firstRank;
    // lane by lane consecutive words; through: past the L2 (launch_topk)
    auto store = [&](uint32_t *to, auto &&word) __attribute__((always_inline)) {
        if (through) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = e * 64 + lane;
                if (i < count)
                    __hip_atomic_store(to + i, word(i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
            }
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const int i = e * 64 + lane;
                if (i < count)
                    to[i] = word(i);
            }
        }
    };
    uint32_t column[E];
#pragma unroll
    for (int e = 0; e < E; ++e) {
        const uint32_t low = Low(s.k[e]), order = (High(s.k[e]) << 12) | (low >> 20);
        column[e] = 4095u - ((low >> 8) & 0xfffu);
        staged[laneRank + e + (laneRank + e) / 16] = (low & 1u) ? kSign : ScoreBits(order);
        if (kStages == 2)
            stagedColumn[laneRank + e + (laneRank + e) / 16] = column[e];
    }
    ordered();
    store(toScore, [&](int i) { return staged[i + i / 16]; });
    if (kStages == 1) {
        ordered();
#pragma unroll
        for (int e = 0; e < E; ++e)
            stagedColumn[laneRank + e + (laneRank + e) / 16] = column[e];
        ordered();
    }
    if (__builtin_expect(!consecutive, 0)) { // (staged: the column, or its rank)
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const int i = e * 64 + lane;
            if (i < count) {
                const uint32_t c = stagedColumn[i + i / 16];
                toIndex[i] = inIdx[increasing ? c : columnOf[c]];
            }
        }
        return;
    }
    store(toIndex, [&](int i) { return first + stagedColumn[i + i / 16]; });
}

template <int E, int W>
int launch_topk(hipStream_t st, float *out_score, uint32_t *out_index, const float *src, const uint32_t *in_idx, int rows, int valid_cols, int ld,
                int topk)
{
    int keepBits = 0;
    while ((E << keepBits) < topk)
        ++keepBits;
    const bool whole = kOnlyWhole<E, W> || keepBits + kWholeBits >= RowSort<E, W, true>::kLaneBits;
    // Lower words between near lanes: with up to four waves on a SIMD the latency of the LDS pipe shows, a DPP move is shorter
    // (LDS / DPP, whole sorts: 300 x 128 3.48 / 3.26 us, 300 x 256 4.53 / 4.28); with more the moves take issue slots (4800 x 128
    // 5.09 / 5.23).  8 and 16 keys per lane cover the latency either way and take DPP.
    const bool dpp = E >= 8 || (long long)rows * W <= 4 * 4 * pto_amd::compute_units();
    constexpr bool kCut = kOnlyWhole<E, W>, kDpp = E >= 8 || kOnlyWhole<E, W>; // (names the one form that there is)
    auto kernel = dpp ? (whole ? TopkRows<E, W, true, true> : TopkRows<E, W, true, kCut>) :
                        (whole ? TopkRows<E, W, kDpp, true> : TopkRows<E, W, kDpp, kCut>);
    // Results past the L2: a kernel ends with every L2 writing back what is dirty in it, 3 us for the 38 MB of 4800 x 1000 (25.4 ->
    // 23.3 us; 8192 x 500, top 333 19.2 -> 17.0; 300 x 128 whole 2.69 -> 2.67).  Not where a row's results are less than a store
    // instruction's 256 bytes (8192 x 64, top 1 3.2 / 3.7, 131072 x 64, top 33 32.6 / 34.1), nor where they are much more than the L2s'
    // 32 MB, which then are written back while others sort (30000 x 2048, top 1500 261 / 268).
    const int through = topk >= 64 && 8ll * rows * topk <= 1ll << 26;
    constexpr int kRows = kTopkWaves / W;
    kernel<<<dim3((unsigned)(((long long)rows + kRows - 1) / kRows)), dim3(kTopkThreads), 0, st>>>(out_score, out_index, src, in_idx, rows, valid_cols,
                                                                                                   ld, topk, keepBits, through);
    return pto_amd::check_launch();
}

} // namespace

extern "C" int pto_topk_f32(void *stream, float *out_score, uint32_t *out_index, const float *src, const uint32_t *in_idx, int rows,
                            int valid_cols, int ld, int topk)
{
    if (!out_score || !out_index || !src || !in_idx || rows <= 0 || valid_cols <= 0 || topk <= 0)
        return PTO_ERR_BAD_ARG;
    if (ld < valid_cols || topk > valid_cols || valid_cols > 4096)
        return PTO_ERR_UNSUPPORTED;
    hipStream_t st = static_cast<hipStream_t>(stream);
    // Waves per row.  One wave per row does the least work, more put more of the chip to work on few rows (one / two / four waves,
    // whole sorts: 1024 columns, 600 rows 9.8 / 8.8 / 7.7 us, 1000 rows 10.3 / 9.3 / 9.2, 2400 rows 17.5 / 16.2 / 17.9, 4800
    // rows 25.3 / 26.9 / 28.8; 1000 rows top 256 8.7 / 8.1 / 8.2): on 256 units four up to 853 rows, two up to 2560.  512 columns:
    // four up to 731 rows (600 rows 5.7 / 5.4 / 5.1, 853 rows 5.8 / 5.5 / 5.6, top 15 4.5 / 4.6 / 5.1), then one.  2048 columns: four
    // up to 1706 rows (1700 rows with two 25.6, with four 24.5; 2000 rows 26.2, 26.9).  129 to 256 columns: four up to 365 rows where
    // more than 16 are wanted (one / four: 128 rows 3.6 / 3.3, 300 rows 3.6 / 3.4, 600 rows 3.7 / 3.7; top 7 of 128 rows 3.2 / 3.6).
    const int most = 5 * 4 * pto_amd::compute_units() / rows; // waves per row for five on every SIMD
#define PTO_TOPK_CASE(E, W) return launch_topk<E, W>(st, out_score, out_index, src, in_idx, rows, valid_cols, ld, topk);
    if (valid_cols <= 64)
        PTO_TOPK_CASE(1, 1)
    if (valid_cols <= 128)
        PTO_TOPK_CASE(2, 1)
    if (valid_cols <= 256) {
        if (most >= 14 && topk > 16)
            PTO_TOPK_CASE(1, 4)
        PTO_TOPK_CASE(4, 1)
    }
    if (valid_cols <= 512) {
        if (most >= 7)
            PTO_TOPK_CASE(2, 4)
        PTO_TOPK_CASE(8, 1)
    }
    if (valid_cols <= 1024) {
        if (most >= 6)
            PTO_TOPK_CASE(4, 4)
        if (most >= 2)
            PTO_TOPK_CASE(8, 2)
        PTO_TOPK_CASE(16, 1)
    }
    if (valid_cols <= 2048) {
        if (most >= 3)
            PTO_TOPK_CASE(8, 4)
        PTO_TOPK_CASE(16, 2)
    }
    PTO_TOPK_CASE(16, 4)
#undef PTO_TOPK_CASE
}
