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
// * Few of many (topk of an eighth of the padded row or less, 257 columns or more): a threshold first, then only the keys that reach it are sorted.  The
//   topk-th largest of the maxima of disjoint groups of keys (64 to 256 groups a wave) is no larger than the topk-th largest key, and not much more
//   than topk keys reach it (of 1024, 256 groups: 68 for topk 60).  It is found by halving an interval of the scores' order, the groups that reach
//   the middle counted by ballots; those keys go into a list in the LDS and through the network of 64, 128, 256 or 512 keys in one wave.
//   Where too many keys equal the threshold (masked rows), as many of them as are wanted are taken in the order of their columns; where that does
//   not do either, or the indices do not increase, the row is sorted as before.  4800 x 1024, top 40 18.7 -> 6.9 us (all equal but 2 % 18.5 -> 7.9);
//   600 x 2048, top 100 10.8 -> 7.1 (ascending 5.9, masked from the middle on 7.4); 600 x 4096, top 100 18.3 -> 7.9.
// * Whole sorts of 257 columns and more (BucketSort): the keys are counted into buckets and put in place, two and more in a bucket by a few exchanges of
//   neighbours; rows too uneven for that go through the network.  4800 x 1024, top 1000 21.2 -> 14.2 us, 1 x 4096 whole 12.5 -> 7.9, 2400 x 2048 26.6 -> 16.9.
// * Any other index vector: the (index, column) pairs are sorted first, once per workgroup (the rows share their
//   indices), by buckets where the indices are below 2^24 and the columns 257 to 2048, or by the network; the rank of a column in that order then stands in
//   the scores' keys for the column.  4800 x 1024 whole: 30 us, 35 with indices of any size (both by the network 40, with keys in the LDS and a pass over it
//   per stage 127); 1000 x 256: 6.6 (15).  Scores by buckets where a row is one wave's; with more waves they go through the network.
// What bounds the network: vector instructions, 2520 per row of 1024 (3850 in the integer network this replaced), behind a phase of
// loads and before one of stores that all waves share (five waves on a SIMD instead of four: no change; persistent waves that load the next row while they sort
// one, and wave priorities that let some run ahead, do not hide them: 32 us and no change).  By buckets 4800 x 1024, top 1000 (58 MB = 9 us at 6.5 TB/s)
// is bound by the launch, the loads and the stores, with 1210 vector and 142 LDS instructions a row between them (SQ_INSTS_VALU, SQ_INSTS_LDS; the LDS is busy for 760 clocks a row,
// 6 us in all, half of them where counters of one bank meet).
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
// kCut: merges that keep what topk asks for; kSelect: by a threshold, kCut where that fails.  What bounds kSelect (4800 x 1024, top 40, 6.9 us):
// the launch, the 20 MB of the rows (3.1 us at 6.5 TB/s), and 480 vector and 280 scalar instructions a row (the whole network: 2520 vector ones).  Four places of the interval at a time instead
// of one took 2.2 us more (scalar instructions), positions in the list by ballots instead of one scan over the lanes 1.2.
constexpr int kMostSelected = 8; // times 64 keys
enum Mode { kCut, kWhole, kSelect, kCountedCut }; // (the last: by buckets, kCut where that fails)
// whole sorts by buckets first
template <int E, int W>
constexpr bool kBuckets = E >= 4 && E * W >= 8;
// the largest value of the wave, the same in every lane's scalar registers; the sum up to and with this lane
__device__ inline uint32_t WaveMax(uint32_t v)
{
    auto with = [&](uint32_t o) { v = o > v ? o : v; };
    with(LaneMove<0>(v));
    with(LaneMove<1>(v));
    with(LaneMove<2>(v));
    with(LaneMove<3>(v));
    with((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false)); // row_bcast:15
    with((uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false)); // row_bcast:31
    return (uint32_t)__builtin_amdgcn_readlane((int)v, 63);
}
__device__ inline uint32_t WaveScan(uint32_t v)
{
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x111, 0xf, 0xf, false); // row_shr:1, 2, 4, 8
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x112, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x114, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x118, 0xf, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x142, 0xa, 0xf, false);
    v += (uint32_t)__builtin_amdgcn_update_dpp(0, (int)v, 0x143, 0xc, 0xf, false);
    return v;
}
// the key of a score: its order, the column's bits (behind equal scores the lower column, with the larger ones, comes first)
__device__ inline double TopkKey(uint32_t bits, uint32_t columnBits)
{
    const bool negZero = bits == kSign; // compares equal to +0: same key, remembered below the column bits
    const uint32_t order = ScoreOrder(negZero ? 0u : bits);
    return Key(__builtin_amdgcn_alignbit(0x3ffu, order, 12), (order << 20) | (columnBits + (negZero ? 1u : 0u)));
}
__device__ inline float Larger(float a, float b, float c)
{
    float r;
    asm("v_max3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
__device__ inline float Smaller(float a, float b, float c)
{
    float r;
    asm("v_min3_f32 %0, %1, %2, %3" : "=v"(r) : "v"(a), "v"(b), "v"(c));
    return r;
}
// the largest and the smallest value of the wave, in every lane (quad_perm twice, row_half_mirror, row_mirror, row_bcast:15 and :31, of which the last lane has
// both; the two chains side by side, each with the wait states that a lane move asks for)
__device__ inline void WaveEnds(float &hi, float &lo)
{
#define PTO_TOPK_BOTH(move) "v_max_f32_dpp %0, %0, %0 " move "\n\tv_min_f32_dpp %1, %1, %1 " move "\n\ts_nop 0\n\t"
    asm volatile("s_nop 1\n\t" PTO_TOPK_BOTH("quad_perm:[1,0,3,2] row_mask:0xf bank_mask:0xf") PTO_TOPK_BOTH("quad_perm:[2,3,0,1] row_mask:0xf bank_mask:0xf")
                     PTO_TOPK_BOTH("row_half_mirror row_mask:0xf bank_mask:0xf") PTO_TOPK_BOTH("row_mirror row_mask:0xf bank_mask:0xf")
                         PTO_TOPK_BOTH("row_bcast:15 row_mask:0xa bank_mask:0xf") PTO_TOPK_BOTH("row_bcast:31 row_mask:0xc bank_mask:0xf") "s_nop 0"
                 : "+v"(hi), "+v"(lo));
#undef PTO_TOPK_BOTH
    hi = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, hi), 63));
    lo = __builtin_bit_cast(float, __builtin_amdgcn_readlane(__builtin_bit_cast(int, lo), 63));
}

// Sorting of the 64 E W keys of a row, descending, by counting: the scores are spread evenly over 2 N buckets between the row's largest
// and its smallest one, the keys in each are counted, sums over the counts say where a bucket begins, every key goes to the next place of its
// bucket in a list, and neighbours change places (odd and even pairs in turn) as often as the fullest bucket has keys (5 to 9 of 1024 random scores).
// 2 N counters of 16 bits: with N of them buckets hold twice as many keys.  Which rows: any whose scores are finite and not crowded in a small part of
// their range; the others go through the network, found by a look at 64 scores of each wave before anything is counted (masked with infinities, half zeros, most squares,
// wide exponentials), or by the count before anything is scattered (forty close scores among spread ones, a twentieth equal).  Microseconds, whole rows, network alone / turned away by
// the look / by the count / buckets of normal scores: 4800 x 1024 21.1 / 22.1 / 24.9 / 14.7; 2400 x 1024 13.9 / 14.1 / 16.1 / 9.8; 600 x 1024 7.5 / 7.6 / 8.6 / 5.6; 100 x 1024 5.4 / 5.5 /
// 6.4 / 4.8; 1600 x 2048 21.2 / 21.5 / 24.2 / 12.0; 300 x 2048 9.6 / 10.0 / 11.8 / 6.8; 9000 x 512 16.9 / 18.2 / 20.7 / 11.8; 1200 x 4096 33.5 / 35.2 / 39.0 / 19.7; 16 x 4096 13.5 /
// 14.0 / 15.8 / 8.7 (a count that is found wanting only behind the scatter and a pass took 1.25 to 1.4 times the network's, up to 1.8 where the look saw less).  Equal scores:
// bfloat16 ones 1200 x 4096 23.3, 16 x 4096 10.8; sixty distinct ones 4800 x 1024 15.3, 2000 x 777 9.1 (network 12.4).  Tried for uneven rows and slower than the network: 64 of the
// row's own scores, sorted, as the limits of ranges that are spread evenly each (4800 x 1024 27 us); tried for masked ones: infinities and equal scores among the 64 told from the others before
// the range is (masked 22.2 -> 21.5, normal 14.75 -> 15.0).  512 columns in up to 731 rows stay with the network (4.2 us; by
// buckets 4.5 in two waves a row, 4.5 in one), as do 256 and less.
// bits[e]: the score in column i0 + 64 e; afterwards key e of the lane with number q = 64 (wave of the row) + lane is of rank q E + e.
// RANKS: rankOf[column] decides among equal scores and is returned in the column's place.
// mem: 8 N bytes for the row; across: four sets of a word per wave of the workgroup.
// Is it so in every lane of the workgroup?  One barrier (__syncthreads_and: three, and an atomic).  votes: a word per wave, another set of them for the next vote
__device__ inline bool Everyone(bool v, uint32_t *votes)
{
    votes[threadIdx.x / 64] = __builtin_amdgcn_ballot_w64(!v) == 0;
    __syncthreads();
    static_assert(kTopkWaves == 4, "four words");
    return __builtin_amdgcn_readfirstlane((int)(votes[0] & votes[1] & votes[2] & votes[3])) != 0;
}
__device__ inline bool WholeWave(bool v) { return __builtin_amdgcn_ballot_w64(!v) == 0; }

enum Counted { kSorted, kNothingDone, kLost }; // kNothingDone: scores too uneven, or some not finite; kLost: the same, and bits is gone
template <int E, int W>
struct BucketSort {
    static constexpr int N = 64 * E * W, kLogN = __builtin_ctz(N);
    // of 64 scores, in a 128th of the range.  (Exponentially distributed ones have 4 there, squares of normal ones 14 to 16; where four waves look, one is enough to turn a row
    // away.  10 everywhere: 4800 x 1024 exponential scores 17.3 us instead of 14.9, 600 x 2500 18.0 instead of 13.1, squares 23.1 and 23.2 instead of 23.8 and 25.1)
    static constexpr int kCrowd = E == 4 ? 10 : N == 4096 ? 15 : 13;
    static constexpr int kSurely = 16, kMost = E == 4 ? 16 : E == 8 ? 24 : 48; // keys in a bucket: up to kMost by neighbours; more than kSurely may be equal ones
    static constexpr int kTries = 4; // passes where more than kMost are taken for equal ones
    double k[E];

    static __device__ inline void Meet()
    {
        if constexpr (W > 1) {
            __syncthreads();
        } else {
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            __builtin_amdgcn_wave_barrier();
        }
    }
    // where place p of the list (and word w of the counters, four at a time) stands, so that lanes E apart meet in no bank
    static __device__ inline uint32_t Place(uint32_t p) { return p ^ ((p >> 5) & (uint32_t)(E - 1)); }
    static __device__ inline uint32_t Word(uint32_t w) { return w ^ ((w >> 4) & (uint32_t)(E - 4)); }
    // how many scores are equal to the one 64 or 128 columns before, in the row (more than one wave to it: in all rows of the workgroup)
    static __device__ inline int Equal(const uint32_t (&bits)[E], uint32_t i0, int validCols, [[maybe_unused]] uint32_t *counts)
    {
        asm volatile("" : "+v"(i0)); // (no mask of the columns is kept in registers for this)
        uint32_t mine = 0;
#pragma unroll
        for (int e = 1; e < E; ++e)
            if (i0 + 64u * (uint32_t)e < (uint32_t)validCols)
                mine += (uint32_t)(bits[e] == bits[e - 1]) + (e > 1 ? (uint32_t)(bits[e] == bits[e > 1 ? e - 2 : 0]) : 0u);
        int n = __builtin_amdgcn_readlane((int)WaveScan(mine), 63);
        if constexpr (W > 1) {
            counts[threadIdx.x / 64] = (uint32_t)n;
            __syncthreads();
            n = 0;
#pragma unroll
            for (int w = 0; w < kTopkWaves; ++w)
                n += (int)counts[w];
            n = __builtin_amdgcn_readfirstlane(n);
        }
        return n;
    }
    // the neighbours' keys across the lanes' borders: the first key of the lane above, the last one of the lane below
    __device__ inline void Neighbours(double &above, double &below, int waveOfRow, int lane, uint64_t *edges)
    {
        StageEdge();
        above = Key((uint32_t)__builtin_amdgcn_update_dpp(0, (int)High(k[0]), 0x130, 0xf, 0xf, false), // wave_shl:1
                    (uint32_t)__builtin_amdgcn_update_dpp(0, (int)Low(k[0]), 0x130, 0xf, 0xf, false));
        below = Key((uint32_t)__builtin_amdgcn_update_dpp(0x40000000, (int)High(k[E - 1]), 0x138, 0xf, 0xf, false), // wave_shr:1
                    (uint32_t)__builtin_amdgcn_update_dpp(0, (int)Low(k[E - 1]), 0x138, 0xf, 0xf, false));
        if constexpr (W > 1) { // edges: the first and the last key of each wave of the row
            if (lane == 0)
                edges[2 * waveOfRow] = __builtin_bit_cast(uint64_t, k[0]);
            if (lane == 63)
                edges[2 * waveOfRow + 1] = __builtin_bit_cast(uint64_t, k[E - 1]);
            __syncthreads();
            if (lane == 63 && waveOfRow + 1 < W)
                above = __builtin_bit_cast(double, edges[2 * (waveOfRow + 1)]);
            if (lane == 0 && waveOfRow > 0)
                below = __builtin_bit_cast(double, edges[2 * (waveOfRow - 1) + 1]);
        }
    }
    static __device__ inline void Exchange(double &hi, double &lo)
    {
        const double a = Max(hi, lo), b = Min(hi, lo);
        hi = a;
        lo = b;
    }

    template <bool RANKS = false>
    __device__ inline __attribute__((always_inline)) Counted Sort(const uint32_t (&bits)[E], uint32_t i0, int validCols, int waveOfRow, int lane, uint32_t *mem, uint32_t *across, [[maybe_unused]] const uint16_t *rankOf = nullptr)
    {
        const uint32_t q = (uint32_t)(waveOfRow * 64 + lane), wave = threadIdx.x / 64;
        // the range
        auto score = [&](int e) { return __builtin_bit_cast(float, bits[e]); };
        float top = score(0), low = score(0);
#pragma unroll
        for (int e = 0; e < E; e += 2) {
            top = Larger(top, score(e), score(e + 1));
            low = Smaller(low, score(e), score(e + 1));
        }
        WaveEnds(top, low);
        float range = top - low;
        // a look at 64 scores of each wave (four columns in turn, a quarter of its columns apart) before anything else is done: how many are near the ends of the
        // range, or near either of two of them
        bool even = (range >= 1e-30f) & (range <= 1e37f);
        {
            uint32_t second = bits[E / 4], fourth = bits[3 * E / 4];
            asm("" : "+v"(second), "+v"(fourth)); // (else the choice is made between their addresses, and bits put into memory)
            uint32_t seen = (lane & 1) ? second : bits[0], further = (lane & 1) ? fourth : bits[E / 2];
            asm("" : "+v"(further));
            seen = (lane & 2) ? further : seen;
            if (validCols != N) // (what stands behind the last column is near nothing)
                seen = i0 + 16u * E * ((uint32_t)lane & 3u) < (uint32_t)validCols ? seen : 0x7fffffffu;
            const float x = __builtin_bit_cast(float, seen);
            auto few = [&](float distance, float within) __attribute__((always_inline)) { return __builtin_popcountll(__builtin_amdgcn_ballot_w64(distance <= range * within)) < kCrowd; };
            even &= few(top - x, 1.0f / 128.0f) & few(x - low, 1.0f / 128.0f);
#pragma unroll
            for (int g = 0; g < 2; ++g)
                even &= few(__builtin_fabsf(x - __builtin_bit_cast(float, __builtin_amdgcn_readlane((int)seen, g == 0 ? 9 : 38))), 1.0f / 256.0f);
            if (validCols != N) // (a wave that has nothing behind the last column)
                even = even || (int)i0 - lane + 64 >= validCols;
        }
        if (W > 1 ? !Everyone(even, across) : !WholeWave(even))
            return kNothingDone;
        // counters of buckets w and N + w in word w; behind them W words for each of a few exchanges
        uint32_t *const count = mem, *const each = mem + N;
#pragma unroll
        for (int c = 0; c < E / 4; ++c)
            reinterpret_cast<uint4 *>(count)[(waveOfRow * (E / 4) + c) * 64 + lane] = make_uint4(0, 0, 0, 0);
        if constexpr (W > 1) {
            reinterpret_cast<float *>(each)[waveOfRow] = top;
            reinterpret_cast<float *>(each)[W + waveOfRow] = low;
        }
        Meet();
        if constexpr (W > 1) {
#pragma unroll
            for (int w = 0; w < W; ++w) {
                top = __builtin_fmaxf(top, reinterpret_cast<const float *>(each)[w]);
                low = __builtin_fminf(low, reinterpret_cast<const float *>(each)[W + w]);
            }
            range = top - low;
        }
        const float scale = (float)(2 * N - 1) * __builtin_amdgcn_rcpf(range);
        auto isColumn = [&](int e) { return i0 + 64u * (uint32_t)e < (uint32_t)validCols; };
        uint32_t at[E], one[E];
        float odd = range <= 1e37f ? 0.0f : __builtin_nanf(""); // a NaN where a score is none
#pragma unroll
        for (int e = 0; e < E; ++e) {
            // (both steps round larger and smaller scores the same way: no score passes another)
            const uint32_t b = (uint32_t)((top - score(e)) * scale);
            odd = __builtin_fmaf(score(e), 0.0f, odd);
            one[e] = 1u << ((b >> (kLogN - 4)) & 16u);
            at[e] = Word(b & (uint32_t)(N - 1));
        }
        if (validCols != N) {
#pragma unroll
            for (int e = 0; e < E; ++e) {
                one[e] = isColumn(e) ? one[e] : 0u;
                at[e] = isColumn(e) ? at[e] : q; // (many lanes at one counter would wait for each other)
            }
        }
#pragma unroll
        for (int e = 0; e < E; ++e)
            __hip_atomic_fetch_add(count + at[e], one[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        Meet();
        // where the buckets begin, both halves of a word at once (no sum is above 4096); the upper half behind all of the lower one
        uint32_t full = 0; // keys in the fullest bucket
        {
            uint4 *const mine = reinterpret_cast<uint4 *>(count) + q * (E / 4);
            auto chunk = [&](int j) { return Word(q * E + 4 * j) / 4 - q * (E / 4); };
            uint32_t c[E], sum = 0;
#pragma unroll
            for (int j = 0; j < E / 4; ++j) {
                const uint4 v = mine[chunk(j)];
                c[4 * j] = v.x, c[4 * j + 1] = v.y, c[4 * j + 2] = v.z, c[4 * j + 3] = v.w;
            }
            typedef uint16_t Pair __attribute__((ext_vector_type(2)));
#pragma unroll
            for (int e = 0; e < E; ++e) {
                sum += c[e];
                full = __builtin_bit_cast(uint32_t, __builtin_elementwise_max(__builtin_bit_cast(Pair, full), __builtin_bit_cast(Pair, c[e])));
            }
            full = (full >> 16) > (full & 0xffffu) ? full >> 16 : full & 0xffffu;
            full = WaveMax(odd == odd ? full : 0xffffu); // (more than any has)
            const uint32_t upTo = WaveScan(sum);
            uint32_t all = (uint32_t)__builtin_amdgcn_readlane((int)upTo, 63), begin = upTo - sum;
            if constexpr (W > 1) {
                each[2 * W + waveOfRow] = all;
                across[kTopkWaves + wave] = full;
                __syncthreads();
                all = 0;
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const uint32_t n = each[2 * W + w];
                    begin += w < waveOfRow ? n : 0u;
                    all += n;
                }
#pragma unroll
                for (int w = 0; w < kTopkWaves; ++w)
                    full = across[kTopkWaves + w] > full ? across[kTopkWaves + w] : full;
                full = (uint32_t)__builtin_amdgcn_readfirstlane((int)full);
            }
            if (full == 0xffffu)
                return kNothingDone;
            begin += all << 16;
#pragma unroll
            for (int e = 0; e < E; ++e) {
                const uint32_t n = c[e];
                c[e] = begin;
                begin += n;
            }
#pragma unroll
            for (int j = 0; j < E / 4; ++j)
                mine[chunk(j)] = make_uint4(c[4 * j], c[4 * j + 1], c[4 * j + 2], c[4 * j + 3]);
        }
        // Many keys in a bucket: mostly few distinct scores, whose equal ones will stand in order by themselves, or too many to be exchanged.  D scores alike in
        // number bring some 2 N / D pairs of equal ones 64 and 128 columns apart, most of what the fullest bucket has keys; a part f of the row that is equal, with
        // other scores among it in the bucket, 2 f times that bucket's; distinct ones none.  (128, and a third: where keys and pairs are few and vary by chance)
        // By rank equal ones are in no order.
        bool equal = false;
        if (full > (uint32_t)(RANKS ? kMost : kSurely)) {
            if (RANKS)
                return kNothingDone;
            const int same = Equal(bits, i0, validCols, across + 2 * kTopkWaves) / (W > 1 ? kTopkWaves / W : 1);
            equal = 3 * same >= (int)full && 3 * same + 128 >= 4 * (int)full;
            if (!equal && full > (uint32_t)kMost)
                return kNothingDone;
        }
        Meet();
        // every key to the next place of its bucket.  (Equal scores in many columns: wave after wave, so that they are not in disorder)
        const int turns = W > 1 && equal ? W : 1;
        for (int turn = 0; turn < turns; ++turn) {
            if (turns == 1 || turn == waveOfRow) {
#pragma unroll
                for (int e = 0; e < E; ++e)
                    at[e] = __hip_atomic_fetch_add(count + at[e], one[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
            }
            if (turns > 1)
                __syncthreads();
        }
        const uint32_t columnBits = (4095u - i0) << 8;
#pragma unroll
        for (int e = 0; e < E; ++e) {
            at[e] = __builtin_amdgcn_ubfe(at[e], one[e] >> 12, 16);
            k[e] = TopkKey(bits[e], RANKS ? (4095u - rankOf[i0 + 64u * (uint32_t)e]) << 8 : columnBits - (uint32_t)(e * 64 << 8));
        }
        if (validCols != N) { // (what stands behind the columns goes behind the keys)
#pragma unroll
            for (int e = 0; e < E; ++e)
                if (!isColumn(e)) {
                    at[e] = i0 + 64u * (uint32_t)e;
                    k[e] = 1.0;
                }
        }
        Meet(); // (the counters are no longer needed)
        uint64_t *const list = reinterpret_cast<uint64_t *>(mem);
#pragma unroll
        for (int e = 0; e < E; ++e)
            list[Place(at[e])] = __builtin_bit_cast(uint64_t, k[e]);
        Meet();
#pragma unroll
        for (int e = 0; e < E; ++e)
            k[e] = __builtin_bit_cast(double, list[Place(q * E + (uint32_t)e)]);
        Meet();
        // As many passes as the fullest bucket can need; with equal scores, which can need none, a look before each whether all is in order (bfloat16 scores: equal ones in
        // the fullest buckets, a few distinct ones in others)
        const bool enough = full <= (uint32_t)kMost;
        const int passes = enough ? (int)(full + 1u) / 2 : kTries;
        for (int pass = 0;; ++pass) { // (two places for the edges in turn, and two others for the look)
            if (pass == passes && enough)
                return kSorted;
            if (__builtin_expect(equal, 0)) {
                double above, below;
                Neighbours(above, below, waveOfRow, lane, list + (pass & 1) * 16 + 8);
                bool sorted = k[E - 1] >= above;
#pragma unroll
                for (int e = 1; e < E; ++e)
                    sorted = sorted & (k[e - 1] >= k[e]);
                if (W > 1 ? Everyone(sorted, across + (2 + (pass & 1)) * kTopkWaves) : WholeWave(sorted))
                    return kSorted;
                if (pass == passes)
                    return kLost;
            }
#pragma unroll
            for (int e = 0; e < E; e += 2)
                Exchange(k[e], k[e + 1]);
            double above, below;
            Neighbours(above, below, waveOfRow, lane, list + (pass & 1) * 16);
#pragma unroll
            for (int e = 1; e + 1 < E; e += 2)
                Exchange(k[e], k[e + 1]);
            k[E - 1] = Max(k[E - 1], above);
            k[0] = Min(k[0], below);
        }
    }
};
// waves on a SIMD at the least: of what few registers more or less decide (1600 x 2048 with five instead of seven 11.8 -> 12.9 us)
constexpr int Resident(int e, int w, Mode mode) { return mode == kSelect ? (e == 16 ? 4 : 1) : mode == kCut ? 1 : e == 16 && w <= 2 ? 4 : e == 8 && w >= 2 ? 7 : 1; }
template <int E, int W, bool LOW_DPP, Mode MODE>
__global__ __launch_bounds__(kTopkThreads, Resident(E, W, MODE)) void TopkRows(float *outScore, uint32_t *outIndex, const float *src, const uint32_t *inIdx,
                                                         int rows, int validCols, int ld, int topk, int keepBits, int through, int buckets)
{
    constexpr int N = 64 * E * W, kRows = kTopkWaves / W, kBits = RowSort<E, W, LOW_DPP>::kLaneBits;
    constexpr int kStaged = 64 * E + 4 * E; // words of a wave's results, one of padding behind every 16
    constexpr int kStages = E <= 8 ? 2 : 1;  // scores and columns side by side, or one after the other (LDS for four workgroups more)
    // exchanges, then results (or, between two sorts, the ranks of the columns); behind them the columns in the order of their indices
    // buckets: per row of one wave a piece of its own, in which its results are staged as well
    constexpr bool kCount = (MODE == kWhole || MODE == kCountedCut) && kBuckets<E, W>;
    constexpr size_t kOwn = kCount && W == 1 && N * 8 > kStaged * 4 * kStages ? N * 8 : kStaged * 4 * kStages;
    constexpr size_t kExchange = W > 1 ? (size_t)kTopkWaves * E * 64 * 8 : 0, kStage = (size_t)kTopkWaves * kOwn;
    constexpr size_t kSelected = MODE == kSelect ? 384 + (size_t)kRows * 68 * kMostSelected * 8 : 0, kSort = kExchange > kStage ? kExchange : kStage;
    constexpr size_t kWork = kSort > kSelected ? kSort : kSelected;
    static_assert(kWork >= (size_t)N * 2, "the ranks fit");
    // (one wave per row and buckets: both tables of the columns' order behind everything, as the rows are still counted when they are read; 16 keys a lane: 36 KiB a
    // workgroup, four to a compute unit, as their registers allow)
    constexpr bool kApart = kCount && W == 1;
    constexpr size_t kColumns = kApart ? kWork + (size_t)N * 2 : kWork;
    __shared__ __attribute__((aligned(16))) char lds[kColumns + (size_t)N * 2];
    [[maybe_unused]] __shared__ uint32_t across[kTopkWaves * 6];
    uint16_t *rankOf = reinterpret_cast<uint16_t *>(lds + (kApart ? kWork : 0)), *columnOf = reinterpret_cast<uint16_t *>(lds + kColumns);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const int waveOfRow = wave % W, row0 = (int)blockIdx.x * kRows, row = row0 + wave / W < rows ? row0 + wave / W : rows - 1;
    // this lane's first column; then every kStep-th.  Where a threshold selects, the waves of a row take blocks of 64 columns in turn, so that each
    // sees the whole row: the lowest of their thresholds counts, and with adjoining columns to a wave the poorest one set it wherever the
    // level of the scores changes along the row (600 x 2048, top 100, ascending 15.6 us, more than the 10.5 without a threshold)
    constexpr uint32_t kStep = MODE == kSelect ? 64 * W : 64;
    uint32_t i0 = (uint32_t)(waveOfRow * (MODE == kSelect ? 1 : E) * 64 + lane);

    // A lane past the last column looks at the last one: loads without branches are all in flight at once (16 of them one
    // behind the other were half of the kernel's time).  Up to four keys and few waves: always so, the branch around
    // it takes longer (1 x 200, top 16: 3.29 / 3.18 us; with many waves 8192 x 256, top 8: 6.4 / 6.7)
    constexpr bool kClamp = E <= 4 && LOW_DPP;
    auto load = [&](const uint32_t *from, uint32_t (&to)[E]) __attribute__((always_inline)) {
        if (!kClamp && validCols == N) {
#pragma unroll
            for (int e = 0; e < E; ++e)
                to[e] = from[i0 + e * kStep];
        } else {
#pragma unroll
            for (int e = 0; e < E; ++e)
                to[e] = from[i0 + e * kStep < (uint32_t)validCols ? i0 + e * kStep : (uint32_t)validCols - 1u];
        }
    };
    uint32_t bits[E];
    const uint32_t *scores = reinterpret_cast<const uint32_t *>(src) + (size_t)row * (size_t)ld;
    load(scores, bits);

    // are the indices first, first + 1, ... or at least increasing with the column?  (then the column decides among equal
    // scores, as the index would; the same answer in every wave of the workgroup.)  Where a threshold selects, the four waves look at
    // a quarter each
    constexpr bool kQuarters = (MODE == kSelect || kCount) && W < 4;
    constexpr int kIds = kQuarters ? E * W / 4 : E;
    constexpr uint32_t kIdStep = kQuarters ? 64 : kStep;
    uint32_t ids[kIds];
    const uint32_t id0 = kQuarters ? (uint32_t)(wave * kIds * 64 + lane) : i0;
    if constexpr (kQuarters) {
#pragma unroll
        for (int e = 0; e < kIds; ++e)
            ids[e] = inIdx[id0 + e * kIdStep < (uint32_t)validCols ? id0 + e * kIdStep : (uint32_t)validCols - 1u];
    } else {
        load(inIdx, ids);
    }
    const uint32_t first = inIdx[0];
    uint32_t wrong = 0;
#pragma unroll
    for (int e = 0; e < kIds; ++e) {
        const uint32_t at = id0 + e * kIdStep < (uint32_t)validCols ? id0 + e * kIdStep : (uint32_t)validCols - 1u;
        wrong |= (ids[e] - first) ^ at;
    }
    auto everyone = [&](bool v, int vote) { return W > 1 || kQuarters ? Everyone(v, across + vote * kTopkWaves) : WholeWave(v); };
    const bool consecutive = everyone(wrong == 0 && first <= 0xffffffffu - (uint32_t)validCols, 4);
    bool increasing = consecutive;
    if (__builtin_expect(!consecutive, 0)) {
        bool ok = true;
        for (int e = 0; e < E; ++e) {
            const int i = (int)(i0 + e * kStep);
            if (i + 1 < validCols)
                ok = ok && inIdx[i] < inIdx[i + 1];
        }
        increasing = everyone(ok, 5);
    }
    RowSort<E, W, LOW_DPP> s;
    s.q = (uint32_t)waveOfRow * 64u + LaneRank((uint32_t)lane);
    s.xchg = reinterpret_cast<uint64_t *>(lds);
    // the ranks of a wave go in order through its piece of LDS, so that its stores cover consecutive addresses
    uint32_t *staged = reinterpret_cast<uint32_t *>(lds + wave * kOwn), *stagedColumn = staged + (kStages - 1) * kStaged;
    const int firstRank = waveOfRow * 64 * E, count = topk - firstRank;
    auto ordered = [] { __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront"); __builtin_amdgcn_wave_barrier(); };
    // lane by lane consecutive words, all read before the first is stored; through: past the L2 (launch_topk)
    constexpr bool kThrough = MODE != kCut || N > 512; // (below, topk is 64 at most: 1000 x 300, top 30 5.2 us with the branch, 5.1 without)
    constexpr int kStored = MODE == kWhole ? E : E * W > 8 ? E * W / 8 : 1; // times 64: of a row that is not sorted whole, an eighth and less
    constexpr auto stored = std::integral_constant<int, kStored>();
    auto store = [&](auto keys, uint32_t *to, int n, int lane, auto &&word) __attribute__((always_inline)) {
        uint32_t w[decltype(keys)::value];
#pragma unroll
        for (int e = 0; e < decltype(keys)::value; ++e)
            w[e] = word(e * 64 + lane);
        if (kThrough && through) {
#pragma unroll
            for (int e = 0; e < decltype(keys)::value; ++e)
                if (e * 64 + lane < n)
                    __hip_atomic_store(to + e * 64 + lane, w[e], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        } else {
#pragma unroll
            for (int e = 0; e < decltype(keys)::value; ++e)
                if (e * 64 + lane < n)
                    to[e * 64 + lane] = w[e];
        }
    };
    if constexpr (MODE == kSelect) {
        if (increasing) {
            constexpr int kList = 68 * kMostSelected; // (twice as many words: a list, or its results with their padding)
            uint32_t *const perWave = reinterpret_cast<uint32_t *>(lds); // T, 16 words on how many a wave has, and E W per row on each block of 64 columns
            static_assert(W > 1 || kList * 2 == kStaged * kStages, "a wave that sorts the whole row stays in its list's memory");
            uint32_t *const list = W == 1 ? staged : perWave + 96 + wave / W * (kList * 2);
            uint32_t order[E], most[4]; // (padding: 0)
#pragma unroll
            for (int e = 0; e < E; ++e) {
                order[e] = ScoreOrder(bits[e]);
                if ((kClamp || validCols != N) && i0 + e * kStep >= (uint32_t)validCols)
                    order[e] = 0;
                most[e % 4] = e < 4 || order[e] > most[e % 4] ? order[e] : most[e % 4];
            }
            // T of this wave: `wanted` of its groups' maxima, and few more, are T or larger; a group: the keys of a lane, or every second or
            // fourth of them
            const int wanted = (topk + W - 1) / W; // (the waves' numbers of columns differ by 64 at most)
            constexpr int kMost = E < 4 ? E : 4;
            uint32_t most2[2] = {most[0], kMost > 1 ? most[1] : 0u};
            if constexpr (kMost == 4) {
                most2[0] = most[0] > most[2] ? most[0] : most[2];
                most2[1] = most[1] > most[3] ? most[1] : most[3];
            }
            const uint32_t most1[1] = {most2[0] > most2[1] ? most2[0] : most2[1]};
            uint32_t above = WaveMax(most1[0]);
            above += above != 0xffffffffu ? 1u : 0u;
            // (all groups reach the smallest of the maxima; 64 lanes the smallest of the lanes')
            uint32_t least = most1[0];
            if (kMost == 4 && wanted > 64) {
                const uint32_t low0 = most[0] < most[2] ? most[0] : most[2], low1 = most[1] < most[3] ? most[1] : most[3];
                least = low0 < low1 ? low0 : low1;
            }
            uint32_t t = ~WaveMax(~least);
            // (groups more than wanted: as many as leave random rows' lists below 256 or 512, which are sorted in the same time; 64 x 4096, top 320 9.3 us, 15.4 where one
            // row is past 512; 600 x 2048, top 160 8.2 and 9.1 past 256)
            const int close = W == 4 && wanted > 64 ? wanted / 32 : wanted / 8;
            const int loose = wanted <= 64 ? (wanted / 2 + 4 < 16 ? wanted / 2 + 4 : 16) : W == 1 ? 32 : W == 2 && wanted <= 96 ? (wanted <= 80 ? 12 : 32) : close;
            // (the first look is right above the smallest: the end already where most are equal.  Few distinct scores may have no place for a tight
            // threshold: from the eighth look on as many groups more will do as no longer a sort pays for; 4800 x 1024, top 40 of 60 distinct 10.2 -> 8.4 us)
            auto search = [&](auto groups, const uint32_t *max) __attribute__((always_inline)) {
                int limit = wanted + close, looks = 0;
                for (uint32_t mid = t + 1u; above - t > 1u; mid = t + (above - t) / 2u) {
                    int n = 0;
#pragma unroll
                    for (int g = 0; g < decltype(groups)::value; ++g)
                        n += __builtin_popcountll(__builtin_amdgcn_ballot_w64(max[g] >= mid));
                    if (++looks == 8)
                        limit = wanted + loose;
                    if (n < wanted) {
                        above = mid;
                    } else {
                        t = mid;
                        if (n <= limit)
                            break;
                    }
                }
            };
            if (wanted <= 24)
                search(std::integral_constant<int, 1>(), most1);
            else if (wanted <= 48 || kMost < 4)
                search(std::integral_constant<int, 2>(), most2);
            else
                search(std::integral_constant<int, kMost>(), most);
            if constexpr (W > 1) {
                if (lane == 0)
                    perWave[wave] = t;
                __syncthreads();
#pragma unroll
                for (int w = 0; w < W; ++w) {
                    const uint32_t other = (uint32_t)__builtin_amdgcn_readfirstlane((int)perWave[wave / W * W + w]);
                    t = other < t ? other : t;
                }
            }
            // larger than T, and as large (-0 compares equal to +0)
            t = (uint32_t)__builtin_amdgcn_readfirstlane((int)t);
            const bool zero = t == kSign || t == kSign - 1u;
            uint32_t tLow = zero ? kSign - 1u : t, tHigh = zero ? kSign : t;
            // Who reaches T, and where in the list; where that are many more than are wanted, for instance as many equal ones (masked rows), once more with
            // as many of those that equal T, by their columns, as are wanted behind the larger ones.  (Many: more than random scores bring, and than the
            // shortest sort takes.  Each block of 64 columns ranked by ballots of its own took 2 us more.)
            int total;
            uint32_t at;
            bool fits;
            for (bool again = false;; again = true) {
                uint32_t mine = 0;
#pragma unroll
                for (int e = 0; e < E; ++e)
                    mine += order[e] >= tLow ? 1u : 0u;
                at = WaveScan(mine); // up to this lane
                total = __builtin_amdgcn_readlane((int)at, 63);
                at -= mine;
                if constexpr (W > 1) {
                    if (lane == 0)
                        perWave[16 + wave] = (uint32_t)total;
                    __syncthreads();
                    total = 0;
#pragma unroll
                    for (int w = 0; w < W; ++w) {
                        const int n = __builtin_amdgcn_readfirstlane((int)perWave[16 + wave / W * W + w]);
                        at += w < waveOfRow ? (uint32_t)n : 0u;
                        total += n;
                    }
                }
                fits = total <= 64 * kMostSelected && tLow != 0u;
                if (!again)
                    fits = fits && total <= 2 * topk + 64;
                if constexpr (W > 1)
                    fits = __syncthreads_and(fits) != 0; // (the other ways have barriers of the whole workgroup)
                // (who reaches T is compared again below: E answers take two scalar registers each, more than there are)
                asm("" : "+s"(tLow), "+s"(tHigh));
                if (again || __builtin_expect(fits, 1))
                    break;
                uint32_t equal = 0; // in the lane's block of 64 columns, of this wave's E, then of the row's E W
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const uint64_t same = __builtin_amdgcn_ballot_w64(order[e] - tLow <= tHigh - tLow);
                    equal = lane == e ? (uint32_t)__builtin_popcountll(same) : equal;
                }
                if constexpr (W > 1) {
                    uint32_t *const blocks = perWave + 32 + wave / W * (E * W);
                    if (lane < E)
                        blocks[lane * W + waveOfRow] = equal;
                    __syncthreads();
                    equal = lane < E * W ? blocks[lane] : 0u;
                }
                const uint32_t upTo = WaveScan(equal);
                // (as many there are: topk keys and more reach T)
                const int taken = tLow == 0u ? 0 : topk - (total - __builtin_amdgcn_readlane((int)upTo, 63));
                uint32_t last = 0xffffffffu; // the column of the last one
                if (taken > 0) {
                    const int block = __builtin_ctzll(__builtin_amdgcn_ballot_w64((int)upTo >= taken));
                    const int nth = taken - __builtin_amdgcn_readlane((int)(upTo - equal), block);
                    const uint32_t column = (uint32_t)(block * 64 + lane), one = ScoreOrder(scores[column < (uint32_t)validCols ? column : 0u]);
                    const uint64_t same = __builtin_amdgcn_ballot_w64(column < (uint32_t)validCols && one - tLow <= tHigh - tLow);
                    const int rank = (int)__builtin_amdgcn_mbcnt_hi((uint32_t)(same >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)same, 0u));
                    last = (uint32_t)(block * 64 + __builtin_ctzll(__builtin_amdgcn_ballot_w64(rank == nth - 1) & same));
                }
#pragma unroll
                for (int e = 0; e < E; ++e)
                    order[e] = order[e] - tLow <= tHigh - tLow && (int)(i0 + e * kStep) > (int)last ? 0u : order[e];
            }
            if (__builtin_expect(fits, 1)) {
#pragma unroll
                for (int e = 0; e < E; ++e)
                    if (order[e] >= tLow)
                        reinterpret_cast<uint64_t *>(list)[at++] = (uint64_t)(i0 + e * kStep) << 32 | order[e];
                if constexpr (W > 1)
                    __syncthreads();
                else
                    ordered();
                if (waveOfRow != 0 || row0 + wave / W >= rows)
                    return;
                uint32_t *toScore = reinterpret_cast<uint32_t *>(outScore) + (size_t)row * (size_t)topk, *toIndex = outIndex + (size_t)row * (size_t)topk;
                auto finish = [&](auto keys) __attribute__((always_inline)) {
                    constexpr int S = decltype(keys)::value;
                    RowSort<S, 1, LOW_DPP> few;
                    few.q = LaneRank((uint32_t)lane);
                    few.xchg = nullptr;
                    few.form = 0;
#pragma unroll
                    for (int e = 0; e < S; ++e) {
                        const uint64_t one = reinterpret_cast<const uint64_t *>(list)[e * 64 + lane];
                        const uint32_t c = 4095u - (uint32_t)(one >> 32), negZero = (uint32_t)one == kSign - 1u ? 1u : 0u, o = (uint32_t)one + negZero;
                        few.k[e] = e * 64 + lane < total ? Key(__builtin_amdgcn_alignbit(0x3ffu, o, 12), (o << 20) | (c << 8) | negZero) : 1.0;
                    }
                    few.template Sort<6>(6);
                    ordered();
                    uint32_t *score = list, *at = list + 68 * S;
                    const int rank0 = (int)LaneRank((uint32_t)lane) * S;
#pragma unroll
                    for (int e = 0; e < S; ++e) {
                        const uint32_t low = Low(few.k[e]), i = (uint32_t)(rank0 + e) + (uint32_t)(rank0 + e) / 16u;
                        score[i] = (low & 1u) ? kSign : ScoreBits((High(few.k[e]) << 12) | (low >> 20));
                        at[i] = 4095u - ((low >> 8) & 0xfffu);
                    }
                    ordered();
                    store(keys, toScore, topk, lane, [&](int i) { return score[i + i / 16]; });
                    if (consecutive)
                        store(keys, toIndex, topk, lane, [&](int i) { return first + at[i + i / 16]; });
                    else
                        store(keys, toIndex, topk, lane, [&](int i) { return inIdx[i < topk ? at[i + i / 16] : 0u]; }); // (behind topk may stand a column that is none)
                };
                if (total <= 64)
                    finish(std::integral_constant<int, 1>());
                else if (total <= 128)
                    finish(std::integral_constant<int, 2>());
                else if (total <= 256)
                    finish(std::integral_constant<int, 4>());
                else
                    finish(std::integral_constant<int, kMostSelected>());
                return;
            }
            asm volatile("" : "+v"(i0)); // (nothing that depends on it is kept so far either)
            load(scores, bits);
        }
    }
    // staging and stores of the sorted keys; rank: of the lane's first one
    auto finish = [&](const double (&k)[E], int rank, int lane) __attribute__((always_inline)) {
        if (W > 1)
            __syncthreads(); // (the exchanges are over)
        if (row0 + wave / W >= rows || count <= 0)
            return;
        uint32_t *toScore = reinterpret_cast<uint32_t *>(outScore) + (size_t)row * (size_t)topk + firstRank;
        uint32_t *toIndex = outIndex + (size_t)row * (size_t)topk + firstRank;
        uint32_t column[E];
#pragma unroll
        for (int e = 0; e < E; ++e) {
            const uint32_t low = Low(k[e]), order = (High(k[e]) << 12) | (low >> 20);
            column[e] = 4095u - ((low >> 8) & 0xfffu);
            staged[rank + e + (rank + e) / 16] = (low & 1u) ? kSign : ScoreBits(order);
            if (kStages == 2)
                stagedColumn[rank + e + (rank + e) / 16] = column[e];
        }
        ordered();
        store(stored, toScore, count, lane, [&](int i) { return staged[i + i / 16]; });
        if (kStages == 1) {
            ordered();
#pragma unroll
            for (int e = 0; e < E; ++e)
                stagedColumn[rank + e + (rank + e) / 16] = column[e];
            ordered();
        }
        if (__builtin_expect(!consecutive, 0)) { // (staged: the column, or its rank)
#pragma unroll
            for (int e = 0; e < kStored; ++e) {
                const int i = e * 64 + lane;
                if (i < count) {
                    const uint32_t c = stagedColumn[i + i / 16];
                    toIndex[i] = inIdx[increasing ? c : columnOf[c]];
                }
            }
            return;
        }
        store(stored, toIndex, count, lane, [&](int i) { return first + stagedColumn[i + i / 16]; });
    };
    if constexpr (kCount) {
        if (increasing && buckets) {
            uint32_t column0 = i0;
            int here = lane;
            asm volatile("" : "+v"(column0), "+v"(here)); // (nothing of this is kept in registers for what comes behind)
            BucketSort<E, W> b;
            const Counted done = b.Sort(bits, column0, validCols, waveOfRow, here, reinterpret_cast<uint32_t *>(lds + (W == 1 ? wave * kOwn : (size_t)(wave / W) * N * 8)), across);
            if (__builtin_expect(done == kSorted, 1)) {
                finish(b.k, here * E, here);
                return;
            }
            if (done == kLost)
                load(scores, bits);
        }
    }
    const uint32_t columnBits = (4095u - i0) << 8;
    if (__builtin_expect(!increasing, 0)) { // the columns in the order of their indices; rows of one wave: the first wave does it for all four
        if (W > 1 || wave == 0) {
            s.form = 0;
            uint32_t all[E];
            load(inIdx, all);
            bool listed = false;
            if constexpr (kCount && N < 4096) { // (4096 columns: scalar registers would be spilled)
                // indices below 2^24 by buckets: as scores, exactly (2400 x 2048, top 2000 54.3 -> 43.7 us, 1000 x 1024, top 700 16.2 -> 13.9; 4800 x 1024
                // whole 39.9 -> 35.0, and 30.0 with its scores by buckets as well; indices that this turns away 15.7 -> 15.8)
                constexpr uint32_t kBelow = 1u << 24;
                bool small = true;
#pragma unroll
                for (int e = 0; e < E; ++e)
                    small = small & (all[e] < kBelow);
                if (W > 1 ? Everyone(small, across + 4 * kTopkWaves) : WholeWave(small)) {
                    uint32_t as[E];
#pragma unroll
                    for (int e = 0; e < E; ++e)
                        as[e] = __builtin_bit_cast(uint32_t, (float)(kBelow - 1u - all[e]));
                    uint32_t column0 = i0;
                    int here = lane;
                    asm volatile("" : "+v"(column0), "+v"(here));
                    BucketSort<E, W> b;
                    listed = b.Sort(as, column0, validCols, waveOfRow, here, reinterpret_cast<uint32_t *>(lds + (W == 1 ? 0 : (size_t)(wave / W) * N * 8)), across) == kSorted;
                    if (listed) {
                        if (W > 1)
                            __syncthreads(); // (neighbours have read each other's keys)
#pragma unroll
                        for (int e = 0; e < E; ++e) {
                            const uint32_t rank = (uint32_t)((waveOfRow * 64 + here) * E + e), column = 4095u - ((Low(b.k[e]) >> 8) & 0xfffu);
                            if (wave < W && rank < (uint32_t)validCols) {
                                rankOf[column] = (uint16_t)rank;
                                columnOf[rank] = (uint16_t)column;
                            }
                        }
                    } else {
                        load(inIdx, all);
                    }
                }
            }
            if (!listed) {
#pragma unroll
                for (int e = 0; e < E; ++e) {
                    const uint32_t order = ~all[e];
                    s.k[e] = Key(__builtin_amdgcn_alignbit(0x3ffu, order, 12), (order << 20) | (columnBits - (e * kStep << 8)));
                    if (i0 + e * kStep >= (uint32_t)validCols)
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
        }
        load(scores, bits);
        if constexpr (kApart) {
            __syncthreads(); // the ranks are there
            uint32_t column0 = i0;
            int here = lane;
            asm volatile("" : "+v"(column0), "+v"(here));
            BucketSort<E, W> b; // (9000 x 512, top 400 29.4 -> 22.7 us with this and the columns' order by buckets; 3000 x 777, top 700 25.6 -> 18.1)
            const Counted done = b.template Sort<true>(bits, column0, validCols, 0, here, reinterpret_cast<uint32_t *>(lds + wave * kOwn), across, rankOf);
            if (done == kSorted) {
                finish(b.k, here * E, here);
                return;
            }
            if (done == kLost)
                load(scores, bits);
        }
    }
    s.form = 0;
#pragma unroll
    for (int e = 0; e < E; ++e)
        s.k[e] = TopkKey(bits[e], columnBits - (e * kStep << 8));
    if (__builtin_expect(!increasing, 0)) {
        if (!kApart)
            __syncthreads(); // the ranks are there
#pragma unroll
        for (int e = 0; e < E; ++e)
            s.k[e] = Key(High(s.k[e]), (Low(s.k[e]) & 0xfff000ffu) | (4095u - rankOf[i0 + e * kStep]) << 8); // (past the row's end: overwritten below)
        if (!kApart)
            __syncthreads(); // and read, before their memory is used for something else
    }
    if (kClamp || validCols != N) {
#pragma unroll
        for (int e = 0; e < E; ++e)
            if (i0 + e * kStep >= (uint32_t)validCols)
                s.k[e] = 1.0;
    }
    s.template Sort<MODE == kWhole ? kBits : kBits - kWholeBits - 1>(keepBits);
    finish(s.k, (int)LaneRank((uint32_t)lane) * E, lane);
}

template <int E, int W>
int launch_topk(hipStream_t st, float *out_score, uint32_t *out_index, const float *src, const uint32_t *in_idx, int rows, int valid_cols, int ld,
                int topk, [[maybe_unused]] bool select = false)
{
    int keepBits = 0;
    while ((E << keepBits) < topk)
        ++keepBits;
    const bool whole = kOnlyWhole<E, W> || keepBits + kWholeBits >= RowSort<E, W, true>::kLaneBits;
    // Lower words between near lanes: with up to four waves on a SIMD the latency of the LDS pipe shows, a DPP move is shorter
    // (LDS / DPP, whole sorts: 300 x 128 3.48 / 3.26 us, 300 x 256 4.53 / 4.28); with more the moves take issue slots (4800 x 128
    // 5.09 / 5.23).  8 and 16 keys per lane cover the latency either way and take DPP.
    const bool dpp = E >= 8 || (long long)rows * W <= 4 * 4 * pto_amd::compute_units();
    // Past 1024 columns buckets instead of merges that keep topk, wherever no threshold is taken (us, merges / buckets, random scores; nearly all equal ones):
    // 2048 columns, 16 rows, top 129 7.0 / 5.5; 7.0 / 7.35, 300 rows, top 256 8.5 / 6.2; 8.4 / 8.8; 4096 columns, 16 rows, top 321 11.4 / 7.5; 11.45 / 11.9,
    // 1500 rows, top 512 34.3 / 19.5; 33.7 / 34.9.  1024 columns, 16 rows, top 64 4.6 / 4.4; 4.6 / 5.0: what it gives and what it takes are alike there
    // (16 keys a lane with up to two waves, eight with two: the dispatch has taken a threshold for every such topk, and no other kernel is built)
    constexpr bool kThresholdBefore = (E == 16 && W <= 2) || (E == 8 && W == 2);
    constexpr Mode kFew = kOnlyWhole<E, W> || kThresholdBefore ? kWhole : W == 4 && E >= 8 ? kCountedCut : kCut;
    constexpr bool kDpp = E >= 8 || kOnlyWhole<E, W>; // (names the one form that there is)
    auto kernel = dpp ? (whole ? TopkRows<E, W, true, kWhole> : TopkRows<E, W, true, kFew>) :
                        (whole ? TopkRows<E, W, kDpp, kWhole> : TopkRows<E, W, kDpp, kFew>);
    if constexpr (E == 16 || (E == 8 && W == 1))
        if (select)
            kernel = TopkRows<E, W, true, kSelect>;
    // Results past the L2: a kernel ends with every L2 writing back what is dirty in it, 3 us for the 38 MB of 4800 x 1000 (25.4 ->
    // 23.3 us; 8192 x 500, top 333 19.2 -> 17.0; 300 x 128 whole 2.69 -> 2.67).  Not where a row's results are less than a store
    // instruction's 256 bytes (8192 x 64, top 1 3.2 / 3.7, 131072 x 64, top 33 32.6 / 34.1), nor where they are much more than the L2s'
    // 32 MB, which then are written back while others sort (30000 x 2048, top 1500 261 / 268).
    const int through = topk >= 64 && 8ll * rows * topk <= 1ll << 26;
    // Just past what a threshold is taken for, 257 to 320 of 1025 to 2048 columns, the network: by buckets random rows would be faster than the top 256 of them are by threshold, and few of
    // many are not to take longer than more (past 2048 columns they do, by a fifth: 64 x 4096, top 320 9.0, top 321 7.5).  What it costs (us, random; masked from the middle on):
    // 600 x 1025, top 256 by threshold 8.8; 8.4, top 257 by the network 11.6; 11.5, by buckets 7.4; 11.9; 1600 x 2048 11.3; 11.0, 19.4; 19.3, 10.9; 20.3.  Buckets for the top 256 too
    // would slow masked rows by 40 to 85 % (below, at the threshold); both in one kernel, buckets ahead of the threshold, is 15 % faster with random rows, 5 to 20 % slower with
    // masked and 50 % with sixty distinct scores
    const int buckets = !(64 * E * W == 2048 && topk > 256 && topk <= 320);
    constexpr int kRows = kTopkWaves / W;
    kernel<<<dim3((unsigned)(((long long)rows + kRows - 1) / kRows)), dim3(kTopkThreads), 0, st>>>(out_score, out_index, src, in_idx, rows, valid_cols,
                                                                                                   ld, topk, keepBits, through, buckets);
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
    // Waves per row.  One wave per row does the least work, more put more of the chip to work on few rows.  1024 columns, one / two / four waves,
    // whole sorts, us, on 256 units (by buckets; the network): 300 rows 6.7 / 5.8 / 5.1; 600 rows 6.6 / 6.4 / 5.6; 9.8 / 8.8 / 7.7, 1000 rows 6.6 / 6.4 / 6.1;
    // 10.3 / 9.3 / 9.2, 1500 rows 8.2 / 7.5 / 7.2, 2400 rows 9.7 / 9.2 / 10.2; 17.5 / 16.2 / 17.9, 4800 rows 25.3 / 26.9 / 28.8 (network): four up to 853 rows, two
    // up to 2560 (1000 rows top 256 by the network 8.7 / 8.1 / 8.2).  512 columns: four waves and the network up to 731 rows (network: 600 rows 5.7 / 5.4 / 5.1,
    // 853 rows 5.8 / 5.5 / 5.6, top 15 4.5 / 4.6 / 5.1; 300 rows network in four 4.1, buckets in one or two 4.5; 700 rows 4.6, 4.5 and 4.9), then one.
    // 2048 columns: four up to 1706 rows (two / four, by buckets: 16 rows 7.9 / 5.6, 800 rows 9.8 / 8.6, 1600 rows 13.4 / 11.5, 2400 rows 17.2 / 17.2; network: 1700
    // rows 25.6 / 24.5, 2000 rows 26.2 / 26.9).  129 to 256 columns: four up to 365 rows where
    // more than 16 are wanted (one / four: 128 rows 3.6 / 3.3, 300 rows 3.6 / 3.4, 600 rows 3.7 / 3.7; top 7 of 128 rows 3.2 / 3.6).
    const int most = 5 * 4 * pto_amd::compute_units() / rows; // waves per row for five on every SIMD
    // A threshold, then a sort of what reaches it (us, merges that keep topk / threshold; random scores):
    //   4096 columns:    1 row,  top   1 7.9 / 5.5    128 rows, top 50 10.4 / 6.6   1200 rows, top 300 31.9 / 18.8
    //   2048 columns:    8 rows, top  10 6.1 / 5.4    900 rows, top 30 10.9 / 6.0   2400 rows, top 256 25.0 / 16.5; few rows and many keys: 64 rows, top 140 7.6 / 8.4
    //   1024 columns:  600 rows, top 128 7.2 / 6.5   1500 rows, top 16  7.6 / 5.4   4800 rows, top 128 19.9 / 9.9; 128 rows, top 16 4.8 / 4.9, top 128 5.4 / 6.6, 700 rows, top 4 5.1 / 5.3
    //    512 columns: 4000 rows, top  16 7.5 / 6.0   8000 rows, top 60 14.7 / 10.6; 1000 rows, top 16 4.7 / 4.7, top 60 5.2 / 5.5
    // One wave per row of 1024 and two per row of 2048 where without the threshold there are four (1500 rows, top 16: 5.2 with one, 6.1 with four).
    // Near the line no kind of row measured is slower by more than 3 % than by merges.  600 x 1024, top 100: random 7.2 / 6.6, sixty distinct scores 7.2 / 6.6, all
    // equal but 2 % 7.2 / 5.7; 8 x 2048, top 30, all equal but 2 %: 6.4 / 6.6.  Buckets (keeping topk) in its place would be faster near its upper end with random rows, and slower
    // with masked ones, which they turn away.  Threshold / buckets, us, random; masked from the middle on: 600 x 1024, top 60 5.2 / 5.2; 5.5 / 7.0, top 128 6.2 / 5.2; 6.0 / 7.2, 4800 x 1024,
    // top 128 9.8 / 11.9; 9.4 / 19.3; 600 x 2048, top 100 6.8 / 7.2; 7.1 / 10.5, top 160 7.7 / 7.3; 7.3 / 11.0, top 256 8.9 / 7.3; 8.6 / 11.1, 1600 x 2048, top 256 11.3 / 10.4; 11.0 / 19.6;
    // 16 x 4096, top 320 9.1 / 7.4; 8.9 / 12.4, 300 x 4096, top 256 8.4 / 9.2; 8.7 / 14.8, 1200 x 4096, top 312 18.2 / 17.2; 17.6 / 30.7 (at top 320 one random
    // row in some hundreds has more than 512 keys at its threshold and goes to the network: 22.9).  Just past 1024 and 2048 columns the waves' thresholds lie lower for the short rows (1600 x 2049, top 100: 37.3 / 20.3).
    const int padded = valid_cols <= 512 ? 512 : valid_cols <= 1024 ? 1024 : valid_cols <= 2048 ? 2048 : 4096;
    if (valid_cols > 256 && topk <= padded / 8 && topk <= (valid_cols > 2048 || most < 10 ? 320 : most < 20 ? 160 : 128)) {
#define PTO_TOPK_SELECT(E, W) return launch_topk<E, W>(st, out_score, out_index, src, in_idx, rows, valid_cols, ld, topk, true);
        if (valid_cols > 2048)
            PTO_TOPK_SELECT(16, 4)
        if (valid_cols > 1024)
            PTO_TOPK_SELECT(16, 2)
        if (valid_cols > 512 && most <= (topk > 16 ? 8 : 6))
            PTO_TOPK_SELECT(16, 1)
        if (valid_cols <= 512 && most <= 1)
            PTO_TOPK_SELECT(8, 1)
#undef PTO_TOPK_SELECT
    }
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
