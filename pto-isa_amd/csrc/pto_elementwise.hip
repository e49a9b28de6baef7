// TCVT and gather kernels for MI355X, pure streaming work (bound by HBM bandwidth).  The conversion of buffers that are not aligned to
// its accesses and the one-tile index gather are written with PTO tile instructions, a workgroup moving one Vec tile
//   TLOAD (16-byte coalesced loads into registers) -> TCVT / TGATHER -> TSTORE (16-byte stores);
// aligned conversions and the row gather are streams below them.
// Test kernels of the same shape in the reference: tests/cpu/st/testcase/tcvt/tcvt_kernel.cpp:18-52,
// tests/cpu/st/testcase/tgather/tgather_kernel.cpp, tests/cpu/st/testcase/mgather/.
// The outputs of these kernels are written once and not read again by them: non-temporal stores keep them from pushing
// the data still to be read out of the caches (measured in tiles: conversion +2.6 %; non-temporal loads of its input +1.3 % alone,
// nothing on top of the stores.  The row gather, 65536 rows of 2 KiB out of 16384: 47.6 us with plain stores, 25.7 so).
#define PTO_VEC_STREAM_NT 2
#include <pto/pto-inst.hpp>

#include "common.hpp"

using namespace pto;

PTO_DEVICE_CODE_BEGIN

namespace {

constexpr int kCvtTile = 8192; // elements per workgroup: 4 chunks of 8 per lane

template <typename D, bool kTail>
__global__ __launch_bounds__(kBlockThreads) AICORE void CvtF32(__gm__ D *dst, __gm__ const float *src, size_t n,
                                                               size_t firstTile, int mode)
{
    const size_t tile = firstTile + get_block_idx();
    const size_t base = tile * (size_t)kCvtTile;
    using Shape1 = Shape<1, 1, 1, 1, DYNAMIC>;
    using Stride1 = Stride<1, 1, 1, DYNAMIC, 1>;
    using GSrc = GlobalTensor<float, Shape1, Stride1>;
    using GDst = GlobalTensor<D, Shape1, Stride1>;
    constexpr int VC = kTail ? DYNAMIC : kCvtTile;
    using TileSrc = Tile<TileType::Vec, float, 1, kCvtTile, BLayout::RowMajor, 1, VC>;
    using TileDst = Tile<TileType::Vec, D, 1, kCvtTile, BLayout::RowMajor, 1, VC>;
    const int valid = kTail ? (int)(n - base) : kCvtTile;
    auto mk = [&](auto tag) {
        using T = decltype(tag);
        if constexpr (kTail)
            return T((size_t)valid);
        else
            return T();
    };
    TileSrc srcTile = mk(TileSrc());
    TileDst dstTile = mk(TileDst());
    GSrc srcGlobal(const_cast<float *>(src) + base, Shape1(valid), Stride1(valid));
    GDst dstGlobal(dst + base, Shape1(valid), Stride1(valid));
    TLOAD(srcTile, srcGlobal);
    set_flag(PIPE_MTE2, PIPE_V, EVENT_ID0);
    wait_flag(PIPE_MTE2, PIPE_V, EVENT_ID0);
    TCVT(dstTile, srcTile, static_cast<RoundMode>(mode));
    set_flag(PIPE_V, PIPE_MTE3, EVENT_ID0);
    wait_flag(PIPE_V, PIPE_MTE3, EVENT_ID0);
    TSTORE(dstGlobal, dstTile);
}

// Buffers aligned to its accesses take a streaming form of the same conversion below the tile instructions: a lane loads
// 16 bytes and stores 8, so that every load instruction of a wave covers 1 KiB of consecutive addresses and every store
// 512 bytes (a Vec tile gives a lane eight consecutive elements, i.e. two loads 32 bytes apart per lane and half-used
// lines per instruction), all loads of a lane are in flight before the first conversion, and there is no barrier; the
// stores go through the L2 to memory (system scope): plain stores leave 32 MB dirty there, which are written back behind the last one (2^27
// elements to fp16: plain 6.2 TB/s, non-temporal 124.1 us = 6.49, through 121.3 = 6.64; 33 M 31.1 and 29.3 us, 16.5 M to bf16 16.0 and
// 15.7, 2 M 2.70 and 2.18; geometric mean of 60 sizes 1.023).  What is not whole pieces stays non-temporal: a part of 64 bytes written through
// holds up the end of the kernel (700001 elements 2.7 and 3.0 us).  Same element function as TCVT (detail::convert), so the results are the same bits.  The last workgroup takes
// what is left behind the whole pieces, element by element past the last four: as a launch of its own that rest took
// 3.7 us (16 524 000 elements 20.0 -> 16.2 us, 6.1 TB/s; 2^27 - 5 elements 126.6 -> 123.9, 6.5 TB/s).  LOADS: 16-byte loads of a
// lane: four; two for the modes that round in integer arithmetic, where more waves hide more of it (2^26 elements downwards: tile
// form 77.4, eight loads 68.7, four 64.3, two 63.5 us), and for fp16 from 2^24 elements on (2^24, 2^25, 2^27 elements: two 17.1, 31.9,
// 123.1 us, four 17.8, 32.9, 126.4, eight 17.5, 33.0, 125.2; below, which is faster depends on where the buffers lie).
template <int LOADS>
constexpr int kCvtPiece = LOADS * 4 * kBlockThreads; // elements per workgroup
template <typename D, int MODE, int LOADS>
__global__ __launch_bounds__(kBlockThreads) void CvtF32Stream(D *dst, const float *src, size_t n, size_t firstPiece)
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    typedef uint16_t u16x4 __attribute__((ext_vector_type(4)));
    constexpr int kPerStep = kBlockThreads * 4, kSteps = LOADS, kPiece = kCvtPiece<LOADS>;
    static_assert(sizeof(D) == 2, "16-bit results");
    auto cvt = [](float v) { return __builtin_bit_cast(uint16_t, ::pto::detail::convert<D, float>(v, static_cast<RoundMode>(MODE))); };
    const size_t first = (firstPiece + blockIdx.x) * (size_t)kPiece, base = first + 4 * threadIdx.x;
    f32x4 x[kSteps];
    if (first + kPiece <= n) {
#pragma unroll
        for (int i = 0; i < kSteps; ++i)
            x[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(src + base + (size_t)i * kPerStep));
#pragma unroll
        for (int i = 0; i < kSteps; ++i) {
            u16x4 y;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                y[j] = cvt(x[i][j]);
            __hip_atomic_store(reinterpret_cast<uint64_t *>(dst + base + (size_t)i * kPerStep), __builtin_bit_cast(uint64_t, y), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
        const size_t at = base + (size_t)i * kPerStep;
        if (at + 4 <= n)
            x[i] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(src + at));
    }
#pragma unroll
    for (int i = 0; i < kSteps; ++i) {
        const size_t at = base + (size_t)i * kPerStep;
        if (at + 4 <= n) {
            u16x4 y;
#pragma unroll
            for (int j = 0; j < 4; ++j)
                y[j] = cvt(x[i][j]);
            __builtin_nontemporal_store(y, reinterpret_cast<u16x4 *>(dst + at));
        } else {
            for (size_t e = at; e < n; ++e) // at most three, of one lane
                dst[e] = __builtin_bit_cast(D, cvt(src[e]));
        }
    }
}

// Row gather as a stream of 16-byte chunks: out is n_idx rows of cpr chunks, chunk c comes from chunk c % cpr of table row
// idx[c / cpr] (zeros for an index outside the table).  Consecutive lanes take consecutive chunks, whatever the width of a
// row, so every store instruction of a wave is 1 KiB of consecutive addresses and every load whole lines of the table's
// rows; the indices, then all loads of a lane are in flight before its first store; no LDS, no barrier.  The division is
// a multiplication: for c < 2^31, c / cpr = c magic >> shift with magic = ceil(2^shift / cpr), shift = 31 + ceil(log2 cpr).
// Table and output need their elements' alignment only (the chunks are typed so; the same instructions).
// The row is cut into `parts` (1, 2, 4 or 8) slices of cpr chunks, and workgroup b works on slice (b % 8) % parts: as the
// workgroups are dealt to the eight XCDs in turn, an XCD's L2 then sees one slice of the table only.  SHORT: the last slice has
// fewer chunks, the lanes past its end idle (a kernel of its own: the test costs the others 2 to 3 %).
constexpr int kGatherSteps = 2, kGatherChunks = kBlockThreads * kGatherSteps;
template <bool SHORT>
__global__ __launch_bounds__(kBlockThreads) void GatherChunks(char *out, const char *table, const int32_t *idx, uint32_t chunks, uint32_t rowChunks,
                                                              uint32_t cpr, uint32_t magic, int shift, uint32_t tableRows, uint32_t parts)
{
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(2)));
    const uint32_t xcd = blockIdx.x % 8, slice = xcd % parts, block = blockIdx.x / 8 * (8 / parts) + xcd / parts;
    const uint32_t first = block * (uint32_t)kGatherChunks + threadIdx.x;
    if (block * (uint32_t)kGatherChunks >= chunks)
        return;
    uint32_t row[kGatherSteps], at[kGatherSteps], part[kGatherSteps];
#pragma unroll
    for (int i = 0; i < kGatherSteps; ++i) {
        const uint32_t c = first + i * kBlockThreads < chunks ? first + i * kBlockThreads : chunks - 1;
        at[i] = (uint32_t)(((uint64_t)c * magic) >> shift);
        part[i] = slice * cpr + (c - at[i] * cpr);
        row[i] = (uint32_t)idx[at[i]];
    }
    u32x4 v[kGatherSteps];
#pragma unroll
    for (int i = 0; i < kGatherSteps; ++i) {
        const bool inside = row[i] < tableRows; // (a negative index is a large one)
        const uint32_t from = !SHORT || part[i] < rowChunks ? part[i] : rowChunks - 1;
        v[i] = *reinterpret_cast<const u32x4 *>(table + ((size_t)(inside ? row[i] : 0u) * rowChunks + from) * 16);
        if (!inside)
            v[i] = u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < kGatherSteps; ++i)
        if (first + i * kBlockThreads < chunks && (!SHORT || part[i] < rowChunks))
            __builtin_nontemporal_store(v[i], reinterpret_cast<u32x4 *>(out + ((size_t)at[i] * rowChunks + part[i]) * 16));
}

// The same for rows of any number of chunks, in slices that no 64 bytes of the output are cut by: what is dealt out is the pieces of four chunks
// (64 bytes) of the whole output, a piece to the slice that the column of its first chunk lies in; its last chunks may belong to the
// slice, or the row, behind.  Lane by lane `slots` chunks per row and slice, as many as a row can have there; a lane without one idles.
__global__ __launch_bounds__(kBlockThreads) void GatherPieces(char *out, const char *table, const int32_t *idx, uint32_t chunks, uint32_t rowChunks,
                                                              uint32_t slots, uint32_t units, uint32_t magic, int shift, uint32_t tableRows, uint32_t parts)
{
    typedef uint32_t u32x4 __attribute__((ext_vector_type(4), aligned(2)));
    const uint32_t xcd = blockIdx.x % 8, slice = xcd % parts, block = blockIdx.x / 8 * (8 / parts) + xcd / parts;
    const uint32_t first = block * (uint32_t)kGatherChunks + threadIdx.x;
    if (block * (uint32_t)kGatherChunks >= units)
        return;
    const uint32_t low = slice * rowChunks / parts, high = (slice + 1) * rowChunks / parts;
    uint32_t row[kGatherSteps], chunk[kGatherSteps], part[kGatherSteps];
    bool mine[kGatherSteps];
#pragma unroll
    for (int i = 0; i < kGatherSteps; ++i) {
        const uint32_t u = first + i * kBlockThreads < units ? first + i * kBlockThreads : units - 1;
        uint32_t at = (uint32_t)(((uint64_t)u * magic) >> shift);
        const uint32_t j = u - at * slots, begin = at * rowChunks, start = (begin + low + 3) & ~3u;
        chunk[i] = start + j;
        mine[i] = first + i * kBlockThreads < units && start + (j & ~3u) < begin + high && chunk[i] < chunks;
        part[i] = mine[i] ? chunk[i] - begin : low;
        if (part[i] >= rowChunks) {
            part[i] -= rowChunks;
            ++at;
        }
        row[i] = (uint32_t)idx[at];
    }
    u32x4 v[kGatherSteps];
#pragma unroll
    for (int i = 0; i < kGatherSteps; ++i) {
        const bool inside = row[i] < tableRows;
        v[i] = *reinterpret_cast<const u32x4 *>(table + ((size_t)(inside ? row[i] : 0u) * rowChunks + part[i]) * 16);
        if (!inside)
            v[i] = u32x4{0, 0, 0, 0};
    }
#pragma unroll
    for (int i = 0; i < kGatherSteps; ++i)
        if (mine[i])
            __builtin_nontemporal_store(v[i], reinterpret_cast<u32x4 *>(out + (size_t)chunk[i] * 16));
}

// One-tile TGATHER (index form), the half 16x1024 -> 16x128 case of the reference's tgather test.
__global__ __launch_bounds__(kBlockThreads) AICORE void TGatherIndex16x1024(__gm__ half *dst, __gm__ const half *src0,
                                                                            __gm__ const int32_t *idx)
{
    using Src0Tile = Tile<TileType::Vec, half, 16, 1024, BLayout::RowMajor>;
    using IdxTile = Tile<TileType::Vec, int32_t, 16, 128, BLayout::RowMajor>;
    using DstTile = Tile<TileType::Vec, half, 16, 128, BLayout::RowMajor>;
    using G0 = GlobalTensor<half, Shape<1, 1, 1, 16, 1024>, Stride<16384, 16384, 16384, 1024, 1>>;
    using GI = GlobalTensor<int32_t, Shape<1, 1, 1, 16, 128>, Stride<2048, 2048, 2048, 128, 1>>;
    using GD = GlobalTensor<half, Shape<1, 1, 1, 16, 128>, Stride<2048, 2048, 2048, 128, 1>>;
    Src0Tile s0;
    IdxTile ti;
    DstTile td;
    G0 g0(const_cast<half *>(src0));
    GI gi(const_cast<int32_t *>(idx));
    GD gd(dst);
    TLOAD(s0, g0);
    TLOAD(ti, gi);
    TGATHER(td, s0, ti);
    TSTORE(gd, td);
}

} // namespace

PTO_DEVICE_CODE_END

namespace {
template <typename D>
int launch_cvt(void *stream, D *dst, const float *src, size_t n, int mode)
{
    if (!dst || !src)
        return n == 0 ? PTO_OK : PTO_ERR_BAD_ARG;
    if (mode < PTO_CAST_RINT || mode > PTO_CAST_ODD)
        return PTO_ERR_BAD_ARG;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const size_t full = n / kCvtTile, tail = n % kCvtTile;
    // (the streaming kernel for buffers aligned to its accesses: 16-byte loads, 8-byte stores)
    const bool aligned = reinterpret_cast<uintptr_t>(src) % 16 == 0 && reinterpret_cast<uintptr_t>(dst) % 8 == 0;
    // the grid's x extent is limited to 2^31-1 blocks; stay far below it per launch
    constexpr size_t kMaxBlocks = 1u << 30;
    if (aligned) {
        using Kernel = void (*)(D *, const float *, size_t, size_t);
        Kernel kernel = CvtF32Stream<D, PTO_CAST_RINT, 4>;
        size_t piece = kCvtPiece<4>;
        if constexpr (std::is_same_v<D, half>) { // (bf16 has the one mode)
            static constexpr Kernel kByMode[] = {CvtF32Stream<D, PTO_CAST_RINT, 2>, CvtF32Stream<D, PTO_CAST_ROUND, 2>, CvtF32Stream<D, PTO_CAST_FLOOR, 2>,
                                                 CvtF32Stream<D, PTO_CAST_CEIL, 2>, CvtF32Stream<D, PTO_CAST_TRUNC, 2>, CvtF32Stream<D, PTO_CAST_ODD, 2>};
            if (mode != PTO_CAST_RINT || n >= (size_t)1 << 24) {
                kernel = kByMode[mode - PTO_CAST_RINT];
                piece = kCvtPiece<2>;
            }
        }
        const size_t pieces = (n + piece - 1) / piece;
        for (size_t t0 = 0; t0 < pieces; t0 += kMaxBlocks) {
            const size_t nb = pieces - t0 < kMaxBlocks ? pieces - t0 : kMaxBlocks;
            kernel<<<dim3((unsigned)nb), dim3(kBlockThreads), 0, st>>>(dst, src, n, t0);
        }
        return pto_amd::check_launch();
    }
    for (size_t t0 = 0; t0 < full; t0 += kMaxBlocks) {
        const size_t nb = full - t0 < kMaxBlocks ? full - t0 : kMaxBlocks;
        CvtF32<D, false><<<dim3((unsigned)nb), dim3(kBlockThreads), 0, st>>>(dst, src, n, t0, mode);
    }
    if (tail)
        CvtF32<D, true><<<dim3(1), dim3(kBlockThreads), 0, st>>>(dst, src, n, full, mode);
    return pto_amd::check_launch();
}
} // namespace

extern "C" int pto_tcvt_f32_f16(void *stream, uint16_t *dst, const float *src, size_t n, int round_mode)
{
    return launch_cvt(stream, reinterpret_cast<half *>(dst), src, n, round_mode);
}

extern "C" int pto_tcvt_f32_bf16(void *stream, uint16_t *dst, const float *src, size_t n, int round_mode)
{
    if (round_mode != PTO_CAST_RINT)
        return PTO_ERR_UNSUPPORTED;
    return launch_cvt(stream, reinterpret_cast<bfloat16_t *>(dst), src, n, round_mode);
}

extern "C" int pto_gather_rows(void *stream, void *out, const void *table, const int32_t *idx, size_t n_idx,
                               size_t table_rows, size_t cols, int elem_bytes)
{
    if (n_idx == 0 || cols == 0)
        return PTO_OK;
    if (!out || !table || !idx || table_rows == 0)
        return PTO_ERR_BAD_ARG;
    if (elem_bytes != 2 && elem_bytes != 4)
        return PTO_ERR_BAD_ARG;
    if (cols % 8 || n_idx > 0x7fffffffu || table_rows > 0x7fffffffu || cols > 0x7fffffffu)
        return PTO_ERR_UNSUPPORTED;
    const size_t rowChunks = cols * (size_t)elem_bytes / 16; // cols % 8 == 0: whole chunks; below 2^30
    uint32_t parts = 1;
    size_t cpr = rowChunks;
    // Slices, as few as bring a slice of the table down to 1 MiB of an XCD's 4 MiB of L2, where the batch reads a row twice or more
    // on average (65536 rows of 2 KiB from a table of 16384: 38.3 us in one slice, 33.1 in four, 28.2 in eight; a table of 65536
    // rows, 43.9 in one, 48.5 in eight; slices of 2 MiB take 6 % longer with tables of 5 and 6 MiB).  Of whole 128-byte lines where
    // the rows are; else of six and more half lines where the rows are whole numbers of those (16639 rows of 5696 bytes out of
    // 1972: 24.6 us whole, 17.5 in eight); at most an eighth of the lanes idle past a shorter last slice (32768 rows of 3840 bytes
    // out of 8192: 33.7 whole, 25.9 in eight).  Lines cut by a slice are written twice, in part: slices of other rows (20000 of
    // 2064 bytes 12.0 us, so cut 14.1) and into an output off the 16 bytes (the first of these 58.6, whole 38.6) lose more than they win.
    if (n_idx >= 2 * table_rows && rowChunks % 4 == 0 && reinterpret_cast<uintptr_t>(out) % 16 == 0)
        for (const size_t unit = rowChunks % 8 == 0 ? 8 : 4, least = rowChunks % 8 == 0 ? 8 : 24;
             parts < 8 && table_rows * rowChunks * 16 / parts > ((size_t)1 << 20); parts *= 2) {
            const size_t next = (rowChunks + 2 * parts * unit - 1) / (2 * parts * unit) * unit;
            if (next < least || next * 2 * parts * 7 > rowChunks * 8)
                break;
            cpr = next;
        }
    // Rows that this leaves whole, most of them of no whole number of 64 bytes: slices of the output's 64-byte pieces (GatherPieces), as few as bring a slice of
    // the table down to 1 MiB (us, whole / slices: a table in the memory-side cache; then one that is in no cache):
    //   8 MiB, 16 times:  rows of 105 chunks 32.7 / 24.5, 33.4 / 28.7   129 chunks 32.8 / 24.2, 33.2 / 28.2      4.25 MiB, 16 times: 129 chunks 16.1 / 13.5, 16.0 / 15.8
    //   8 MiB,  8 times:  rows of 253 chunks 17.6 / 14.1, 18.6 / 17.3   501 chunks 17.4 / 12.4, 18.4 / 16.7      24 MiB, 5 times: 501 chunks 34.5 / 24.5, 37.6 / 36.1
    // A slice reads lines at its edges that it uses in part, and those come from memory again where no cache has them.  Where the batch reads a row sixteen
    // times or more on average a slice of 24 chunks and more pays (of nine: 4.25 MiB read so 16.0 / 17.9; rows of 49 chunks in two 16.2 / 17.0); where it
    // reads it less often, four of 32 and more and eight of 56 and more (8 MiB read eight times, 129 chunks in four 17.8 / 14.4, 18.7 / 19.5; 73 in eight 17.9 / 14.7,
    // 19.1 / 23.0; 257 in eight 17.6 / 12.7, 18.6 / 18.8, in four 14.3, 18.0).  Nor where the L2 holds the whole table (88560 rows of 592 bytes out of
    // 4428 9.2 / 10.6), nor slices of short rows that it does not hold (57 chunks in two, 24 MiB read five times 36.3 / 39.5), nor for less than 28 MiB of
    // output (1100 of 4016 out of 275 3.9 / 4.2).
    const size_t tableBytes = table_rows * rowChunks * 16;
    const bool often = n_idx >= 16 * table_rows;
    uint32_t pieces = 1;
    if (parts == 1 && n_idx >= 4 * table_rows && rowChunks >= (often ? 64 : 128) && n_idx * rowChunks >= (size_t)7 << 18 && tableBytes > ((size_t)15 << 18) &&
        reinterpret_cast<uintptr_t>(out) % 64 == 0) {
        while (pieces < 8 && tableBytes / pieces > ((size_t)1 << 20) && rowChunks >= (often ? 48 : pieces < 4 ? 64 : 112) * pieces)
            pieces *= 2;
        if (rowChunks < 240 && tableBytes / pieces > ((size_t)1 << 22))
            pieces = 1;
    }
    if (pieces > 1)
        cpr = ((rowChunks + pieces - 1) / pieces + 3) / 4 * 4; // (chunks of a row whose number is a multiple of four, with the three behind: no more)
    int shift = 31;
    while (((size_t)1 << (shift - 31)) < cpr)
        ++shift;
    const uint32_t magic = (uint32_t)((((uint64_t)1 << shift) + cpr - 1) / cpr);
    hipStream_t st = static_cast<hipStream_t>(stream);
    const auto kernel = cpr * parts == rowChunks ? GatherChunks<false> : GatherChunks<true>;
    // (whole rows per launch, fewer than 2^31 chunks a slice)
    if (pieces > 1) { // (whole pieces per launch)
        const size_t most = 0x7fffffffu / rowChunks / 4 * 4;
        for (size_t r0 = 0; r0 < n_idx; r0 += most) {
            const size_t rows = n_idx - r0 < most ? n_idx - r0 : most, units = rows * cpr, blocks = (units + kGatherChunks - 1) / kGatherChunks;
            const size_t perGroup = 8 / pieces, groups = (blocks + perGroup - 1) / perGroup;
            GatherPieces<<<dim3((unsigned)(groups * 8)), dim3(kBlockThreads), 0, st>>>(
                static_cast<char *>(out) + r0 * rowChunks * 16, static_cast<const char *>(table), idx + r0, (uint32_t)(rows * rowChunks), (uint32_t)rowChunks,
                (uint32_t)cpr, (uint32_t)units, magic, shift, (uint32_t)table_rows, pieces);
        }
        return pto_amd::check_launch();
    }
    const size_t rowsPerLaunch = 0x7fffffffu / rowChunks;
    for (size_t r0 = 0; r0 < n_idx; r0 += rowsPerLaunch) {
        const size_t chunks = (n_idx - r0 < rowsPerLaunch ? n_idx - r0 : rowsPerLaunch) * cpr, blocks = (chunks + kGatherChunks - 1) / kGatherChunks;
        const size_t perGroup = 8 / parts, groups = (blocks + perGroup - 1) / perGroup;
        kernel<<<dim3((unsigned)(groups * 8)), dim3(kBlockThreads), 0, st>>>(
            static_cast<char *>(out) + r0 * rowChunks * 16, static_cast<const char *>(table), idx + r0, (uint32_t)chunks, (uint32_t)rowChunks,
            (uint32_t)cpr, magic, shift, (uint32_t)table_rows, parts);
    }
    return pto_amd::check_launch();
}

extern "C" int pto_tgather_index_f16_16x1024_16x128(void *stream, uint16_t *dst, const uint16_t *src0, const int32_t *idx)
{
    if (!dst || !src0 || !idx)
        return PTO_ERR_BAD_ARG;
    TGatherIndex16x1024<<<dim3(1), dim3(kBlockThreads), 0, static_cast<hipStream_t>(stream)>>>(
        reinterpret_cast<half *>(dst), reinterpret_cast<const half *>(src0), idx);
    return pto_amd::check_launch();
}
