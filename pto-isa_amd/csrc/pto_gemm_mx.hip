// MXFP8 / MXFP4 GEMM for MI355X: C[m,n] = (A .* 2^(scaleA-127)) x (B .* 2^(scaleB-127)), fp8 (e4m3 / e5m2) or fp4
// (e2m1, two per byte) operands with one e8m0 scale per row (column) and 32-wide k block, fp32 accumulation, bf16 or
// fp32 result.
//
// Mirrors the reference kernels kernels/manual/a5/matmul_mxfp8_performance/mxmatmul_performance_kernel.cpp:149-241 and
// kernels/manual/a5/matmul_mxfp4_performance/mxmatmul_performance_kernel.cpp (TLOAD of operand and scale panels ->
// TEXTRACT -> TMATMUL_MX -> TSTORE): A [m,k], B stored [n,k], scaleA [m,k/32], scaleB stored [n,k/32]
// (scripts/gen_data.py:31-66).
//
// Structure: the fp16 GEMM's K-step pipeline (workgroup tile 256 x 256, 8 waves in a 2 x 4 grid, four LDS stages of
// one 64-byte K-step filled by asynchronous copies, copies / fragment reads / MFMAs interleaved by the scheduler
// directives).  A K-step is 64 fp8 values = the same 64 bytes per row as 32 fp16 values, and one
// v_mfma_scale_f32_32x32x64_f8f6f4 (16 passes) takes the place of two v_mfma_f32_32x32x16_f16 (8 passes each), so
// bytes moved per MFMA cycle are those of the fp16 kernel at twice the flops.  The scales of 512 k (16 blocks = 16
// bytes per row) come into LDS once per eight K-steps with one 16-byte asynchronous copy instruction per wave, are
// rearranged there into the image of a Mat tile of block scales (the scales of one step of consecutive rows in
// consecutive words: a 64-lane read of words 16 bytes apart costs 6 LDS cycles instead of 2), and the two scales a lane
// needs for a K-step are read with the step's fragments (one ds_read_u8 per 32-row block); the MFMA applies them.
// fp4: a 64-byte K-step holds 128 k = two MFMAs (8 passes each) per fragment pair and four scale blocks (one ds_read_b32
// per 32-row block); a scale group is four K-steps.  Same bytes per step again, at four times the fp16 flops.
// m and n need not be multiples of the tile: the last tile row / column is moved back to end at m / n and recomputes
// what it overlaps (m, n >= 256).
#define PTO_WAVES_M 2
#define PTO_WAVES_N 4
#include "gemm_kernels.hpp"


PTO_DEVICE_CODE_BEGIN

namespace {

constexpr int kMxStepBytes = 64; // one K-step per operand row in LDS
// K-steps per scale group (16 k blocks = one 16-byte scale row): 8 steps of 64 k (8-bit) or 4 steps of 128 k (4-bit)
template <typename T>
constexpr int kMxGroupSteps = 16 / (kMxStepBytes * 8 / detail::elem_bits<T> / 32);

// One asynchronous copy instruction per wave: the 16-byte scale rows (16 k blocks = one scale group) of the workgroup's
// BM rows of A and BN columns of B -> LDS [BM + BN][16 bytes].  Instruction i covers 64 rows; wave w issues instruction
// w % ((BM + BN) / 64) (with fewer instructions than waves some waves repeat one: same data to the same place).
template <int BM, int BN>
AICORE inline void LoadScaleRows(uint32_t ldsOff, __gm__ const uint8_t *sa, __gm__ const uint8_t *sb, int64_t ld)
{
    constexpr int nA = BM / 64, nB = BN / 64;
    static_assert(BM % 64 == 0 && BN % 64 == 0 && nA + nB <= kBlockWaves, "one scale copy instruction per wave");
    int lane = hw::lane();
    // (used once per eight K-steps: keeps the address arithmetic from being hoisted into registers that live across the loop)
    asm volatile("" : "+v"(lane));
    const int inst = hw::wave() % (nA + nB);
    const bool isA = inst < nA;
    const char *base = reinterpret_cast<const char *>(isA ? sa : sb);
    const int row = (isA ? inst : inst - nA) * 64;
    const char *g = detail::uniform_ptr(base + (int64_t)row * ld) + (uint32_t)lane * (uint32_t)ld;
    __builtin_amdgcn_global_load_lds(PTO_GLOBAL_PTR(g), PTO_LDS_PTR(hw::lds_base() + ldsOff + inst * 1024), 16, 0, 0);
}

// [BM + BN][16 bytes] scale rows at `rawOff` -> the LDS images of a [BM, 16] left and a [16, BN] right Mat tile of block
// scales at `dstOff` and `dstOff + BM * 16` ([k block / 4][row][4 k blocks], see detail::ScaleMatGeom): one row per thread
// (with more threads than rows some rows are done twice: same data to the same place, no branch).
template <int BM, int BN>
AICORE inline void RearrangeScaleRows(uint32_t dstOff, uint32_t rawOff)
{
    static_assert(kBlockThreads % (BM + BN) == 0, "one scale row per thread");
    int t = hw::tid();
    asm volatile("" : "+v"(t)); // (as in LoadScaleRows: recompute the addresses rather than keep them in registers)
    t %= BM + BN;
    char *lds = hw::lds_base();
    const u32x4 v = *reinterpret_cast<const u32x4 *>(lds + rawOff + t * 16);
    const bool isA = t < BM;
    char *dst = lds + dstOff + (isA ? 0 : BM * 16) + (isA ? t : t - BM) * 4;
    const int major = isA ? BM : BN;
#pragma unroll
    for (int q = 0; q < 4; ++q)
        *reinterpret_cast<uint32_t *>(dst + q * major * 4) = v[q];
}

template <typename FA, typename FB, typename OutT, int BM, int BN, int STAGES, bool DEEP>
AICORE inline __attribute__((always_inline)) void MxTileRows(__gm__ OutT *out, __gm__ const FA *src0, __gm__ const FB *src1,
                                                             __gm__ const uint8_t *scale0, __gm__ const uint8_t *scale1, int m,
                                                             int n, int k, int row0, int col0)
{
    static_assert(detail::elem_bits<FA> == detail::elem_bits<FB>, "operands of one width");
    // the tile origin comes out of integer divisions, which run on the vector unit: move it (and with it every panel
    // pointer below) into scalar registers
    row0 = __builtin_amdgcn_readfirstlane(row0);
    col0 = __builtin_amdgcn_readfirstlane(col0);
    constexpr int BK = kMxStepBytes * 8 / detail::elem_bits<FA>; // k per K-step
    constexpr int kGroupSteps = kMxGroupSteps<FA>, kStepBlocks = BK / 32;
    constexpr int HM = BM / 2, KB = 16;
    using X = float8_e8m0_t;
    using TileMatA = Tile<TileType::Mat, FA, BM, BK, BLayout::ColMajor, BM, BK, SLayout::RowMajor>;
    using TileMatB = Tile<TileType::Mat, FB, BK, BN, BLayout::RowMajor, BK, BN, SLayout::ColMajor>;
    using TileScaleA = Tile<TileType::Mat, X, BM, KB, BLayout::RowMajor, BM, KB, SLayout::NoneBox>;
    using TileScaleB = Tile<TileType::Mat, X, KB, BN, BLayout::ColMajor, KB, BN, SLayout::NoneBox>;
    using LeftHalf = TileLeft<FA, HM, BK, HM, BK>;
    using RightTile = TileRight<FB, BK, BN, BK, BN>;
    using LeftScaleStep = TileLeftScale<X, HM, kStepBlocks>;
    using RightScaleStep = TileRightScale<X, kStepBlocks, BN>;
    using AccHalf = TileAcc<float, HM, BN, HM, BN>;
    using ShapeA = TileShape2D<FA, BM, BK, Layout::ND>;
    using StrideA = BaseShape2D<FA, DYNAMIC, DYNAMIC, Layout::ND>;
    using GlobalA = GlobalTensor<FA, ShapeA, StrideA, Layout::ND>;
    using ShapeB = TileShape2D<FB, BK, BN, Layout::DN>;
    using StrideB = BaseShape2D<FB, DYNAMIC, DYNAMIC, Layout::DN>;
    using GlobalB = GlobalTensor<FB, ShapeB, StrideB, Layout::DN>;
    using ShapeC = TileShape2D<OutT, HM, BN, Layout::ND>;
    using StrideC = BaseShape2D<OutT, DYNAMIC, DYNAMIC, Layout::ND>;
    using GlobalC = GlobalTensor<OutT, ShapeC, StrideC, Layout::ND>;

    constexpr uint32_t kABytes = BM * kMxStepBytes, kBBytes = kMxStepBytes * BN;
    constexpr uint32_t kStage = kABytes + kBBytes;
    // scale rows as copied, then two buffers of rearranged scales (the current group's and the next one's)
    constexpr uint32_t kScaleBytes = (BM + BN) * 16, kRawOff = STAGES * kStage, kScaleOff = kRawOff + kScaleBytes;
    constexpr int kLoadsPerStep = TLoadInstrs<TileMatA>() + TLoadInstrs<TileMatB>();
    constexpr int kScaleLoads = 1; // copy instructions per wave and scale group
    constexpr int kMfma = 2 * AccHalf::Storage::MB * AccHalf::Storage::NB * LeftHalf::Storage::KS;
    constexpr int kReadsA = 2 * LeftHalf::Storage::MB, kReadsB = 2 * RightTile::Storage::NB; // two ds_read_b128 per fragment
    constexpr int kReads = 2 * kReadsA + kReadsB + (2 * LeftHalf::Storage::MB + RightTile::Storage::NB); // + the scale reads
    // issue pattern of a step: the copies first, one MFMA before each; the fragment reads spread over the next MFMAs;
    // the last MFMA has no read after it
    constexpr int kMfmaCopies = kMfma >= 8 ? kLoadsPerStep : 1, kMfmaTail = 1;
    constexpr int kMfmaForReads = kMfma - kMfmaCopies - kMfmaTail;
    static_assert(STAGES == 4, "two fragment sets alternate with the stage index");
    static_assert(kMfmaForReads >= 0, "issue pattern below");

    // (operand pointers advance in bytes: one byte per 8-bit element, two 4-bit elements per byte)
    __gm__ FA *aPanel = const_cast<FA *>(src0) + (int64_t)row0 * k * detail::elem_bits<FA> / 8;
    __gm__ FB *bPanel = const_cast<FB *>(src1) + (int64_t)col0 * k * detail::elem_bits<FB> / 8;
    const int64_t ldScale = k / 32;
    __gm__ const uint8_t *saPanel = scale0 + (int64_t)row0 * ldScale;
    __gm__ const uint8_t *sbPanel = scale1 + (int64_t)col0 * ldScale;
    const StrideA strideA(m, k);
    const StrideB strideB(k, n);
    const int kLoop = k / BK, groups = kLoop / kGroupSteps;

    TileMatA aMat[STAGES];
    TileMatB bMat[STAGES];
#pragma unroll
    for (int s = 0; s < STAGES; ++s) {
        TASSIGN(aMat[s], s * kStage);
        TASSIGN(bMat[s], s * kStage + kABytes);
    }
    TileScaleA aScaleMat;
    TileScaleB bScaleMat;
    TASSIGN(aScaleMat, kScaleOff);
    TASSIGN(bScaleMat, kScaleOff + BM * 16);

    // Operand fragments and their scales.  The lower row half and B have two sets: the MFMAs of step it read set it % 2
    // while the other arrives.  The upper row half, whose MFMAs come first in a step, has one (the register file of two
    // waves per SIMD does not hold a second): its reads for the next step follow its last MFMA and have half a step to land.
    LeftHalf aUp, aDn[2];
    RightTile bAll[2];
    LeftScaleStep saUp, saDn[2];
    RightScaleStep sbAll[2];
    AccHalf cUp, cDn;
#pragma unroll
    for (int mb = 0; mb < AccHalf::Storage::MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < AccHalf::Storage::NB; ++nb)
#pragma unroll
            for (int i = 0; i < detail::kAccElems; ++i) {
                cUp.st.f[mb][nb][i] = 0.0f;
                cDn.st.f[mb][nb][i] = 0.0f;
            }

    // prologue: the scales of group 0, then kAhead K-steps in flight.  DEEP: a step's copies are issued STAGES steps
    // ahead, into the stage whose fragments were read one step earlier (every wave drains its LDS reads before the step's
    // barrier), instead of STAGES-1 steps ahead: they have three K-steps to land instead of two.
    constexpr int kAhead = DEEP ? STAGES : STAGES - 1;
    LoadScaleRows<BM, BN>(kRawOff, saPanel, sbPanel, ldScale);
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
        GlobalA gmA(aPanel + (int64_t)s * kMxStepBytes, ShapeA(), strideA);
        GlobalB gmB(bPanel + (int64_t)s * kMxStepBytes, ShapeB(), strideB);
        TLOAD(aMat[s], gmA);
        TLOAD(bMat[s], gmB);
    }
    wait_flag_pending<(kAhead - 1) * kLoadsPerStep>(PIPE_MTE2, PIPE_MTE1, EVENT_ID0); // scales and stage 0 are complete
    RearrangeScaleRows<BM, BN>(kScaleOff, kRawOff);
    hw::lds_barrier();
    {   // scale rows of group 1: rearranged two steps into group 0
        const int g = 1 < groups ? 1 : groups - 1;
        LoadScaleRows<BM, BN>(kRawOff, saPanel + g * 16, sbPanel + g * 16, ldScale);
    }
    TEXTRACT(saUp, aScaleMat, 0, 0);
    TEXTRACT(saDn[0], aScaleMat, HM, 0);
    TEXTRACT(sbAll[0], bScaleMat, 0, 0);
    TEXTRACT(aUp, aMat[0], 0, 0);
    TEXTRACT(aDn[0], aMat[0], HM, 0);
    TEXTRACT(bAll[0], bMat[0], 0, 0);

    // K-step j of a scale group (compile-time: LDS stage j % 4, fragment set j % 2, scales of k blocks 2j, 2j+1 of the
    // group).  Scale buffer group % 2 holds the group's scales.  Past the end of K the copies re-fetch the last K-step /
    // scale group and the reads fetch values nobody uses.
    auto step = [&](auto jTag, int it, int group) {
        constexpr int j = decltype(jTag)::value;
        constexpr int s = j % STAGES, sNext = (s + 1) % STAGES, sLoad = (s + kAhead) % STAGES;
        // the copies of K-step it+1 have landed; only those of the kAhead-2 steps after it may still be in flight, and the
        // scale copy that follows the copies of a group's last step while that step is among them
        hw::wait_vm<(kAhead - 2) * kLoadsPerStep + (j <= kAhead - 3 ? kScaleLoads : 0)>();
        if constexpr (DEEP)
            hw::wait_lgkm0(); // this wave's reads of the stage that the copies below overwrite (issued last step) are done
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_sched_barrier(0);
        const uint32_t otherBuf = kScaleOff + (uint32_t)((group + 1) & 1) * kScaleBytes;
        if constexpr (j == 2) {
            // The scale rows of the next group, copied during the previous group's last step (in the prologue for
            // group 1), have landed: the wait above covers every copy older than step 0's.  Into the other buffer, whose
            // scales were last read in the previous group; first read in this group's last step, a barrier later.
            static_assert(kAhead - 3 < 2 && kGroupSteps > 3, "the scale copy is older than every copy that may be in flight here");
            RearrangeScaleRows<BM, BN>(otherBuf, kRawOff);
            __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (j == kGroupSteps - 1) { // the next step is the first of the next group
            TASSIGN(aScaleMat, otherBuf);
            TASSIGN(bScaleMat, otherBuf + BM * 16);
        }
        const int fetch = it + kAhead < kLoop ? it + kAhead : kLoop - 1;
        GlobalA gmA(aPanel + (int64_t)fetch * kMxStepBytes, ShapeA(), strideA);
        GlobalB gmB(bPanel + (int64_t)fetch * kMxStepBytes, ShapeB(), strideB);
        TLOAD(aMat[sLoad], gmA);
        TLOAD(bMat[sLoad], gmB);
        if constexpr (j == kGroupSteps - 1) {
            // scale rows of the group after the next one (every wave rearranged the next group's earlier in this group)
            const int g = group + 2 < groups ? group + 2 : groups - 1;
            LoadScaleRows<BM, BN>(kRawOff, saPanel + g * 16, sbPanel + g * 16, ldScale);
        }
        constexpr int p = j & 1, q = p ^ 1, kbNext = kStepBlocks * ((j + 1) % kGroupSteps);
        TMATMUL_MX(cUp, cUp, aUp, saUp, bAll[p], sbAll[p]);
        TEXTRACT(aUp, aMat[sNext], 0, 0);
        TEXTRACT(saUp, aScaleMat, 0, +kbNext);
        TMATMUL_MX(cDn, cDn, aDn[p], saDn[p], bAll[p], sbAll[p]);
        TEXTRACT(bAll[q], bMat[sNext], 0, 0);
        TEXTRACT(sbAll[q], bScaleMat, +kbNext, 0);
        TEXTRACT(aDn[q], aMat[sNext], HM, 0);
        TEXTRACT(saDn[q], aScaleMat, +HM, +kbNext);
#pragma unroll
        for (int i = 0; i < kLoadsPerStep + (j == kGroupSteps - 1 ? kScaleLoads : 0); ++i) {
            if (i < kMfmaCopies)
                __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
            __builtin_amdgcn_sched_group_barrier(0x010, 1, 0);
        }
        StaticFor<0, kReads>([](auto iTag) {
            constexpr int i = decltype(iTag)::value;
            constexpr int cnt = (i + 1) * kMfmaForReads / kReads - i * kMfmaForReads / kReads;
            if constexpr (cnt > 0)
                __builtin_amdgcn_sched_group_barrier(0x008, cnt, 0);
            __builtin_amdgcn_sched_group_barrier(0x100, 1, 0);
        });
        __builtin_amdgcn_sched_group_barrier(0x008, kMfmaTail, 0);
        __builtin_amdgcn_sched_barrier(0);
    };
    static_assert(kGroupSteps % STAGES == 0, "the LDS stage of a step is a compile-time constant");
    for (int group = 0; group < groups; ++group) {
        const int it = group * kGroupSteps;
        StaticFor<0, kGroupSteps>([&](auto jTag) { step(jTag, it + decltype(jTag)::value, group); });
    }
    hw::wait_vm0(); // the copies issued past the end of K must not outlive the workgroup's LDS
    GlobalC dstUp(out + (int64_t)row0 * n + col0, ShapeC(), StrideC(m, n));
    GlobalC dstDn(out + (int64_t)(row0 + HM) * n + col0, ShapeC(), StrideC(m, n));
    TSTORE(dstUp, cUp);
    TSTORE(dstDn, cDn);
}

// The first `fullTiles` workgroups (whole rounds over the compute units) own one BM x BN C tile each; with quarter != 0
// the tiles of the last, partial round are cut into four (BM/2) x (BN/2) tiles, one workgroup each.
template <typename FA, typename FB, typename OutT, int BM, int BN, int STAGES, int GROUP_M, bool DEEP>
__global__ __launch_bounds__(kBlockThreads, 1) AICORE
    void GemmMx(__gm__ OutT *out, __gm__ const FA *src0, __gm__ const FB *src1, __gm__ const uint8_t *scale0,
                __gm__ const uint8_t *scale1, int m, int n, int k, int fullTiles)
{
    const int tilesM = (m + BM - 1) / BM, tilesN = (n + BN - 1) / BN;
    const int block = (int)get_block_idx();
    int tm, tn;
    if (block >= fullTiles) { // (only when m and n are multiples of the tile)
        const int u = RegroupXcd(block - fullTiles, (tilesM * tilesN - fullTiles) * 4);
        TileOfId<GROUP_M>(fullTiles + u / 4, tilesM, tilesN, tm, tn);
        const int sub = u % 4;
        MxTileRows<FA, FB, OutT, BM / 2, BN / 2, STAGES, DEEP>(out, src0, src1, scale0, scale1, m, n, k, tm * BM + (sub >> 1) * (BM / 2),
                                                        tn * BN + (sub & 1) * (BN / 2));
        return;
    }
    TileOfId<GROUP_M>(RegroupXcd(block, fullTiles), tilesM, tilesN, tm, tn);
    // the last tile row / column ends at m / n: it recomputes the rows / columns it shares with its neighbour
    const int row0 = tm * BM + BM <= m ? tm * BM : m - BM, col0 = tn * BN + BN <= n ? tn * BN : n - BN;
    MxTileRows<FA, FB, OutT, BM, BN, STAGES, DEEP>(out, src0, src1, scale0, scale1, m, n, k, row0, col0);
}

} // namespace

PTO_DEVICE_CODE_END

namespace {

template <typename FA, typename FB, typename OutT, bool DEEP = true>
int launch_gemm_mx(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n,
                   int k, int tailMode)
{
    constexpr int BM = 256, BN = 256, STAGES = 4, GROUP_M = 4;
    if (m < BM || n < BN || k % 512) // 512 k = one 16-byte scale row in either operand width
        return PTO_ERR_UNSUPPORTED;
    constexpr int lds = STAGES * (BM + BN) * 64 + 3 * (BM + BN) * 16;
    auto kernel = GemmMx<FA, FB, OutT, BM, BN, STAGES, GROUP_M, DEEP>;
    static const int attr = pto_amd::allow_lds(kernel, lds);
    if (attr != PTO_OK)
        return attr;
    const int tiles = ((m + BM - 1) / BM) * ((n + BN - 1) / BN), cus = pto_amd::compute_units();
    int full = tiles / cus * cus;
    // quarter tiles move twice the operand bytes per flop: only when they fit one round
    if (tailMode == 0 || full == 0 || (tiles - full) * 4 > cus || m % BM || n % BN)
        full = tiles;
    kernel<<<dim3(full + (tiles - full) * 4), dim3(kBlockThreads), lds, st>>>(
        reinterpret_cast<OutT *>(c), reinterpret_cast<const FA *>(a), reinterpret_cast<const FB *>(b), sa, sb, m, n, k, full);
    return pto_amd::check_launch();
}

template <bool DEEP>
int gemm_mx_dispatch_fmt(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m,
                         int n, int k, int format, int c_fp32, int tailMode)
{
    if (format == 0)
        return c_fp32 ? launch_gemm_mx<float8_e4m3_t, float8_e4m3_t, float, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode) :
                        launch_gemm_mx<float8_e4m3_t, float8_e4m3_t, bfloat16_t, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode);
    if (format == 1)
        return c_fp32 ? launch_gemm_mx<float8_e5m2_t, float8_e5m2_t, float, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode) :
                        launch_gemm_mx<float8_e5m2_t, float8_e5m2_t, bfloat16_t, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode);
    // mixed fp8 operands (the MFMA takes a format per operand): 2 = A e4m3 x B e5m2, 3 = A e5m2 x B e4m3
    if (format == 2)
        return c_fp32 ? launch_gemm_mx<float8_e4m3_t, float8_e5m2_t, float, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode) :
                        launch_gemm_mx<float8_e4m3_t, float8_e5m2_t, bfloat16_t, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode);
    if (format == 3)
        return c_fp32 ? launch_gemm_mx<float8_e5m2_t, float8_e4m3_t, float, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode) :
                        launch_gemm_mx<float8_e5m2_t, float8_e4m3_t, bfloat16_t, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode);
    if (format == 4)
        return c_fp32 ? launch_gemm_mx<float4_e2m1x2_t, float4_e2m1x2_t, float, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode) :
                        launch_gemm_mx<float4_e2m1x2_t, float4_e2m1x2_t, bfloat16_t, DEEP>(st, c, a, b, sa, sb, m, n, k, tailMode);
    return PTO_ERR_UNSUPPORTED;
}

// variant: bit 0 = quarter tiles in the last round, bit 1 = copies issued STAGES-1 instead of STAGES steps ahead
int gemm_mx_dispatch(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n,
                     int k, int format, int c_fp32, int variant)
{
    return (variant & 2) ? gemm_mx_dispatch_fmt<false>(st, c, a, b, sa, sb, m, n, k, format, c_fp32, variant & 1) :
                           gemm_mx_dispatch_fmt<true>(st, c, a, b, sa, sb, m, n, k, format, c_fp32, variant & 1);
}

} // namespace

namespace {
// Three kernels: 256 x 256 tiles on eight wavefronts (this file; quarter tiles in a last partial round), tiles of 256 rows and 96 to 256
// columns on four (pto_gemm_mxw4_*.hip), and tiles of 32 .. 192 rows with k split over two groups of wavefronts
// (pto_gemm_mxks.hip).  What a problem takes with one tile shape, in microseconds, launch included: tiles are dealt to the
// compute units, `more` rounds beyond the first, `share` of the units busy in the last one, steps of 128 bytes,
//   time = fixed + per_round more + steps (step + step_round more + step_share share) + (per_mega + fp32 result: per_mega_f32) (4e-6 m n);
// the 256 x 256 tiles take `ragged` longer a step and round where m or n is no multiple of 256 (the last tiles are moved back).
// Least-squares fits to 1520 problems (256 x 256 x 512 .. 6144^3 ragged, .. 16384 x 8192 x 8192 in whole tiles, both results,
// three operand sets in turn) in which those near a shape's best use count most (root mean square of the relative error there
// 2 .. 5 %).  The k-split shapes are taken 2 %, the 256 x 256 tiles of either kind 3 % dearer than fitted (against moves on the noise of the
// fit); so chosen, a problem is 0.4 % (fp8) and 0.3 % (fp4) from its best shape on average, 12 % at worst, and 8 of the 1520
// are over 2 % slower than on 256-row tiles alone, the worst 10.6 % (with a fit to ragged bf16 problems only: 16, and 24 %).
// Against the 256-row tiles alone: 256 x 256 x 6144 fp8 34.0 -> 12.0 us, 512 x 512 x 2048 fp4 12.0 -> 4.9, 592 x 736 x 4096
// 24.6 -> 9.8, 2048^3 17.3 -> 13.5, geometric mean of the problems 1.58 (fp8), 1.66 (fp4).  (128 x 192 with fp8 is the best
// shape of 9 of 1002 problems, by up to 5 %: 1024 x 4608 x 1536.)
// 256 x 256 tiles on four wavefronts: fitted to 440 problems of 150 to 1024 such tiles, and compared with the other shapes only where the last round is
// 78 % full or more.  Taken for 133 of them, by 10 % on average (fp8, one of 0.980 the least gain) and 7 % (fp4, three 3 to 5 % slower):
// 2040 x 8100 x 8192 fp8 121 -> 104 us, fp4 70.3 -> 66.0; 4096^3 62 -> 54 and 40.6 -> 36.6; 8192^3 492 -> 418 and 308 -> 256.  Below 78 % and k of 1024 and more they are 4 to 17 % slower.
struct MxShape {
    enum Kernel { kBlock, kW4, kKs } kernel;
    int number, bm, bn;
    double fixed, perRound, step, stepRound, perMega, stepShare, perMegaF32;
};
// 256 x 96, 160 and 224: fitted to 300 problems of 0.7 million results and more each in fp8 and fp4, compared where the last round is 70 % full and taken 2 % dearer: for 61 of the
// 300 by 7 % (fp8) and 53 by 9 % (fp4) on average, for one of either more than 2 % slower (5 and 7 %).  5632 x 1536 x 512 fp8 to fp32 on 256 x 160 tiles -16 %,
// 3840 x 1536 x 1024 fp4 on 256 x 96 -15 %, 7424 x 3584 x 7168 fp8 on 256 x 224 -17 %.
// 32 x 32 and 32 x 64 with k split: fitted to 249 problems of up to 1.3 million results each in fp8 and fp4, both results (256 x 256 x 512 .. 1400 x 1000 x 7168), taken 3 % dearer and up to the
// five rounds of that fit: for 303 of 498 by 17 % (fp8) and 255 by 15 % (fp4) on average, for one 3 % slower (512 x 1024 x 2048 fp8; operands in turn, from
// graphs: times at gemm_kernels_mxks.hpp); past their two rounds the larger ones are faster (1024^3 fp8 64 x 64 5.1, 32 x 64 5.8, 32 x 32 6.4).
constexpr int kMxShapeCount = 15;
constexpr MxShape kMxShapes[2][kMxShapeCount] = {
    {{MxShape::kKs, 6, 32, 32, 2.750, 0.419, 0.117, 0.066, 0.000, 0.032, 0.081},
     {MxShape::kKs, 7, 32, 64, 2.922, 0.785, 0.120, 0.124, 0.000, 0.082, 0.086},
     {MxShape::kKs, 0, 64, 64, 2.595, 0.634, 0.196, 0.185, 0.191, 0.051, 0.027},
     {MxShape::kKs, 1, 64, 128, 3.318, 1.592, 0.277, 0.320, 0.188, 0.054, 0.039},
     {MxShape::kKs, 2, 128, 64, 3.318, 1.545, 0.284, 0.315, 0.201, 0.039, 0.036},
     {MxShape::kKs, 3, 128, 128, 4.635, 2.138, 0.354, 0.508, 0.146, 0.110, 0.048},
     {MxShape::kKs, 4, 128, 192, 5.785, 2.957, 0.481, 0.728, 0.124, 0.168, 0.059},
     {MxShape::kKs, 5, 192, 128, 5.833, 2.802, 0.482, 0.730, 0.129, 0.170, 0.056},
     {MxShape::kW4, 0, 256, 96, 4.642, 1.735, 0.532, 0.751, 0.065, 0.144, 0.101},
     {MxShape::kW4, 0, 256, 160, 7.914, 5.683, 0.436, 0.980, 0.024, 0.535, 0.069},
     {MxShape::kW4, 0, 256, 224, 8.683, 6.830, 0.837, 1.359, 0.000, 0.492, 0.075},
     {MxShape::kBlock, 0, 256, 256, 6.233, 4.744, 0.882, 1.791, 0.025, 0.728, 0.076},
     {MxShape::kW4, 0, 256, 256, 9.531, 8.670, 0.647, 1.435, 0.000, 0.784, 0.075},
     {MxShape::kW4, 0, 256, 192, 8.332, 5.596, 0.666, 1.163, 0.062, 0.369, 0.033},
     {MxShape::kW4, 0, 256, 128, 6.086, 2.935, 0.553, 0.842, 0.093, 0.144, 0.035}}, // fp8
    {{MxShape::kKs, 6, 32, 32, 3.162, 0.265, 0.121, 0.075, 0.000, 0.035, 0.076},
     {MxShape::kKs, 7, 32, 64, 3.255, 0.578, 0.136, 0.119, 0.000, 0.073, 0.101},
     {MxShape::kKs, 0, 64, 64, 2.952, 0.929, 0.213, 0.209, 0.125, 0.078, 0.033},
     {MxShape::kKs, 1, 64, 128, 3.633, 2.235, 0.289, 0.363, 0.135, 0.113, 0.039},
     {MxShape::kKs, 2, 128, 64, 3.647, 2.183, 0.294, 0.356, 0.147, 0.100, 0.038},
     {MxShape::kKs, 3, 128, 128, 4.723, 2.682, 0.406, 0.591, 0.136, 0.166, 0.045},
     {MxShape::kKs, 4, 128, 192, 5.718, 3.475, 0.547, 0.827, 0.125, 0.234, 0.054},
     {MxShape::kKs, 5, 192, 128, 5.765, 3.304, 0.543, 0.883, 0.122, 0.257, 0.056},
     {MxShape::kW4, 0, 256, 96, 5.728, 3.703, 0.484, 0.757, 0.000, 0.394, 0.113},
     {MxShape::kW4, 0, 256, 160, 8.388, 4.324, 0.510, 1.238, 0.000, 0.644, 0.094},
     {MxShape::kW4, 0, 256, 224, 7.526, 7.963, 1.089, 1.412, 0.000, 0.701, 0.098},
     {MxShape::kBlock, 0, 256, 256, 5.763, 3.741, 1.024, 2.102, 0.045, 0.821, 0.085},
     {MxShape::kW4, 0, 256, 256, 9.012, 5.823, 0.809, 2.199, 0.000, 0.939, 0.076},
     {MxShape::kW4, 0, 256, 192, 8.060, 6.472, 0.880, 1.293, 0.066, 0.435, 0.026},
     {MxShape::kW4, 0, 256, 128, 6.084, 3.053, 0.645, 0.951, 0.098, 0.213, 0.036}}, // fp4
};
// fp8, fp4: the round of 128 x 128 quarter tiles, fixed and a step; `ragged`
constexpr double kMxQuarter[2] = {0.000, 4.513}, kMxStepQuarter[2] = {0.830, 0.753}, kMxStepRagged[2] = {0.080, 0.125};

// Which shape; as pto_gemm.hip chooses, small tiles first and shapes passed over that could not win in one round of full speed
struct MxChoice {
    int m, n, k, cus;
    bool fp4, c_fp32;
    bool block = m >= 256 && n >= 256 && k % 512 == 0, w4 = m >= 256 && n >= 128 && n % 4 == 0 && k % (fp4 ? 1024 : 512) == 0;
    double steps = k / (fp4 ? 256 : 128), mega = 4e-6 * m * n;
    static bool Wide(const MxShape &s) { return s.kernel == MxShape::kW4 && s.bn == 256; }
    static bool Between(const MxShape &s) { return s.kernel == MxShape::kW4 && s.bn % 64 == 32; }
    bool Any() const { return block || w4; }
    bool Takes(const MxShape &s) const { return s.kernel == MxShape::kBlock ? block : s.kernel == MxShape::kW4 ? w4 && n >= s.bn : n % 4 == 0; }
    static double Factor(const MxShape &s)
    {
        return s.kernel == MxShape::kBlock || Wide(s) || s.bm == 32 ? 1.03 : s.kernel == MxShape::kKs || Between(s) ? 1.02 : 1.0;
    }
    double AtLeast(const MxShape &s) const { return (s.fixed + steps * s.step) * Factor(s); } // (no figure of a shape is negative)
    double Time(const MxShape &s) const
    {
        const long long tiles = (long long)((m + s.bm - 1) / s.bm) * ((n + s.bn - 1) / s.bn), rest = tiles % cus;
        double more = (double)((tiles - 1) / cus), share = (double)((tiles - 1) % cus + 1) / cus, extra = 0.0;
        if ((Wide(s) && share < 0.78) || (Between(s) && share < 0.70) || (s.bm == 32 && more > 4.0))
            return __builtin_inf();
        if (s.kernel == MxShape::kBlock && !(m % 256 == 0 && n % 256 == 0)) {
            extra = steps * kMxStepRagged[fp4] * (more + 1.0);
        } else if (s.kernel == MxShape::kBlock && rest > 0 && rest * 4 <= cus && tiles > cus) {
            more -= 1.0;
            share = 1.0;
            extra = kMxQuarter[fp4] + steps * kMxStepQuarter[fp4];
        }
        return (s.fixed + s.perRound * more + steps * (s.step + s.stepRound * more + s.stepShare * share) + (s.perMega + (c_fp32 ? s.perMegaF32 : 0.0)) * mega + extra) *
               Factor(s);
    }
    const MxShape &Best() const
    {
        const MxShape *best = nullptr;
        double bestTime = __builtin_inf();
        for (const MxShape &s : kMxShapes[fp4]) {
            if (!Takes(s) || AtLeast(s) >= bestTime)
                continue;
            const double time = Time(s);
            if (time < bestTime) {
                best = &s;
                bestTime = time;
            }
        }
        return *best; // (Any(): the 256 x 256 tiles of eight wavefronts, or those of 128 columns of four, take it)
    }
};

int gemm_mx_any(hipStream_t st, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *sa, const uint8_t *sb, int m, int n, int k,
                int format, int c_fp32)
{
    const MxChoice choice{m, n, k, pto_amd::compute_units(), format == 4, c_fp32 != 0};
    if (!choice.Any())
        return PTO_ERR_UNSUPPORTED;
    const MxShape &best = choice.Best();
    switch (best.kernel) {
    case MxShape::kW4: return pto_amd::gemm_mx_w4(st, c, a, b, sa, sb, m, n, k, format, c_fp32, best.bn);
    case MxShape::kKs: return pto_amd::gemm_mx_ks(st, c, a, b, sa, sb, m, n, k, format, c_fp32, best.number);
    default: return gemm_mx_dispatch(st, c, a, b, sa, sb, m, n, k, format, c_fp32, 1);
    }
}
} // namespace

extern "C" int pto_gemm_mxfp8(void *stream, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *scale_a,
                              const uint8_t *scale_b, int m, int n, int k, int format, int c_fp32)
{
    if (!c || !a || !b || !scale_a || !scale_b || m <= 0 || n <= 0 || k <= 0)
        return PTO_ERR_BAD_ARG;
    if (format < 0 || format > 3)
        return PTO_ERR_UNSUPPORTED;
    return gemm_mx_any(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, format, c_fp32);
}

extern "C" int pto_gemm_mxfp4(void *stream, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *scale_a,
                              const uint8_t *scale_b, int m, int n, int k, int c_fp32)
{
    if (!c || !a || !b || !scale_a || !scale_b || m <= 0 || n <= 0 || k <= 0)
        return PTO_ERR_BAD_ARG;
    return gemm_mx_any(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, 4, c_fp32);
}

#if defined(PTO_ST_HOOKS)
// The choice among the shapes without a launch (needs no device): the variant, as below (1: the 256 x 256 tiles of eight wavefronts), that the entry points take
// on `units` compute units; expected: the time of each variant, an infinity where it is none of them or does not take the problem
extern "C" int pto_gemm_mx_choice(int m, int n, int k, int format, int c_fp32, int units, double *expected)
{
    if (m <= 0 || n <= 0 || k <= 0 || units <= 0)
        return PTO_ERR_BAD_ARG;
    const MxChoice choice{m, n, k, units, format == 4, c_fp32 != 0};
    if (!choice.Any())
        return PTO_ERR_UNSUPPORTED;
    auto variant = [](const MxShape &s) {
        if (s.kernel == MxShape::kKs)
            return s.number + (s.number < 6 ? 7 : 11);
        return s.kernel == MxShape::kBlock ? 1 : s.bn == 192 ? 5 : s.bn == 128 ? 6 : s.bn == 256 ? 13 : s.bn == 96 ? 14 : s.bn == 160 ? 15 : 16;
    };
    if (expected != nullptr) {
        for (int v = 0; v < 19; ++v)
            expected[v] = __builtin_inf();
        for (const MxShape &s : kMxShapes[choice.fp4])
            if (choice.Takes(s))
                expected[variant(s)] = choice.Time(s);
    }
    return variant(choice.Best());
}

// Tuning hook (not part of the public header): variant bit 0 = quarter tiles in the last round, bit 1 = the shallower copy
// pipeline; format 0 / 1 = fp8 e4m3 / e5m2, 4 = fp4 e2m1.
extern "C" int pto_gemm_mxfp8_variant(void *stream, void *c, const uint8_t *a, const uint8_t *b, const uint8_t *scale_a,
                                      const uint8_t *scale_b, int m, int n, int k, int format, int c_fp32, int variant)
{
    if (!c || !a || !b || !scale_a || !scale_b || m <= 0 || n <= 0 || k <= 0 || variant < 0 || variant > 18)
        return PTO_ERR_BAD_ARG;
    if (variant >= 17) // 32 x 32 and 32 x 64 with k split
        return pto_amd::gemm_mx_ks(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, format, c_fp32, variant - 11);
    if (variant >= 13) // further widths on four wavefronts: 256, 96, 160, 224
        return pto_amd::gemm_mx_w4(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, format, c_fp32,
                                   variant == 13 ? 256 : variant == 14 ? 96 : variant == 15 ? 160 : 224);
    if (variant >= 7) // k split over two groups of wavefronts, shape by number
        return pto_amd::gemm_mx_ks(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, format, c_fp32, variant - 7);
    if (variant >= 5) // the four-wave engine: 5 = 256 x 192 tiles, 6 = 256 x 128
        return pto_amd::gemm_mx_w4(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, format, c_fp32, variant == 5 ? 192 : 128);
    if (variant == 4) // what the public entry points take
        return gemm_mx_any(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, format, c_fp32);
    return gemm_mx_dispatch(static_cast<hipStream_t>(stream), c, a, b, scale_a, scale_b, m, n, k, format, c_fp32, variant);
}
#endif // PTO_ST_HOOKS
