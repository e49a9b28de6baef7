// Flash-attention forward with the keys split over groups of wavefronts inside a workgroup of eight (FlashAttnFwd with
// G > 1): launches whose 128-query workgroups would leave SIMDs idle.  Two groups of four waves share
// 128 queries, four groups of two waves 64, eight groups of one wave 32; 128 KiB of K / V stages at head_dim 128 (key tiles of 64 and 32), 64 and
// 128 KiB at 64 (key tiles of 64).  What bounds a round: its chain of barrier, score MFMAs, softmax and output MFMAs, which all
// waves of the two- and four-group forms walk through together (128 queries x 4096 keys x 128, four groups: 1.05 us per round of 128 keys, of which the
// MFMAs of a SIMD take 0.43 and the copies 0.52).  16 heads x 512 queries x 2048 keys x 128, causal: 37.6 us with 64
// workgroups of four waves, 29.7 with two groups, 21.6 with four (23.2 with four groups of one wave, 256 workgroups).
// Eight groups of one wave have no such chain (FlashAttnFwd): the same problem 17.4 us, on 256 workgroups.  Bound there: a compute unit
// takes in all keys for 32 queries, 1 MiB at 64 bytes a clock = 7.3 us, of 10.2 us between first tile and last (MFMAs of a SIMD
// 3.6); 2.9 before the first tile is there, 2.2 for joining the groups, 2 at the launch.  Without raised priority for the MFMAs
// 17.4 becomes 17.7, with the V copies in a row behind the output MFMAs 18.3.  Measured and not taken: query blocks of a head that
// start at different keys (19.0: more lines on the way into the L2 at once), key tiles of 32 at head_dim 64 (no change).
#define PTO_WAVES_M 1
#define PTO_WAVES_N 8
#include <pto/pto-inst.hpp>

#include "fa_kernels.hpp"

namespace {
template <int D, int BKV, int G>
int launch_split(hipStream_t st, void *o, float *lse, const half *q, const half *k, const half *v, int batch, int heads, int seqQ, int seqKv,
                 bool causal, bool oFp32, int causalOff)
{
    if (causal)
        return oFp32 ? launch_fa<D, true, true, 1, BKV, false, 1, G>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff)
                     : launch_fa<D, true, false, 1, BKV, false, 1, G>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff);
    return oFp32 ? launch_fa<D, false, true, 1, BKV, false, 1, G>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff)
                 : launch_fa<D, false, false, 1, BKV, false, 1, G>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff);
}
} // namespace

namespace pto_amd {
int fa_fwd_split(hipStream_t st, void *o, float *lse, const half *q, const half *k, const half *v, int batch, int heads, int seqQ, int seqKv,
                 int headDim, bool causal, bool oFp32, int causalOff, int groups)
{
    if (headDim == 128 && groups == 2)
        return launch_split<128, 64, 2>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causal, oFp32, causalOff);
    if (headDim == 128 && groups == 4)
        return launch_split<128, 32, 4>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causal, oFp32, causalOff);
    if (headDim == 64 && groups == 2)
        return launch_split<64, 64, 2>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causal, oFp32, causalOff);
    if (headDim == 64 && groups == 4)
        return launch_split<64, 64, 4>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causal, oFp32, causalOff);
    if (headDim == 128 && groups == 8)
        return launch_split<128, 32, 8>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causal, oFp32, causalOff);
    if (headDim == 64 && groups == 8)
        return launch_split<64, 64, 8>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causal, oFp32, causalOff);
    return PTO_ERR_UNSUPPORTED;
}
} // namespace pto_amd
