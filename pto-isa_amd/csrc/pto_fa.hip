// Flash-attention forward for MI355X: one fused kernel built from PTO tile instructions.
//
// Arithmetic follows the reference's streaming softmax and rescale stages
// (kernels/manual/common/flash_atten/pto_macro_fa_softmax.hpp:47-215, pto_macro_fa_gu.hpp:33-56):
//   per key tile X = q k^T (fp32);  M' = max(M, rowmax X);  alpha = exp(s (M - M'));
//   P = exp(s (X - M'));  S = alpha S + rowsum P;  O = alpha O + half(P) v;  at the end O /= S,
// s = 1/sqrt(head_dim), causal mask = -3.40282e38 added to the hidden scores.
//
// Structure.  The reference runs the four stages on two kinds of cores that hand tiles over
// through global-memory FIFOs (fa_performance_kernel.cpp:607-963).  A CDNA4 compute unit does
// matrix and vector work itself, so here a workgroup owns 128 query rows of one head and keeps
// scores, probabilities and the output accumulator in registers for the whole sweep over the keys:
//   * wave grid 1 x 4: every wave owns 32 queries and sees every key of the tile,
//   * the score tile is computed transposed, X^T = K Q^T (TMATMUL with K as the Left operand and
//     Q^T as the Right operand), so that in the MFMA accumulator layout one lane holds one query
//     and the per-query quantities (max, sum, alpha) are per-lane scalars: the row reductions of
//     the softmax are in-register, plus one exchange between the two half-waves for the max,
//   * P^T in accumulator layout already is a Right (B) operand for O^T = V^T P^T up to a
//     permutation of the keys inside a 16-key step; V^T is read from the row-major V tile in LDS
//     with the transposing ds_read_b64_tr_b16 using the same permutation, so P never moves,
//   * K and V tiles are double-buffered in LDS by asynchronous TLOADs.
#define PTO_WAVES_M 1
#define PTO_WAVES_N 4
#include <pto/pto-inst.hpp>

#include "fa_kernels.hpp"

namespace {
// head_dim 64, the keys split over two groups of two waves: 64 queries per workgroup, two workgroups per compute unit
int launch_split_w4(hipStream_t st, void *o, float *lse, const half *q, const half *k, const half *v, int batch, int heads, int seqQ, int seqKv,
                    bool causal, bool oFp32, int causalOff)
{
    if (causal)
        return oFp32 ? launch_fa<64, true, true, 2, 64, false, 1, 2>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff)
                     : launch_fa<64, true, false, 2, 64, false, 1, 2>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff);
    return oFp32 ? launch_fa<64, false, true, 2, 64, false, 1, 2>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff)
                 : launch_fa<64, false, false, 2, 64, false, 1, 2>(st, o, lse, q, k, v, batch, heads, seqQ, seqKv, causalOff);
}
} // namespace

#if defined(PTO_ST_HOOKS)
// Tuning hook (not part of the public header).
extern "C" int pto_fa_fwd_f16_variant(void *stream, void *o, float *lse, const uint16_t *q, const uint16_t *k,
                                      const uint16_t *v, int batch, int heads, int seq_q, int seq_kv, int head_dim,
                                      int causal, int variant)
{
    if (!o || !q || !k || !v || batch <= 0 || heads <= 0 || seq_q <= 0 || seq_kv <= 0)
        return PTO_ERR_BAD_ARG;
    if (causal && seq_kv < seq_q)
        return PTO_ERR_UNSUPPORTED;
    const int causalOff = seq_kv - seq_q;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const half *hq = reinterpret_cast<const half *>(q), *hk = reinterpret_cast<const half *>(k),
               *hv = reinterpret_cast<const half *>(v);
#define PTO_FA_VARIANT(VV, DD, CC, MB)                           \
    if (variant == VV && head_dim == DD && (causal != 0) == CC) \
        return launch_fa<DD, CC, false, MB>(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causalOff);
    PTO_FA_VARIANT(1, 128, false, 1)
    PTO_FA_VARIANT(2, 128, false, 2)
    PTO_FA_VARIANT(2, 128, true, 2)
    PTO_FA_VARIANT(1, 64, true, 1)
    PTO_FA_VARIANT(2, 64, true, 2)
    PTO_FA_VARIANT(5, 64, true, 3)
#undef PTO_FA_VARIANT
    if (variant == 10 && head_dim == 128)
        return pto_amd::fa_fwd_d128_w8(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causal != 0, false, causalOff);
    if (variant == 20 && head_dim == 128)
        return pto_amd::fa_fwd_d128_w8m16(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causal != 0, false, causalOff);
    if (variant == 21 && head_dim == 128) // fp32 output and LSE
        return pto_amd::fa_fwd_d128_w8m16(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causal != 0, true, causalOff);
    if (variant == 42 || variant == 44 || variant == 48) // keys over two, four or eight groups of waves
        return pto_amd::fa_fwd_split(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, head_dim, causal != 0, false, causalOff, variant - 40);
    if (variant == 32 && head_dim == 64) // over two groups of two waves
        return launch_split_w4(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causal != 0, false, causalOff);
    if (variant == 6 && head_dim == 128 && !causal)
        return launch_fa<128, false, false, 2, 32>(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causalOff);
    if (variant == 6 && head_dim == 64 && causal)
        return launch_fa<64, true, false, 3, 32>(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causalOff);
    if (variant == 8 && head_dim == 64 && causal) // 64 queries per wave
        return launch_fa<64, true, false, 2, 64, false, 2>(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causalOff);
    if (variant == 8 && head_dim == 64 && !causal)
        return launch_fa<64, false, false, 2, 64, false, 2>(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causalOff);
    return PTO_ERR_BAD_ARG;
}
#endif // PTO_ST_HOOKS

extern "C" int pto_fa_fwd_f16(void *stream, void *o, float *lse, const uint16_t *q, const uint16_t *k, const uint16_t *v,
                              int batch, int heads, int seq_q, int seq_kv, int head_dim, int causal, int o_fp32)
{
    if (!o || !q || !k || !v || batch <= 0 || heads <= 0 || seq_q <= 0 || seq_kv <= 0)
        return PTO_ERR_BAD_ARG;
    if ((head_dim != 64 && head_dim != 128) || seq_q % kBQ1 || seq_kv % kBKVDefault)
        return PTO_ERR_UNSUPPORTED;
    // causal == 1: the diagonal ends in the last key (query i sees keys j <= i + seq_kv - seq_q; needs seq_kv >= seq_q);
    // causal == 2: the diagonal starts in the first key (j <= i, the rule of the reference's kernel and generator:
    // fa_performance_kernel.cpp:298-299 and :757, scripts/gen_data.py:53), any seq_kv.  The same when seq_kv == seq_q.
    if (causal != 0 && causal != 1 && causal != 2)
        return PTO_ERR_BAD_ARG;
    if (causal == 1 && seq_kv < seq_q)
        return PTO_ERR_UNSUPPORTED;
    const int causalOff = causal == 2 ? 0 : seq_kv - seq_q;
    hipStream_t st = static_cast<hipStream_t>(stream);
    const half *hq = reinterpret_cast<const half *>(q), *hk = reinterpret_cast<const half *>(k),
               *hv = reinterpret_cast<const half *>(v);
    const int cus = pto_amd::compute_units();
    // At most one 128-query workgroup of four waves per compute unit: every SIMD has one wave or none, and the launch takes as
    // long as that wave needs for all keys of its queries.  The keys are split over groups of waves (FlashAttnFwd, G > 1) where
    // there are enough of them to pay for joining the groups.  With 64-query workgroups one per compute unit (us, 128 of 128
    // queries, no mask; four waves / two groups of four / four groups of two):
    //   head_dim 128, keys  128:  6.6 /  8.4 /  7.4   256:  8.8 / 10.0 /  8.7   1024: 21.5 / 19.2 / 15.2   4096: 71.1 / 54.2 / 44.1
    //   head_dim  64, keys  128:  4.7 /  5.7 /  5.5   512:  8.5 /  8.7 /  7.3   1024: 13.4 / 12.6 /  9.7   4096: 45.2 / 37.2 / 26.4
    // at head_dim 64 and fewer than 1024 keys workgroups of four waves, two groups of two, are better still (128: 4.6, 512: 6.9).
    // Between one half and one whole workgroup per compute unit two groups of four waves (us, 192 workgroups, four waves / split):
    //   head_dim 128, keys 512: 13.3 / 13.5   1024: 21.3 / 19.8   4096: 71.7 / 60.9;   64, 512: 8.7 / 8.8   1024: 13.7 / 13.0   4096: 45.2 / 38.3
    // and at head_dim 64 with a mask that hides a good part of the keys (up to two keys per query), where the 64-query
    // workgroups even out: 256: 6.8 / 6.0 (two groups of two), 1024: 15.2 / 10.4, 2048: 26.5 / 19.2.
    // Nearly one workgroup per compute unit and one to a head at head_dim 128: K and V come from memory once and bound the launch, from
    // 2048 keys (256 heads x 128 queries, four waves / split, keys 1024: 24.9 / 27.8   1536: 34.5 / 36.6   2048: 53.4 / 47.2).
    const long long blocks = (long long)batch * heads * (seq_q / 128);
    const bool fromMemory = head_dim == 128 && seq_q == 128 && blocks * 8 > cus * 7ll;
    const int keys = causal && seq_q < seq_kv - causalOff ? seq_q + causalOff : seq_kv; // that the last query sees
    int groups = 0; // 1: two groups of two waves
    // Four 32-query workgroups per 128 queries and still no more than one for a compute unit: eight groups of one wave, each
    // streaming its own keys without a barrier (us, form taken before / eight groups, 128 queries, no mask):
    //   64 heads,  128 keys: 6.5 /  6.0   320: 9.1 / 7.9   768: 12.5 / 10.6   1536: 18.8 / 15.2, at head_dim  64: 4.25 / 4.40, 5.7 / 5.2, 8.4 / 7.0, 11.8 / 9.6
    //    4 heads,  128 keys: 6.2 /  5.4   320: 8.2 / 7.0   768: 11.0 /  8.9   1536: 16.3 / 12.4, at head_dim  64: 4.11 / 4.10, 5.5 / 4.8, 7.6 / 6.0, 10.9 / 8.0
    // With more of them a second round comes in that costs as much as the first (80 heads, 1024 keys: 15.3 / 22.0).
    if (blocks * 4 <= cus && (head_dim == 128 || keys > 128))
        groups = 8;
    else if (blocks * 2 <= cus)
        groups = keys >= (head_dim == 128 ? 256 : 1024) ? 4 : head_dim == 64 ? 1 : 0;
    else if (blocks <= cus)
        groups = head_dim == 64 && causal && keys >= 256 && keys / 2 <= seq_q ? 1 : keys >= (fromMemory ? 2048 : 1024) ? 2 : 0;
    if (groups == 1)
        return launch_split_w4(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causal != 0, o_fp32 != 0, causalOff);
    if (groups > 1)
        return pto_amd::fa_fwd_split(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, head_dim, causal != 0, o_fp32 != 0, causalOff, groups);
    // head_dim 128 with enough work to give every compute unit a workgroup of eight wavefronts (256 queries): the
    // K / V tiles are shared by twice the queries and the two waves of a SIMD alternate between MFMA and softmax
    // phases (measured +10-15 % at B1 H16 S4096 over workgroups of four waves)
    if (head_dim == 128 && seq_q % 256 == 0) {
        const long long pairs = (long long)batch * heads, perPair = seq_q / 256;
        // Workgroups beyond the last whole round take as long as that round.  Up to half a round of them, whole heads, go into a launch
        // of their own, on the form that is best for so few (us, one launch / two; a round and 1/32, 1/8, 1/4, 1/2 of one):
        //   1024 keys: 61 / 46   61 / 47   62 / 52   64 / 62      2048: 109 / 76   108 / 77   108 / 85   111 / 102      8192: 406 / 280   405 / 307   417 / 337   431 / 381
        // (256 keys: 25 / 23, 25 / 23, 26 / 25, 27 / 28.  With a mask the workgroups differ in length and the last round fills by itself.)
        const long long whole = pairs * perPair / cus * cus / perPair, rest = pairs - whole;
        if (!causal && whole > 0 && rest > 0 && rest * perPair * 2 <= cus && seq_kv >= 512 && pairs <= 0x7fffffffLL) {
            const int r = pto_amd::fa_fwd_d128_w8m16(st, o, lse, hq, hk, hv, 1, (int)whole, seq_q, seq_kv, false, o_fp32 != 0, causalOff);
            if (r != PTO_OK)
                return r;
            const long long rows = whole * seq_q, keyRows = whole * seq_kv;
            return pto_fa_fwd_f16(stream, static_cast<char *>(o) + rows * head_dim * (o_fp32 ? 4 : 2), lse ? lse + rows : nullptr, q + rows * head_dim,
                                  k + keyRows * head_dim, v + keyRows * head_dim, 1, (int)rest, seq_q, seq_kv, head_dim, causal, o_fp32);
        }
        if (pairs * perPair >= cus) {
            // the same schedule on 16 x 16 x 32 MFMAs: +1.5 .. 3.6 % without a mask and for long causal sequences
            // (interleaved runs; B2 H16 S2048 causal is 6 % slower on it and stays on the 32 x 32 x 16 kernel)
            if (!causal || seq_kv >= 4096)
                return pto_amd::fa_fwd_d128_w8m16(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causal != 0, o_fp32 != 0, causalOff);
            return pto_amd::fa_fwd_d128_w8(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causal != 0, o_fp32 != 0, causalOff);
        }
    }
    // otherwise workgroups of four wavefronts (128 queries): two per compute unit at head_dim 128, three at 64
#define PTO_FA_CASE(DD, CC, FF)                                                                      \
    if (head_dim == DD && (causal != 0) == CC && (o_fp32 != 0) == FF)                                \
        return launch_fa<DD, CC, FF, (DD == 128 ? 2 : 3)>(st, o, lse, hq, hk, hv, batch, heads, seq_q, seq_kv, causalOff);
    PTO_FA_CASE(128, false, false)
    PTO_FA_CASE(128, false, true)
    PTO_FA_CASE(128, true, false)
    PTO_FA_CASE(128, true, true)
    PTO_FA_CASE(64, false, false)
    PTO_FA_CASE(64, false, true)
    PTO_FA_CASE(64, true, false)
    PTO_FA_CASE(64, true, true)
#undef PTO_FA_CASE
    return PTO_ERR_UNSUPPORTED;
}
