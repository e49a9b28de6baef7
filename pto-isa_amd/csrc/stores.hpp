// How the GEMM and attention kernels store their results: 16 bytes a lane and 64 bytes of a row to an instruction, for which lanes change
// places where the matrix instruction left them with less, and past the L2 where pto_amd::store_through says so.  Include after
// <pto/pto-inst.hpp>.  Attention 16 x 4096 x 128 121.5 -> 118.5 us against 8 bytes a lane into the L2, 128 x 2048 x 64 causal 96.2 -> 94.1, 256 heads x 256 x
// 256 x 64 11.0 -> 9.1 (10.0 in 64-byte pieces into the L2), 256 x 512 x 512 x 128 causal 47.6 -> 41.3 (43.7).
#pragma once
#include "common.hpp"

PTO_DEVICE_CODE_BEGIN

namespace {

// Four results, past the L2 or into it (pto_amd::store_through), at the alignment of an element.
// (s_nop 1: a store of more than 8 bytes reads its registers up to two wait states behind it, and the compiler does not see that this is one)
typedef float Four __attribute__((ext_vector_type(4)));
AICORE inline __attribute__((always_inline)) void StoreFour(float *p, Four v, int through)
{
    typedef float C4 __attribute__((ext_vector_type(4), aligned(4)));
    if (through)
        asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
    else
        *reinterpret_cast<C4 *>(p) = v;
}

typedef uint32_t Words4 __attribute__((ext_vector_type(4)));
// Eight results of two bytes likewise; the second four only where `both`
template <typename T>
AICORE inline __attribute__((always_inline)) void StoreEight(T *p, Words4 v, bool both, int through)
{
    static_assert(sizeof(T) == 2, "16-bit results");
    typedef uint32_t C4 __attribute__((ext_vector_type(4), aligned(2)));
    typedef uint32_t C2 __attribute__((ext_vector_type(2), aligned(2)));
    if (through) // (whole 64-byte pieces of a row: both)
        asm volatile("global_store_dwordx4 %0, %1, off sc0 sc1\n\ts_nop 1" ::"v"(p), "v"(v) : "memory");
    else if (both)
        *reinterpret_cast<C4 *>(p) = v;
    else
        *reinterpret_cast<C2 *>(p) = C2{v[0], v[1]};
}
AICORE inline uint32_t Bf16Pair(float lo, float hi) { return ::pto::detail::f32x2_to_bf16_bits_rne(lo, hi); }
AICORE inline uint32_t HalfPair(float lo, float hi)
{
    typedef _Float16 H2 __attribute__((ext_vector_type(2)));
    return __builtin_bit_cast(uint32_t, H2{(_Float16)lo, (_Float16)hi});
}
// The lanes 16 .. 31 (48 .. 63) of a against the lanes 0 .. 15 (32 .. 47) of b; the upper half of a against the lower half of b
AICORE inline __attribute__((always_inline)) void SwapRows(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
AICORE inline __attribute__((always_inline)) void SwapHalves(uint32_t &a, uint32_t &b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

} // namespace

PTO_DEVICE_CODE_END

namespace {
// is O [numBH, seqQ, D] stored past the L2?
inline int fa_through(const void *o, int d, bool f32, int numBH, int seqQ)
{
    const uint64_t row = (f32 ? 4ull : 2ull) * d;
    return pto_amd::store_through(o, row, row * seqQ * numBH);
}
} // namespace
