// sg_lanes.h -- register reductions over the lanes of a wave and the work item
// order shared by the unordered-pair kernels (sg_sym.hip, sg_sym64.hip, sg_adjsym.hip).
#pragma once

#include "sg_internal.h"

namespace sg {

// -------------------------------------------------------- lane reductions
// a + a of the other register half (lanes below 32) or b + b of the other
// half (lanes from 32): one step of a reduce-scatter in a swap and an add.
__device__ __forceinline__ float halves32(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(unsigned, a),
                                                    __builtin_bit_cast(unsigned, b), false, false);
    const unsigned lo = r[0], hi = r[1];
    return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
__device__ __forceinline__ float halves16(float a, float b)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(unsigned, a),
                                                    __builtin_bit_cast(unsigned, b), false, false);
    const unsigned lo = r[0], hi = r[1];
    return __builtin_bit_cast(float, lo) + __builtin_bit_cast(float, hi);
}
template <int CTRL>
__device__ __forceinline__ float dpp(float v)
{
    return __builtin_bit_cast(
        float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, true));
}
// One step over the lanes of a quad: the lanes with `upper` unset keep a, the
// others b, and both add the partner lane's.
template <int CTRL>
__device__ __forceinline__ float quad_step(float a, float b, bool upper)
{
    const float keep = upper ? b : a, send = upper ? a : b;
    return keep + dpp<CTRL>(send);
}
// The same over the two halves of a 16-lane row (lane l with l ^ 8), and over
// the halves of its eight-lane groups (l with l ^ 7): bank masks let two adds
// do what a select, a move and an add do, v[k] and v[k + half] becoming v[k].
// The s_nop are the two wait states a DPP operand needs after a VALU write
// (the compiler does not see into the block).
#define SG_STEP8(a, b)                                                                \
    "v_add_f32_dpp %" #a ", %" #a ", %" #a " row_ror:8 row_mask:0xf bank_mask:0x3\n\t" \
    "v_add_f32_dpp %" #a ", %" #b ", %" #b " row_ror:8 row_mask:0xf bank_mask:0xc\n\t"
#define SG_STEP4(a, b)                                                                       \
    "v_add_f32_dpp %" #a ", %" #a ", %" #a " row_half_mirror row_mask:0xf bank_mask:0x5\n\t" \
    "v_add_f32_dpp %" #a ", %" #b ", %" #b " row_half_mirror row_mask:0xf bank_mask:0xa\n\t"
__device__ __forceinline__ void row_halves8(float (&v)[16])
{
    asm("s_nop 1\n\t" SG_STEP8(0, 8) SG_STEP8(1, 9) SG_STEP8(2, 10) SG_STEP8(3, 11) SG_STEP8(4, 12)
            SG_STEP8(5, 13) SG_STEP8(6, 14) SG_STEP8(7, 15)
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]), "+v"(v[4]), "+v"(v[5]), "+v"(v[6]),
          "+v"(v[7])
        : "v"(v[8]), "v"(v[9]), "v"(v[10]), "v"(v[11]), "v"(v[12]), "v"(v[13]), "v"(v[14]),
          "v"(v[15]));
}
__device__ __forceinline__ void row_halves8(float (&v)[8])
{
    asm("s_nop 1\n\t" SG_STEP8(0, 4) SG_STEP8(1, 5) SG_STEP8(2, 6) SG_STEP8(3, 7)
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])
        : "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
}
template <int N>   // N >= 8 values, the first eight used
__device__ __forceinline__ void row_halves4(float (&v)[N])
{
    asm("s_nop 1\n\t" SG_STEP4(0, 4) SG_STEP4(1, 5) SG_STEP4(2, 6) SG_STEP4(3, 7) "s_nop 1\n\t"
        : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3])
        : "v"(v[4]), "v"(v[5]), "v"(v[6]), "v"(v[7]));
}
#undef SG_STEP8
#undef SG_STEP4

// Superblock pair of work item k: all pairs bi < bj first, then the
// diagonal ones (half the work), so that the launch ends on short items.
__device__ __forceinline__ void sym_item(int k, int nsb, int &bi, int &bj)
{
    const int noff = nsb * (nsb - 1) / 2;
    if (k >= noff) {
        bi = bj = k - noff;
        return;
    }
    bj = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)k)) * 0.5f);
    while (bj * (bj - 1) / 2 > k) --bj;
    while ((bj + 1) * bj / 2 <= k) ++bj;
    bi = k - bj * (bj - 1) / 2;
}

}  // namespace sg
