// Decode of the dense operands (gemm_dense_kernel, gemm_tiled_kernel and gemm_prefill_kernel
// in iq3s_gemm.hip, gemm_wide_kernel in iq3s_wide.hip): every weight as an exact
// pair of E4M3 terms (SplitTables), in the order of the dense MFMA's B operand.
#pragma once
#include "iq3s_stream.h"

namespace {

// hi and lo words of code C of a group: level bytes select from the split table entry
// (tab.x/.y: hi of levels 0-3/4-7, tab.z/.w: lo); the four signs, moved onto bits
// 7,15,23,31 by one shift of the transposed sign word, are OR-ed into hi and XOR-ed into
// lo (one v_bitop3 each: a | (b & c) = 0xF8, a ^ (b & c) = 0x78).
template <int C>
__device__ __forceinline__ void split_word(uint32_t lv, uint32_t p, uint4 tab, int &hi, int &lo)
{
    const uint32_t r = funnel_shr(p, p, (25 + C) & 31);
    hi = (int)__builtin_amdgcn_bitop3_b32(__builtin_amdgcn_perm(tab.y, tab.x, lv), r, 0x80808080u, 0xF8);
    lo = (int)__builtin_amdgcn_bitop3_b32(__builtin_amdgcn_perm(tab.w, tab.z, lv), r, 0x80808080u, 0x78);
}

// Split-table entry of operand half X (0: bytes 0-15, 1: bytes 16-31) of MFMA H, from the
// lane's dense scale word (dense_scales: nibble 2X + H).
template <int H, int X>
__device__ __forceinline__ uint4 split_entry(const uint4 *split, uint32_t sc)
{
    return split[(sc >> (4 * (2 * X + H))) & 15u];
}

// MFMA H's hi and lo operands: codes 0-3 with the entry of half 0 (ta), 4-7 of half 1 (tb).
template <int H, int... C>
__device__ __forceinline__ void decode_split(const uint32_t (&s)[5], uint32_t p, const uint8_t *lvl, uint4 ta,
                                             uint4 tb, v8i &bhi, v8i &blo, std::integer_sequence<int, C...>)
{
    int h[8], l[8];
    (split_word<C>(*reinterpret_cast<const uint32_t *>(lvl + code_addr<8 * H + C>(s)), p, C < 4 ? ta : tb, h[C],
                   l[C]),
     ...);
    bhi = v8i{h[0], h[1], h[2], h[3], h[4], h[5], h[6], h[7]};
    blo = v8i{l[0], l[1], l[2], l[3], l[4], l[5], l[6], l[7]};
}

// Both halves of one tile-block (MFMA H = 0, 1).
__device__ __forceinline__ void decode_block(const WTile &w, const uint8_t *lvl, const uint4 *split, v8i (&bh)[2],
                                             v8i (&bl)[2])
{
    const uint32_t s[5] = {w.ia.x, w.ia.y, w.ia.z, w.ia.w, (uint32_t)w.ib};
    const uint32_t sc = dense_scales(w.sc);
    decode_split<0>(s, w.sg.x, lvl, split_entry<0, 0>(split, sc), split_entry<0, 1>(split, sc), bh[0], bl[0],
                    std::make_integer_sequence<int, 8>{});
    decode_split<1>(s, w.sg.y, lvl, split_entry<1, 0>(split, sc), split_entry<1, 1>(split, sc), bh[1], bl[1],
                    std::make_integer_sequence<int, 8>{});
}

} // namespace
