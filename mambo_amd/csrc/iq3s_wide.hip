// Projection for 33 tokens and more on V_MFMA_SCALE_F32_32X32X64_F8F6F4.
//
// A workgroup computes 32*MT tokens x 32*W weight rows with KG groups of W waves, each group
// taking a KG-th of the workgroup's K blocks; a wave owns two 16-row weight tiles (32 rows) and
// MT sub-tiles of 32 tokens. As in the tiled kernel
// (iq3s_gemm.hip) the block's activations are copied straight into double-buffered LDS, the
// weights are the exact two-term E4M3 operands of iq3s_dense.h, a block's sums are one MFMA
// chain (four K steps of 64 x hi/lo) and the block's fp16 d is applied in f32.
//
// Why 32 x 32 x 64 and not the 16 x 16 x 128 of the other kernels (measured in a loop of
// MFMAs and independent v_perm): a scaled MFMA of either shape keeps the SIMD's vector ALU
// from issuing for ~20 cycles, whatever the wave mix, so beside n vector instructions the
// 16 x 16 MFMA (32 cycles) takes max(37, 20 + 4.2 n) and the 32 x 32 one (64 cycles, twice
// the flops) max(74, 20 + 4.2 n): 53 against 2 x 37 cycles per 32 cycles of matrix work at 8
// instructions per 16 x 16 MFMA. And an activation fragment read from LDS (2 KiB) feeds 64
// MFMA cycles per term instead of 32, which halves the LDS traffic that the tiled kernel
// (51% of the CU's LDS cycles at 128 tokens) pays per flop.
//
// One K step (64 of K) is the pipeline's unit: its 2*MT MFMAs run while the next step's eight
// codes per lane are decoded between them (codebook words requested one sub-tile ahead, the
// activation fragment of sub-tile mt+1 requested before sub-tile mt's second MFMA), and the
// block's 16*MT f32 scalings are spread over the last and the next block's first step. The
// packed words of the next block are requested as soon as their registers' last code is
// decoded (a second block in flight measured no faster). 233 to 244 VGPRs at MT = 4, so two waves
// per SIMD. What bounds it there is both the clock, which falls to 1.9 of 2.4 GHz under these MFMAs
// (1.83 to 1.94 by GRBM_GUI_ACTIVE over launches of 0.3 ms and more), and the third of the MFMA cycles
// that stay idle (60-69% busy at 8192 tokens, 67% on the 70B gate/up at 512; the waves wait for LDS,
// memory or the barrier for 19-30% of their cycles and to issue for 32-38%): 2.45 to 2.67 PFLOP/s
// executed, half of it useful. Up to a few hundred tokens it is the latency of a step's dependent chain.
//
// Two K groups (their sums meet in LDS at the end) put two waves on each SIMD where a launch
// has a workgroup per CU or less: one wave leaves its SIMD idle while a step's chain of LDS
// reads, decode and MFMAs completes (1.26 us a block of 64 tokens against 1.82 for two waves'),
// and a K split over half as many workgroups costs half the atomics. One group against two,
// each at its fastest split (us): 28672 x 4096 at 48 tokens 29.3 -> 26.2, 10240 x 8192 at 256
// 59 -> 57, 6144 x 4096 at 256 25.9 -> 22.7, 8192 x 28672 at 128 75 -> 72, 4096 x 14336 at 256
// 45.4 -> 44.7. Launches that fill the chip gain nothing from it (57344 x 8192 at 48: 82 and 85).
// Four groups of two waves (64 x 64 tiles) where even that leaves CUs without a workgroup: 8192 x
// 8192 at 96 and 128 tokens 30.4 -> 27.6 and 32.8 -> 28.2, 6144 x 4096 18.3 -> 16.0 and 19.7 -> 16.2.
// One 32-token sub-tile (MT = 1, reads a K step ahead) was built too and is level with the tiled
// and dense kernels at 8 to 32 tokens (57344 x 8192 at 16 / 32 63 and 70 us against 54 and 70, 28672
// x 4096 18 and 20 against 17 and 20): left out.
//
// Measured against the kernels it takes over from, same box, one launch in a replayed graph
// over rotated weights (us): 57344 x 8192 at 40 / 128 / 512 tokens 140 -> 87, 144 -> 122, 504 ->
// 420; 10240 x 8192 at 256 / 512 65 -> 56, 113 -> 87; 8192 x 28672 at 128 / 192 / 512 86 -> 73, 149 ->
// 114, 247 -> 210; 28672 x 4096 at 40 / 2048 29.5 -> 25.4, 476 -> 414; 6204 x 2816 at 128 27 -> 14.
#include "iq3s_wide.h"
#include "iq3s_wide_copies.h"

#include "iq3s_dense.h"

namespace {

// A lane's share of half a 32-row weight block (128 of K: two K steps): the record of lane
// (row r32 & 15, q = 2 * half + (lane >> 5)) of the 16-row tile r32 >> 4, whose 16 codes are in
// the order of the dense K operand (mambo_common.h). In the 32 x 32 x 64 MFMA, lane l holds
// column l & 31; operand bytes 0-15 lie in K block 0 and bytes 16-31 in K block 1 of the step
// (their E8M0 scales come from lanes 0-31 and 32-63), half l >> 5 of each. So K step h of the
// record is its codes 8h .. 8h+7 as they are: codes 0-3 are half q & 1 of group 4 * half + h
// and codes 4-7 of group 4 * half + 2 + h, and the activation bytes and scales to match are
// those of the same groups. Layout checked on gfx950 with one-hot operands.
struct WRec {
    uint4 ia;
    uint16_t ib;
    uint2 sg;
    uint8_t sc;
};

template <int kPolicy>
__device__ __forceinline__ WRec load_rec(__amdgpu_buffer_rsrc_t r, uint32_t step, uint32_t o16, uint32_t o8,
                                         uint32_t o2, uint32_t o1, int half)
{
    WRec w;
    const auto ia = __builtin_amdgcn_raw_buffer_load_b128(r, o16 + kTileIdxA + 512u * half, step, kPolicy);
    w.ia = uint4{ia[0], ia[1], ia[2], ia[3]};
    w.ib = __builtin_amdgcn_raw_buffer_load_b16(r, o2 + kTileIdxB + 64u * half, step, kPolicy);
    const auto sg = __builtin_amdgcn_raw_buffer_load_b64(r, o8 + kTileSigns + 256u * half, step, kPolicy);
    w.sg = uint2{sg[0], sg[1]};
    w.sc = __builtin_amdgcn_raw_buffer_load_b8(r, o1 + kTileScales + 32u * half, step, kPolicy);
    return w;
}

// A record being decoded.
struct WState {
    uint32_t s[5];
    uint32_t p[2];
    uint32_t sc; // nibble 2X + H: group of operand half X of K step H
};

// The scale bytes of groups 4 * half .. +3 are those of lanes l & 31 and l | 32: one swap.
__device__ __forceinline__ void begin_rec(WState &st, const WRec &w)
{
    st.s[0] = w.ia.x;
    st.s[1] = w.ia.y;
    st.s[2] = w.ia.z;
    st.s[3] = w.ia.w;
    st.s[4] = (uint32_t)w.ib;
    st.p[0] = w.sg.x;
    st.p[1] = w.sg.y;
    const auto r = __builtin_amdgcn_permlane32_swap((uint32_t)w.sc, (uint32_t)w.sc, false, false);
    st.sc = r[0] | (r[1] << 8);
}

// Decoded operands of one K step.
struct StepOps {
    v8i hi, lo;
};

// Codebook words of codes C0 .. C0+N-1 of K step H of a record.
template <int H, int C0, int N>
__device__ __forceinline__ void fetch_words(const WState &st, const uint8_t *lvl, uint32_t (&lw)[8])
{
    if constexpr (N > 0) {
        lw[C0] = *reinterpret_cast<const uint32_t *>(lvl + code_addr<8 * H + C0>(st.s));
        fetch_words<H, C0 + 1, N - 1>(st, lvl, lw);
    }
}
// Codes C0 .. C0+N-1 of the step from their codebook words.
template <int C0, int N>
__device__ __forceinline__ void finish_words(uint32_t p, const uint32_t (&lw)[8], const uint4 (&tab)[2], StepOps &o)
{
    if constexpr (N > 0) {
        int hi, lo;
        split_word<C0>(lw[C0], p, tab[C0 / 4], hi, lo);
        o.hi[C0] = hi;
        o.lo[C0] = lo;
        finish_words<C0 + 1, N - 1>(p, lw, tab, o);
    }
}

// kPolicy: cache policy of the weight loads, non-temporal where one token tile reads each
// weight once (57344 x 8192 at 128 tokens 0-2%), the default where several do.
template <int MT, int W, int KG, int kPolicy>
__global__ __launch_bounds__(W * KG * 64) __attribute__((amdgpu_waves_per_eu(2))) void gemm_wide_kernel(
    const uint8_t *__restrict__ xv, int64_t ldxv, const uint8_t *__restrict__ xs, int64_t ldxs, int64_t M, GroupArgs ga,
    int B, int bps, int atomic)
{
    constexpr int kRows = 32 * MT;
    constexpr int kVCopies = kRows / 4 / W;
    static_assert(MT % 2 == 0, "the scalings are split over two steps");
    static_assert(kRows / 4 % W == 0 && MT <= W && (W % 4 == 0 || 4 % W == 0), "staging must spread evenly over the waves");
    // the alignments place the tables and scales first, below the 64 KiB that an LDS
    // instruction's offset reaches (above it every read needs its address or-ed together: 38
    // more vector instructions per block, 3-5% of the kernel)
    __shared__ __align__(1024) uint32_t s_lvl[512];
    __shared__ __align__(256) uint4 s_split[16];
    __shared__ __align__(128) uint8_t s_scale0[KG * kRows * 8];
    __shared__ __align__(128) uint8_t s_scale1[KG * kRows * 8];
    __shared__ __align__(16) uint8_t s_vals0[KG * kRows * 256];
    __shared__ __align__(16) uint8_t s_vals1[KG * kRows * 256];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wgwave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wave = wgwave % W, kg = wgwave / W; // wave within its K group
    const int col = lane & 15, r32 = lane & 31, g = lane >> 5;

    const uint8_t *packed = ga.packed[0];
    float *out = ga.out[0];
    int64_t N = ga.n[0], ldo = ga.ldo[0], wg = blockIdx.x;
#pragma unroll
    for (int i = 1; i < kMaxGroup; ++i)
        if (i < ga.count && (int64_t)blockIdx.x >= ga.tile_begin[i]) {
            packed = ga.packed[i];
            out = ga.out[i];
            N = ga.n[i];
            ldo = ga.ldo[i];
            wg = blockIdx.x - ga.tile_begin[i];
        }
    const int64_t tiles = (N + kTileRows - 1) / kTileRows;
    const int64_t m0 = (int64_t)blockIdx.y * kRows;
    const int64_t tile = 2 * (wg * W + wave); // first of this wave's two 16-row tiles
    const __amdgpu_buffer_rsrc_t wt = byte_rsrc(packed + min(tile, tiles - 1) * (int64_t)B * kTileBytes);
    const uint32_t second = (lane & 16) && tile + 1 < tiles ? (uint32_t)B * kTileBytes : 0u;
    const uint32_t rl = (uint32_t)(col + 16 * g);
    const uint32_t o16 = second + 16u * rl, o8 = second + 8u * rl, o2 = second + 2u * rl, o1 = second + rl,
                   od = second + 2u * col;

    // Rows past M read row M-1 (their outputs are never stored), by offsets made once
    // (iq3s_wide_copies.h). The resources end with that row too; nothing depends on it, but with open ones the
    // compiler's code around the stores is slower where N is no multiple of 16 (2286 x 2048 at 1920 tokens
    // 28.0 us and 27.4, 2897 x 1024 at 1536 18.5 and 17.9).
    const auto rows_rsrc = [&](const uint8_t *base, int64_t ld, int row_bytes) {
        const uint64_t bytes = (uint64_t)(M - 1 - m0) * (uint64_t)ld + (uint64_t)row_bytes;
        const uint32_t n = (bytes >> 32) ? 0xFFFFFFFFu : (uint32_t)bytes;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base + m0 * ld), 0,
                                                 __builtin_amdgcn_readfirstlane((int)n), 0x00020000);
    };
    const __amdgpu_buffer_rsrc_t xrows = rows_rsrc(xv, ldxv, B * 256), srows = rows_rsrc(xs, ldxs, B * 8);
    const int last_row = (int)min<int64_t>(M - 1 - m0, kRows - 1);
    const int srow = wave & (MT - 1); // waves past MT repeat a scale copy (the same bytes): no branch
    uint32_t voff[kVCopies];
#pragma unroll
    for (int j = 0; j < kVCopies; ++j)
        voff[j] = wide_value_offset(wave, lane, W, j, last_row, (uint32_t)ldxv);
    const uint32_t soff_stage = wide_scale_offset(srow, lane, last_row, (uint32_t)ldxs);

    const uint32_t a0 = (uint32_t)(kg * kRows * 256) + 256u * r32 + 16u * (uint32_t)(g ^ col);
    const uint32_t soff = (uint32_t)(kg * kRows * 8) + 8u * r32 + 2u * g;
    const uint8_t *lvl = reinterpret_cast<const uint8_t *>(s_lvl);

    float acc[MT][16];
    v16f c[MT];
#pragma unroll
    for (int mt = 0; mt < MT; ++mt)
#pragma unroll
        for (int i = 0; i < 16; ++i)
            acc[mt][i] = c[mt][i] = 0.0f;
    // K group kg takes blocks [b0, end); those from b1 on are a block again with its sums scaled to
    // 2^-128 (an infinite sum must not meet the zero) and a zero d
    const int z0 = blockIdx.z * bps, b1 = min(B, z0 + bps), per = (b1 - z0 + KG - 1) / KG;
    const int b0 = z0 + kg * per, end = b0 + per;
    auto wblock = [&](int b) { return (uint32_t)min(b, b1 - 1) * kTileBytes; };

    auto stage = [&](uint8_t *vals, uint8_t *scl, int b) {
#pragma unroll
        for (int j = 0; j < kVCopies; ++j) {
            const uint32_t vo = voff[j]; // (the host pass drops the kernel with the element as an argument)
            __builtin_amdgcn_raw_ptr_buffer_load_lds(xrows, (lds_ptr)(vals + kg * kRows * 256 + 1024 * (wave + W * j)),
                                                     16, vo, 256u * b, 0, 0);
        }
        __builtin_amdgcn_raw_ptr_buffer_load_lds(srows, (lds_ptr)(scl + kg * kRows * 8 + 256 * srow), 4, soff_stage, 8u * b, 0, 0);
    };

    WRec rec[2];
    uint16_t dh;
    StepOps op[2];
    int bscale = 128;
    float dcur = 0.0f;
    v8i a[2];
    int sc[2];
    uint32_t al = 0, ah = 0;
    // Prologue: the tables' and block b0's copies into LDS, then b0's weights; the barrier waits
    // for the copies only (vector memory completes in issue order).
    {
        const __amdgpu_buffer_rsrc_t gr = byte_rsrc(c_grid.level), tr = byte_rsrc(&c_split.w[0][0]);
        for (int i = wgwave; i < 9; i += W * KG) {
            if (i < 8)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(gr, (lds_ptr)(s_lvl + 64 * i), 4, 4u * lane, 256u * i, 0, 0);
            else
                __builtin_amdgcn_raw_ptr_buffer_load_lds(tr, (lds_ptr)s_split, 4, 4u * lane, 0, 0, 0);
        }
    }
    stage(s_vals0, s_scale0, min(b0, b1 - 1));
    __builtin_amdgcn_sched_barrier(0);
    rec[0] = load_rec<kPolicy>(wt, wblock(b0), o16, o8, o2, o1, 0);
    dh = __builtin_amdgcn_raw_buffer_load_b16(wt, od + kTileD, wblock(b0), kPolicy);
    rec[1] = load_rec<kPolicy>(wt, wblock(b0), o16, o8, o2, o1, 1);
    __builtin_amdgcn_sched_barrier(0);
    __builtin_amdgcn_s_waitcnt(9 | (7 << 4) | (15 << 8)); // vmcnt(9): the weights stay in flight
    __syncthreads();
    {
        WState st;
        begin_rec(st, rec[0]);
        uint32_t lw[8];
        const uint4 tab[2] = {split_entry<0, 0>(s_split, st.sc), split_entry<0, 1>(s_split, st.sc)};
        fetch_words<0, 0, 8>(st, lvl, lw);
        finish_words<0, 8>(st.p[0], lw, tab, op[0]);
    }

    // Activation fragment of sub-tile mt for K step S (= 2r + h): row r32, 16-byte chunks 8r + 2h +
    // g and + 4 at their swizzled slots (chunk c of row i at slot c ^ (i & 15)), and the row's
    // scales of K block g for both h. The chunk addresses are hidden from the compiler, which
    // otherwise or-s the sub-tile's offset into them instead of folding it into the read.
    auto load_frag = [&]<int S>(const uint8_t *vals, const uint8_t *scl, int slot, int mt) {
        constexpr int r = S >> 1, h = S & 1;
        if (mt == 0) {
            al = a0 ^ (16u * (8 * r + 2 * h));
            ah = a0 ^ (16u * (8 * r + 2 * h + 4));
            asm volatile("" : "+v"(al), "+v"(ah));
        }
        const uint4 lo = *reinterpret_cast<const uint4 *>(vals + 8192 * mt + al);
        const uint4 hi = *reinterpret_cast<const uint4 *>(vals + 8192 * mt + ah);
        a[slot] = v8i{(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
        sc[slot] = (int)*reinterpret_cast<const uint16_t *>(scl + 256 * mt + soff + 4 * r);
    };
    auto scale_acc = [&](int mt, int i0, int n) {
#pragma unroll
        for (int i = 0; i < n; ++i) {
            acc[mt][i0 + i] = __builtin_fmaf(c[mt][i0 + i], dcur, acc[mt][i0 + i]);
            asm volatile("" : "+v"(acc[mt][i0 + i]));
        }
    };
    // K step S of the block in buffers vals/scl with operands op[S & 1], while the next step's
    // are decoded into op[(S & 1) ^ 1]. kLast: no block follows.
    auto kstep = [&]<int S, bool kLast>(const uint8_t *vals, const uint8_t *scl, int b) {
        constexpr int h = S & 1;
        constexpr int NS = (S + 1) & 3, nr = NS >> 1, nh = NS & 1;
        // codes fetched per 32-token tile (of the first MT - 1; finished one tile later)
        constexpr int kF = (8 + MT - 2) / (MT - 1);
        constexpr bool kDecode = !(kLast && S == 3);
        const StepOps &cur = op[S & 1];
        StepOps &nxt = op[(S & 1) ^ 1];
        WState st;
        uint4 tab[2];
        uint32_t lw[8];
        [&]<int... I>(std::integer_sequence<int, I...>) {
            (
                [&] {
                    constexpr int mt = I;
                    constexpr int sl = (S * MT + mt) & 1;
                    // the sub-tile whose finished sums are scaled here (step 3: the first half's,
                    // step 0: the second half's of the block before)
                    constexpr int due = S == 3   ? (mt >= MT / 2 ? mt - MT / 2 : -1)
                                        : S == 0 ? (mt < MT / 2 ? mt + MT / 2 : -1)
                                                 : -1;
                    if constexpr (S == 0) {
                        v16f zero;
#pragma unroll
                        for (int i = 0; i < 16; ++i)
                            zero[i] = 0.0f;
                        c[mt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[sl], cur.hi, zero, 0, 0, h, sc[sl], 0,
                                                                                bscale);
                    } else {
                        c[mt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[sl], cur.hi, c[mt], 0, 0, h, sc[sl],
                                                                                0, bscale);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (mt == 0 && kDecode) {
                        begin_rec(st, rec[nr]);
                        tab[0] = split_entry<nh, 0>(s_split, st.sc);
                        tab[1] = split_entry<nh, 1>(s_split, st.sc);
                    }
                    if constexpr (mt + 1 < MT)
                        load_frag.template operator()<S>(vals, scl, sl ^ 1, mt + 1);
                    else if constexpr (S < 3)
                        load_frag.template operator()<(S + 1) & 3>(vals, scl, sl ^ 1, 0);
                    constexpr int f0 = kF * mt, fn = 8 - f0 < kF ? 8 - f0 : kF;
                    if constexpr (mt + 1 < MT && kDecode)
                        fetch_words<nh, f0, fn>(st, lvl, lw);
                    constexpr int d0 = kF * (mt - 1), dn = mt == 0 ? 0 : (8 - d0 < kF ? 8 - d0 : kF);
                    if constexpr (due >= 0)
                        scale_acc(due, 0, 8);
                    if constexpr (mt > 0 && kDecode)
                        finish_words<d0, dn / 2>(st.p[nh], lw, tab, nxt);
                    __builtin_amdgcn_sched_barrier(0);
                    c[mt] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[sl], cur.lo, c[mt], 0, 0, h, sc[sl], 0,
                                                                            bscale);
                    __builtin_amdgcn_sched_barrier(0);
                    if constexpr (due >= 0)
                        scale_acc(due, 8, 8);
                    if constexpr (mt > 0 && kDecode)
                        finish_words<d0 + dn / 2, dn - dn / 2>(st.p[nh], lw, tab, nxt);
                    __builtin_amdgcn_sched_barrier(0);
                }(),
                ...);
        }(std::make_integer_sequence<int, MT>{});
        // (pinned here: the compiler would sink the decode past the barrier, next to its use)
        if constexpr (kDecode)
            asm volatile("" : "+v"(nxt.hi), "+v"(nxt.lo));
        if constexpr (S == 0) {
            dcur = KG == 1 || b < b1 ? half_bits_to_float(dh) : 0.0f;
            asm volatile("" : "+v"(dcur));
        }
        if constexpr (S == 0 && !kLast) {
            rec[0] = load_rec<kPolicy>(wt, wblock(b + 1), o16, o8, o2, o1, 0);
            dh = __builtin_amdgcn_raw_buffer_load_b16(wt, od + kTileD, wblock(b + 1), kPolicy);
        }
        if constexpr (S == 2 && !kLast)
            rec[1] = load_rec<kPolicy>(wt, wblock(b + 1), o16, o8, o2, o1, 1);
        __builtin_amdgcn_sched_barrier(0);
    };

    // A block in buffer CUR while the next one's copies go to buffer NXT: they were issued before
    // the nine loads of its weights, so the barrier's wait leaves those in flight. The loop takes
    // two blocks per pass, so that the buffers are fixed arrays and the compiler can tell the
    // copy's target from the buffer being read; no pass branches in the middle (with a break
    // there the accumulators of both paths cost 70 spilled registers).
#define MAMBO_WIDE_STEPS(CUR, LAST)                                                                                \
    load_frag.template operator()<0>(s_vals##CUR, s_scale##CUR, 0, 0);                                             \
    __builtin_amdgcn_sched_barrier(0);                                                                             \
    if constexpr (KG > 1)                                                                                          \
        bscale = b < b1 ? 128 : 0;                                                                                 \
    kstep.template operator()<0, LAST>(s_vals##CUR, s_scale##CUR, b);                                              \
    kstep.template operator()<1, LAST>(s_vals##CUR, s_scale##CUR, b);                                              \
    kstep.template operator()<2, LAST>(s_vals##CUR, s_scale##CUR, b);                                              \
    kstep.template operator()<3, LAST>(s_vals##CUR, s_scale##CUR, b)
#define MAMBO_WIDE_BLOCK(CUR, NXT)                                                                                 \
    do {                                                                                                           \
        stage(s_vals##NXT, s_scale##NXT, min(b + 1, b1 - 1));                                                      \
        MAMBO_WIDE_STEPS(CUR, false);                                                                              \
        __builtin_amdgcn_s_waitcnt(9 | (7 << 4) | (15 << 8));                                                      \
        __syncthreads();                                                                                           \
    } while (0)
    int b = b0;
    for (; b + 1 < end; ++b) {
        MAMBO_WIDE_BLOCK(0, 1);
        ++b;
        MAMBO_WIDE_BLOCK(1, 0);
    }
    if (b < end) {
        MAMBO_WIDE_STEPS(0, true);
    }
#undef MAMBO_WIDE_BLOCK
#undef MAMBO_WIDE_STEPS

    const int64_t n = tile * kTileRows + r32;
#pragma unroll
    for (int mt = MT / 2; mt < MT; ++mt) // the last block's sums that no step 0 followed
        scale_acc(mt, 0, 16);
    if constexpr (KG > 1) {
        // the other K groups' sums over the first buffer (every wave has left it), added by the first
        static_assert((KG - 1) * W * MT * 4096 <= KG * kRows * 256, "one buffer holds the groups' sums");
        float4 *red = reinterpret_cast<float4 *>(s_vals0) + wave * (MT * 4 * 64) + lane;
        __syncthreads();
        if (kg)
#pragma unroll
            for (int j = 0; j < 4 * MT; ++j)
                red[(kg - 1) * (W * MT * 4 * 64) + 64 * j] =
                    make_float4(acc[j / 4][4 * (j & 3)], acc[j / 4][4 * (j & 3) + 1], acc[j / 4][4 * (j & 3) + 2],
                                acc[j / 4][4 * (j & 3) + 3]);
        __syncthreads();
        if (kg)
            return;
#pragma unroll
        for (int k = 0; k < KG - 1; ++k)
#pragma unroll
            for (int j = 0; j < 4 * MT; ++j) {
                const float4 v = red[k * (W * MT * 4 * 64) + 64 * j];
                acc[j / 4][4 * (j & 3)] += v.x;
                acc[j / 4][4 * (j & 3) + 1] += v.y;
                acc[j / 4][4 * (j & 3) + 2] += v.z;
                acc[j / 4][4 * (j & 3) + 3] += v.w;
            }
    }
    if (n < N) {
#pragma unroll
        for (int mt = 0; mt < MT; ++mt)
#pragma unroll
            for (int i = 0; i < 16; ++i) {
                const int64_t m = m0 + 32 * mt + 8 * (i >> 2) + 4 * g + (i & 3);
                if (m < M) {
                    if (atomic)
                        atomicAdd(out + m * ldo + n, acc[mt][i]);
                    else
                        __builtin_nontemporal_store(acc[mt][i], out + m * ldo + n);
                }
            }
    }
}

int64_t cdiv(int64_t a, int64_t b) { return (a + b - 1) / b; }

// The kernel's shapes, with what one workgroup of K blocks takes on a CU that holds 1, 2, ..
// of them (as many as its registers allow): microseconds per launch round and per block of a
// K group.
struct WideShape {
    int mt, waves, kg, resident;
    double round, block[3];
};
constexpr WideShape kWideShapes[] = {{2, 4, 1, 3, 0.37, {1.26, 1.82, 2.49}},
                                     {2, 4, 2, 1, 1.6, {1.82, 0.0, 0.0}},
                                     {4, 4, 1, 2, 2.2, {1.64, 2.60, 0.0}},
                                     {2, 2, 4, 1, 1.6, {2.3, 0.0, 0.0}},
                                     {4, 4, 2, 1, 2.7, {2.43, 0.0, 0.0}},
                                     {4, 8, 1, 1, 1.35, {2.45, 0.0, 0.0}}};
constexpr int kWideSplits[] = {1, 2, 3, 4, 6, 8, 12, 16};
constexpr int64_t kCUs = 256;

// Microseconds of a launch of `wgs` workgroups of `b` K blocks each writing `mb` MB of outputs,
// K in `splits` slices: the busiest CU's rounds, the output stores, and with several slices
// the zero fill and the f32 atomics (~1.5 TB/s alone). One K group fitted to 12000 launches (42
// shapes of 128 to 57344 rows, K 512 to 28672, 33 to 4096 tokens, each at every shape and split;
// rms error 6%), two to 250, four to the launches named above only; the plan it picks is 1% behind the
// fastest measured one on average over 66 shapes and token counts (most: 8%, 8192 x 4096 at 64 tokens).
// Large launches at 128 tokens lie outside that error: 57344 x 8192 takes 102 to 122 us where it says
// 91, 8192 x 28672 62 to 73 where it says 56.
double wide_time(const WideShape &w, int64_t wgs, int64_t b, int splits, double mb)
{
    b = cdiv(b, w.kg);
    const int64_t per = cdiv(wgs, kCUs), full = per / w.resident, rem = per % w.resident;
    double t = 3.62 + w.round * (double)(full + (rem ? 1 : 0)) +
               (double)b * ((double)full * w.block[w.resident - 1] + (rem ? w.block[rem - 1] : 0.0)) + 0.25 * mb;
    if (splits > 1)
        t += 1.48 + 0.8 * mb * splits;
    return t;
}

int64_t wide_workgroups(const mambo_projection *proj, int count, int waves)
{
    int64_t wgs = 0;
    for (int g = 0; g < count; ++g)
        wgs += cdiv(cdiv(proj[g].n, 32), waves);
    return wgs;
}

template <int MT, int W, int KG>
void launch_wide(const WidePlan &p, dim3 grid, hipStream_t stream, const uint8_t *xv, int64_t ldxv, const uint8_t *xs,
                 int64_t ldxs, int64_t m, const GroupArgs &ga, int blocks)
{
    if (grid.y > 1)
        MAMBO_LAUNCH((gemm_wide_kernel<MT, W, KG, 0>), grid, dim3(W * KG * 64), 0, stream, xv, ldxv, xs, ldxs, m,
                     ga, blocks, p.bps, p.splits > 1);
    else
        MAMBO_LAUNCH((gemm_wide_kernel<MT, W, KG, kStreamPolicy>), grid, dim3(W * KG * 64), 0, stream, xv, ldxv, xs,
                     ldxs, m, ga, blocks, p.bps, p.splits > 1);
}

} // namespace

bool mambo_wide_plan(int64_t m, const mambo_projection *proj, int count, int64_t blocks, int64_t ldxv,
                     const uint8_t *xs, int64_t ldxs, const mambo_gemm_config &other, WidePlan *plan)
{
    // what the kernel's addressing assumes: scale rows copied as dwords (8-byte aligned, as the
    // tiled kernel asks), a token tile's values and scales within 32-bit offsets, grid limits
    if (m < 33 || blocks < 4 || (uintptr_t)xs % 8 != 0 || ldxs % 8 != 0 ||
        256 * ldxv + blocks * 256 >= ((int64_t)1 << 32) || 256 * ldxs + blocks * 8 >= ((int64_t)1 << 32) ||
        cdiv(m, 64) > 65535)
        return false;
    int64_t n = 0;
    for (int g = 0; g < count; ++g)
        n += proj[g].n;
    // Where it is the faster kernel (672 shapes and token counts, each at the fastest plan of
    // either side): wherever the other plan splits K (64 tokens and more; 1-35%), so that sums
    // that were in a fixed order stay so; against an unsplit tiled plan from 9 K blocks on
    // (4-35%; on 4 and 8 blocks launches of 7-17 us, the 64-token tiles are 1-12% ahead) or
    // where 128 x 128 tiles give every CU one, but on 4 blocks not where the other's 64 x 128 tiles are
    // a single round of two per CU (8192 x 1024 at 400 tokens 13.1 and 14.7); against the dense kernel (which decodes a weight
    // once per 32 tokens) where 64 x 128 tiles take 80 CUs (us at 40 tokens: 28672
    // x 4096 46 against 25, 14336 x 8192 42 and 29, 10240 x 4096 22 and 16; 8192 x 4096,
    // 64 workgroups, 16.3 and 19.9), or where its waves do not divide few K blocks and it takes 64
    // rows a workgroup (measured at 11 blocks, K = 2816, alone: 6144 rows 23 against 16; with 32 rows,
    // 4096, 13.4 and 16.2; the small tiles take most of these launches from either).
    const bool split = blocks > cdiv(blocks, other.split_k);
    const int64_t row_wgs = wide_workgroups(proj, count, 4);
    const bool fills = row_wgs * cdiv(m, 128) >= kCUs;
    if (!split) {
        const int64_t wgs64 = row_wgs * cdiv(m, 64);
        if (other.kernel == MAMBO_GEMM_DENSE ? !(wgs64 >= 80 || (blocks % 4 != 0 && blocks <= 11 && other.tile_n >= 64))
                                             : !(blocks >= 9 || fills) ||
                                                   (blocks == 4 && other.tile_m == 64 && wgs64 <= 2 * kCUs))
            return false;
    }
    const double mb = 4e-6 * (double)m * (double)n;
    double best = 0.0;
    for (const WideShape &w : kWideShapes) {
        // 64-token tiles decode each weight twice as often: only while 128-token ones leave CUs
        // idle, or where they pad away most of the last tile
        if (w.mt == 2 && fills && (m % 128 == 0 || m % 128 > 64))
            continue;
        const int64_t wgs = wide_workgroups(proj, count, w.waves) * cdiv(m, 32 * w.mt);
        // on fewer than 9 blocks eight waves only where four would just pass one workgroup per CU (13208 x
        // 1536 at 384 tokens, 156 workgroups, 24.8 us and 25.9 with four); else four of them on 128 x 128
        // tiles are 4-17% faster (7383 x 1280 at 959, 232, 30.6 and 25.6; 22818 x 2048 at 921, 720,
        // 112 and 102)
        if (w.waves == 8 && blocks < 9 && wgs > kCUs * 11 / 16)
            continue;
        if (wgs > 0x7FFFFFFF)
            return false;
        for (const int s : kWideSplits) {
            const int64_t bps = cdiv(blocks, s);
            const int splits = (int)cdiv(blocks, bps);
            if (s > 1 && (!split || wgs * s > 1100 || blocks < 2 * s))
                continue;
            // two K groups only while every CU has at most one workgroup: beyond, other workgroups
            // fill the waits (28672 x 4096 at 1024 tokens 207 us with one group, 230 with two)
            if (w.kg > 1 && wgs * splits > kCUs)
                continue;
            const double t = wide_time(w, wgs * splits, bps, splits, mb);
            if (best == 0.0 || t < best) {
                best = t;
                *plan = {w.mt, w.waves, w.kg, splits, (int)bps, t};
            }
        }
    }
    return true;
}

int mambo_wide_launch(const WidePlan &p, const uint8_t *xv, int64_t ldxv, const uint8_t *xs, int64_t ldxs, int64_t m,
                      const mambo_projection *proj, int count, int64_t blocks, hipStream_t stream)
{
    GroupArgs ga = {};
    ga.count = count;
    int64_t wgs = 0;
    for (int g = 0; g < count; ++g) {
        ga.packed[g] = proj[g].packed;
        ga.out[g] = proj[g].out;
        ga.n[g] = proj[g].n;
        ga.ldo[g] = proj[g].ldo;
        ga.tile_begin[g] = wgs;
        wgs += cdiv(cdiv(proj[g].n, 32), p.waves);
    }
    const dim3 grid((unsigned)wgs, (unsigned)cdiv(m, 32 * p.mt), (unsigned)p.splits);
    const auto is = [&](int mt, int waves, int kg) { return p.mt == mt && p.waves == waves && p.kg == kg; };
#define MAMBO_WIDE_SHAPE(MT, W, KG)                                                                                \
    if (is(MT, W, KG))                                                                                             \
    launch_wide<MT, W, KG>(p, grid, stream, xv, ldxv, xs, ldxs, m, ga, (int)blocks)
    MAMBO_WIDE_SHAPE(2, 2, 4);
    MAMBO_WIDE_SHAPE(2, 4, 1);
    MAMBO_WIDE_SHAPE(2, 4, 2);
    MAMBO_WIDE_SHAPE(4, 4, 1);
    MAMBO_WIDE_SHAPE(4, 4, 2);
    MAMBO_WIDE_SHAPE(4, 8, 1);
#undef MAMBO_WIDE_SHAPE
    return mambo_check_launch("iq3s_fp8_matmul (wide)");
}
