// IQ3_S weight preparation and the standalone decoder.
//
// prepare: raw GGUF blocks u8[N, B, 110] (any strides and alignment) -> the reference's
// SoA fields (iq3_s_weight.py:25-54: d [B,N], qs [B,N,16], qh [B,N,4], signs [B,N,8],
// scales [B,N]) and/or the private tile layout read by the projection kernels (layout in
// mambo_common.h). Contiguous blocks (what a GGUF tensor is) go through prepare_rows_kernel,
// any other strides through prepare_kernel (one 16-row x 1-block tile per workgroup, bytes).
// pack reads the fields where they are (pack_fields_kernel).
//
// dequant: SoA fields -> E4M3 bits [N, K] + f32 group scales [N, K/32], the FP8 form of
// decode_iq3_s_blocks (iq3_s_fp8.py:202-222): bits = iq3_s_fp8_table[qs | qh<<8] with
// the sign bits of the group ORed into each byte's bit 7 (iq3_s_fp8.py:105-166), scale
// = f32(d) * (1 + 2*nibble) (iq3_s_fp8.py:186-199).
#include "mambo_common.h"

namespace {

__constant__ GridTables c_grid = kGridTables;

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4), aligned(4)));

// Stores past the caches, for whole lines that nothing here reads again.
template <class T>
__device__ __forceinline__ void put(T v, void *p)
{
    __builtin_nontemporal_store(v, reinterpret_cast<T *>(p));
}

struct RawSrc {
    const uint8_t *raw;
    int64_t sn, sb, sbyte;
};

struct SoaSrc {
    const uint16_t *d;
    const uint32_t *qs;
    const uint16_t *qh;
    const int32_t *signs;
    const uint32_t *scales;
};

// Outputs of prepare (each may be null).
struct PrepareOut {
    uint16_t *d;
    uint32_t *qs;
    uint16_t *qh;
    int32_t *signs;
    uint32_t *scales;
    uint8_t *packed;
};

// Stage tile (t, b) as 16 rows x 110 bytes in GGUF block order; rows >= n are zero.
__device__ void stage(const RawSrc &s, int64_t n, int64_t t, int64_t b, uint8_t (*blk)[112])
{
    for (int i = threadIdx.x; i < kTileRows * kIq3sBlockBytes; i += blockDim.x) {
        int r = i / kIq3sBlockBytes, c = i % kIq3sBlockBytes;
        int64_t row = t * kTileRows + r;
        blk[r][c] = row < n ? s.raw[row * s.sn + b * s.sb + c * s.sbyte] : 0;
    }
}

__device__ __forceinline__ uint32_t le32(const uint8_t *p)
{
    return (uint32_t)p[0] | ((uint32_t)p[1] << 8) | ((uint32_t)p[2] << 16) | ((uint32_t)p[3] << 24);
}

// What lane l = r + 16q of a tile-block stores (tile layout in mambo_common.h), from its row's
// block. Slots 8h + 4X + k (k = 0..3) hold the four consecutive codes of half q & 1 of weight
// group g = tile_group(2X + (q >> 1), h), so each (h, X) takes one word of qs, one byte of qh
// and 16 sign bits, and fills 36 bits of the index stream. src gives those pieces of a row:
// qs_word(g, half), qh_byte(g), sign_half(g, half), scale_byte(q), d_bits().
template <class Src>
__device__ __forceinline__ void pack_lane(const Src &src, int l, uint8_t *__restrict__ tile)
{
    const int r = l & 15, q = l >> 4;
    uint64_t idx[4];
    uint32_t sign[2] = {0u, 0u};
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int x = 0; x < 2; ++x) {
            const int g = tile_group(2 * x + (q >> 1), h);
            const uint32_t w = src.qs_word(g, q & 1);
            const uint32_t hi = (uint32_t)src.qh_byte(g) >> (4 * (q & 1));
            uint64_t v = 0;
#pragma unroll
            for (int k = 0; k < 4; ++k)
                v |= (uint64_t)(((w >> (8 * k)) & 0xFFu) | (((hi >> k) & 1u) << 8)) << (9 * k);
            idx[2 * h + x] = v;
            // transpose the codes' sign nibbles (bit 4k + j -> bit 4j + k), then nibble j to bit 8j
            uint32_t t = src.sign_half(g, q & 1);
            uint32_t d = (t ^ (t >> 3)) & 0x0A0Au;
            t ^= d ^ (d << 3);
            d = (t ^ (t >> 6)) & 0x00CCu;
            t ^= d ^ (d << 6);
            t = (t & 0xFu) | ((t & 0xF0u) << 4) | ((t & 0xF00u) << 8) | ((t & 0xF000u) << 12);
            sign[h] |= t << (4 * x);
        }
    // four 36-bit pieces to 144 bits
    const uint64_t lo = idx[0] | (idx[1] << 36), hi = (idx[1] >> 28) | (idx[2] << 8) | (idx[3] << 44);
    put(u32x4{(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)}, tile + kTileIdxA + 16 * l);
    *reinterpret_cast<uint16_t *>(tile + kTileIdxB + 2 * l) = (uint16_t)(idx[3] >> 20);
    put(u32x2{sign[0], sign[1]}, tile + kTileSigns + 8 * l);
    tile[kTileScales + l] = src.scale_byte(q);
    if (q == 0)
        *reinterpret_cast<uint16_t *>(tile + kTileD + 2 * r) = src.d_bits();
}

// A row's block in LDS, as GGUF bytes.
struct LdsBlock {
    const uint8_t *o;
    __device__ uint32_t qs_word(int g, int half) const { return le32(o + 2 + 8 * g + 4 * half); }
    __device__ uint8_t qh_byte(int g) const { return o[66 + g]; }
    __device__ uint32_t sign_half(int g, int half) const
    {
        return (uint32_t)o[74 + 4 * g + 2 * half] | ((uint32_t)o[75 + 4 * g + 2 * half] << 8);
    }
    __device__ uint8_t scale_byte(int q) const { return o[106 + q]; }
    __device__ uint16_t d_bits() const { return (uint16_t)(o[0] | (o[1] << 8)); }
};

__global__ __launch_bounds__(256) void prepare_kernel(RawSrc src, int64_t n, int64_t blocks, PrepareOut out)
{
    __shared__ uint8_t blk[kTileRows][112];
    const int64_t t = blockIdx.x;
    for (int64_t b = blockIdx.y; b < blocks; b += gridDim.y) {
        __syncthreads();
        stage(src, n, t, b, blk);
        __syncthreads();
        const int i = threadIdx.x;
        const int r = i >> 4, w = i & 15; // 16 rows x 16 words
        const int64_t row = t * kTileRows + r;
        if (row < n) {
            const int64_t e = b * n + row;
            const uint8_t *o = blk[r];
            if (out.qs)
                out.qs[e * 16 + w] = le32(o + 2 + 4 * w);
            if (out.signs && w < 8)
                out.signs[e * 8 + w] = (int32_t)le32(o + 74 + 4 * w);
            if (out.qh && w < 4)
                out.qh[e * 4 + w] = (uint16_t)(o[66 + 2 * w] | (o[67 + 2 * w] << 8));
            if (w == 0) {
                if (out.d)
                    out.d[e] = (uint16_t)(o[0] | (o[1] << 8));
                if (out.scales)
                    out.scales[e] = le32(o + 106);
            }
        }
        if (out.packed && i < 64)
            pack_lane(LdsBlock{blk[i & 15]}, i, out.packed + (t * blocks + b) * (int64_t)kTileBytes);
    }
}

// Contiguous blocks, of any alignment. A workgroup takes 64 rows x 4 blocks: 440 contiguous bytes
// of each row go to LDS eight bytes a lane, and every field and tile is stored from there in
// 16-, 8-, 4- and 2-byte pieces. Bound by memory (110 bytes of blocks in, 110 or 220 out), and by
// the latency of one workgroup's load-then-store, which 16 loads in flight per wave and four
// workgroups per CU hide: 64 rows so that d and scales are stored in lines of 128 and 256 bytes
// (a tile per workgroup wrote 32 and 64 of them, from different XCDs), four blocks so that the
// lines which neighbouring segments share are a fourth of all. 28672 x 4096, fields and tiles:
// 106 us a tile per workgroup -> 44 us, two blocks 56, one 80, 96 registers for a fifth workgroup per
// CU (13 spilled) 46. The fields and a tile's index words and signs are stored nontemporal (nothing
// here reads them again): 28672 x 4096 44 -> 29 us (5.3 TB/s; a copy moves 4.8), 4096 x 14336 24 ->
// 17, 8192 x 28672 87 -> 58; tiles alone 25.6 -> 23.7, 15.1 -> 14.5, 68 -> 48. With the tile's
// small pieces (32 to 128 bytes) nontemporal too 28672 x 4096 takes 32.
constexpr int kPrepRows = 64, kPrepBlocks = 4;
constexpr int kPrepPitch = (kPrepBlocks * kIq3sBlockBytes + 7) / 8 * 2 + 1; // words; odd: rows in all banks

// A row's block in the word image: the block starts at byte 110j, two bytes off a word for odd
// j, and its words are cut out of two neighbours.
struct ImageBlock {
    const uint32_t *w; // the row's words
    int at;            // byte of the block's start
    __device__ uint32_t word(int byte) const
    {
        const int p = at + byte;
        return __builtin_amdgcn_alignbyte(w[(p >> 2) + 1], w[p >> 2], (uint32_t)p & 3u);
    }
    __device__ uint8_t byte(int b) const { return reinterpret_cast<const uint8_t *>(w)[at + b]; }
    __device__ uint32_t half(int b) const // b is even, as at is
    {
        return *reinterpret_cast<const uint16_t *>(reinterpret_cast<const uint8_t *>(w) + at + b);
    }
    __device__ uint32_t qs_word(int g, int h) const { return word(2 + 8 * g + 4 * h); }
    __device__ uint8_t qh_byte(int g) const { return byte(66 + g); }
    __device__ uint32_t sign_half(int g, int h) const { return half(74 + 4 * g + 2 * h); }
    __device__ uint8_t scale_byte(int q) const { return byte(106 + q); }
    __device__ uint16_t d_bits() const { return (uint16_t)half(0); }
};

__global__ __launch_bounds__(256) void prepare_rows_kernel(const uint8_t *__restrict__ raw, int64_t row_bytes,
                                                           int64_t n, int64_t blocks, PrepareOut out)
{
    __shared__ uint32_t img[kPrepRows * kPrepPitch + 1];
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t row0 = (int64_t)blockIdx.x * kPrepRows;
    for (int64_t b0 = (int64_t)blockIdx.y * kPrepBlocks; b0 < blocks; b0 += (int64_t)gridDim.y * kPrepBlocks) {
        const int nb = (int)min<int64_t>(kPrepBlocks, blocks - b0);
        const int bytes = nb * kIq3sBlockBytes;
        __syncthreads();
        if (8 * lane < bytes) {
            // a row per load of the wave, all of them in flight together; the last eight bytes of
            // the segment are shifted down to where the lane's place is
            const int at = min(8 * lane, bytes - 8), shift = 8 * (8 * lane - at);
#pragma unroll
            for (int i = 0; i < kPrepRows / 4; ++i) {
                const int r = 4 * i + wave;
                uint64_t v;
                __builtin_memcpy(&v, raw + min(row0 + r, n - 1) * row_bytes + b0 * kIq3sBlockBytes + at, 8);
                v = row0 + r < n ? v >> shift : 0; // rows past the weight are zero
                img[r * kPrepPitch + 2 * lane] = (uint32_t)v;
                img[r * kPrepPitch + 2 * lane + 1] = (uint32_t)(v >> 32);
            }
        }
        __syncthreads();
        const auto block = [&](int r, int j) { return ImageBlock{img + r * kPrepPitch, j * kIq3sBlockBytes}; };
        if (out.qs)
            for (int j = 0; j < nb; ++j) { // 64 rows x 4 chunks of 16 bytes
                const int r = tid >> 2, c = tid & 3;
                if (row0 + r < n) {
                    const ImageBlock o = block(r, j);
                    put(u32x4{o.word(2 + 16 * c), o.word(6 + 16 * c), o.word(10 + 16 * c), o.word(14 + 16 * c)},
                        out.qs + ((b0 + j) * n + row0 + r) * 16 + 4 * c);
                }
            }
        if (out.signs)
            for (int j = tid >> 7; j < nb; j += 2) { // 64 rows x 2 chunks
                const int r = (tid & 127) >> 1, c = tid & 1;
                if (row0 + r < n) {
                    const ImageBlock o = block(r, j);
                    put(u32x4{o.word(74 + 16 * c), o.word(78 + 16 * c), o.word(82 + 16 * c), o.word(86 + 16 * c)},
                        out.signs + ((b0 + j) * n + row0 + r) * 8 + 4 * c);
                }
            }
        if (wave < nb && row0 + lane < n) { // one block of every row per wave
            const ImageBlock o = block(lane, wave);
            const int64_t e = (b0 + wave) * n + row0 + lane;
            if (out.qh)
                put(u32x2{o.word(66), o.word(70)}, out.qh + e * 4);
            if (out.scales)
                put(o.half(106) | (o.half(108) << 16), out.scales + e);
            if (out.d)
                put(o.d_bits(), out.d + e);
        }
        const int64_t t = row0 / kTileRows + wave; // one 16-row tile per wave
        if (out.packed && t * kTileRows < n)
            for (int j = 0; j < nb; ++j)
                pack_lane(block(wave * kTileRows + (lane & 15), j), lane,
                          out.packed + (t * blocks + b0 + j) * (int64_t)kTileBytes);
    }
}

// A row's block in the SoA fields; rows past the weight are zero.
struct FieldBlock {
    SoaSrc s;
    int64_t e; // b * n + row
    bool ok;
    __device__ uint32_t qs_word(int g, int half) const { return ok ? s.qs[e * 16 + 2 * g + half] : 0u; }
    __device__ uint8_t qh_byte(int g) const
    {
        return ok ? reinterpret_cast<const uint8_t *>(s.qh)[e * 8 + g] : (uint8_t)0;
    }
    __device__ uint32_t sign_half(int g, int half) const
    {
        return ok ? reinterpret_cast<const uint16_t *>(s.signs)[e * 16 + 2 * g + half] : 0u;
    }
    __device__ uint8_t scale_byte(int q) const { return ok ? (uint8_t)(s.scales[e] >> (8 * q)) : (uint8_t)0; }
    __device__ uint16_t d_bits() const { return ok ? s.d[e] : (uint16_t)0; }
};

// Fields to tiles: one wave per tile-block, reading its 16 rows' fields (contiguous runs of 1 KiB,
// 512, 128, 64 and 32 bytes) straight into the lanes that hold them: 28672 x 4096 88 -> 34 us.
__global__ __launch_bounds__(256) void pack_fields_kernel(SoaSrc src, int64_t n, int64_t blocks, int64_t tiles,
                                                          uint8_t *__restrict__ packed)
{
    const int lane = threadIdx.x & 63;
    const int64_t t = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
    if (t >= tiles)
        return;
    const int64_t row = t * kTileRows + (lane & 15);
    for (int64_t b = blockIdx.y; b < blocks; b += gridDim.y)
        pack_lane(FieldBlock{src, b * n + row, row < n}, lane, packed + (t * blocks + b) * (int64_t)kTileBytes);
}

// Rows x Blocks per workgroup, 16 values (half a weight group) per thread, 16 rows and block.
// Memory-bound (110 bytes in, 288 out per block), so what counts is whole lines: a store of the
// wave covers 1 KiB of values without holes (a thread with the 32 values of a group stored every
// second 16 bytes, twice), the scales of a row leave in one piece of up to 128 bytes, and a
// field of a block is read in runs of Rows rows (2 KiB of qs for 32). With whole lines the nontemporal
// hint pays: nothing written is read here again. Workgroups next to each other take blocks of the same rows.
// Thread per group -> halves -> halves, nontemporal (us), 32 x 4: 4096 x 14336 30.7 -> 22.2 -> 15.2 (6.0 TB/s; a
// copy moves 4.8), 28672 x 4096 57 -> 40 -> 28, 8192 x 28672 107 -> 79 -> 54, 4096 x 4096 7.2 -> 6.4 ->
// 5.8. Rows before blocks in the launch 1-6% slower at 4096 columns, 16 x 8 the same,
// 64 x 4 up to 25% slower.
template <int Rows, int Blocks>
__global__ __launch_bounds__(256) void dequant_kernel(const uint16_t *__restrict__ d, const uint32_t *__restrict__ qs,
                                                      const uint16_t *__restrict__ qh,
                                                      const int32_t *__restrict__ signs,
                                                      const uint32_t *__restrict__ scales, int64_t n, int64_t blocks,
                                                      uint32_t groups, uint8_t *__restrict__ values,
                                                      float *__restrict__ out_scales)
{
    __shared__ uint32_t lut[512];
    constexpr int kPasses = Rows / 16, kPieces = 2 * Blocks; // kPieces: four scales each, of a row
    static_assert(Rows % 16 == 0 && Rows * kPieces <= 256, "a thread writes four scales at most");
    const int tid = threadIdx.x, u = tid & 15; // u: half of a group of the thread's row
    for (int i = tid; i < 512; i += 256)
        lut[i] = c_grid.fp8[i];
    const int64_t row0 = (int64_t)(blockIdx.x / groups) * Rows;
    const int64_t b0 = (int64_t)(blockIdx.x % groups) * Blocks;
    // all loads first; past the weight the last block and row again
    const auto element = [&](int row, int j) { return min(b0 + j, blocks - 1) * n + min(row0 + row, n - 1); };
    uint32_t q[kPasses][Blocks], hb[kPasses][Blocks], sw[kPasses][Blocks];
#pragma unroll
    for (int p = 0; p < kPasses; ++p)
#pragma unroll
        for (int j = 0; j < Blocks; ++j) {
            const int64_t e = element(16 * p + (tid >> 4), j);
            q[p][j] = qs[e * 16 + u];
            hb[p][j] = (uint32_t)reinterpret_cast<const uint8_t *>(qh)[e * 8 + (u >> 1)] >> (4 * (u & 1));
            sw[p][j] = reinterpret_cast<const uint16_t *>(signs)[e * 16 + u];
        }
    // scales: half tid & 1 of block tid / 2 of row tid / kPieces
    const int srow = tid / kPieces, sblock = tid % kPieces >> 1;
    const int64_t es = element(srow, sblock);
    const uint32_t sc = scales[es] >> (16 * (tid & 1));
    const float df = half_bits_to_float(d[es]);
    __syncthreads();
#pragma unroll
    for (int p = 0; p < kPasses; ++p)
#pragma unroll
        for (int j = 0; j < Blocks; ++j) {
            u32x4 out;
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                const uint32_t idx = ((q[p][j] >> (8 * c)) & 0xFFu) | (((hb[p][j] >> c) & 1u) << 8);
                const uint32_t nib = (sw[p][j] >> (4 * c)) & 15u;
                out[c] = lut[idx] | ((nib * 0x00204081u & 0x01010101u) << 7);
            }
            const int64_t row = row0 + 16 * p + (tid >> 4), b = b0 + j;
            if (row < n && b < blocks)
                __builtin_nontemporal_store(out, reinterpret_cast<u32x4 *>(values + (row * blocks + b) * 256) + u);
        }
    const int64_t row = row0 + srow, b = b0 + sblock;
    if (srow < Rows && row < n && b < blocks) {
        f32x4 out;
#pragma unroll
        for (int i = 0; i < 4; ++i)
            out[i] = df * (float)(1u + 2u * ((sc >> (4 * i)) & 15u));
        *reinterpret_cast<f32x4 *>(out_scales + (row * blocks + b) * 8 + 4 * (tid & 1)) = out;
    }
}

template <int Rows, int Blocks>
int launch_dequant(const uint16_t *d, const uint32_t *qs, const uint16_t *qh, const int32_t *signs,
                   const uint32_t *scales, int64_t n, int64_t blocks, uint8_t *values, float *out_scales,
                   hipStream_t stream)
{
    const int64_t rows = (n + Rows - 1) / Rows, groups = (blocks + Blocks - 1) / Blocks;
    MAMBO_REQUIRE(rows <= 0x7FFFFFFF / groups, MAMBO_ERR_VALUE, "weight too large");
    MAMBO_LAUNCH((dequant_kernel<Rows, Blocks>), dim3((unsigned)(rows * groups)), dim3(256), 0, stream, d, qs, qh,
                 signs, scales, n, blocks, (uint32_t)groups, values, out_scales);
    return mambo_check_launch("iq3s_dequant");
}

} // namespace

extern "C" int64_t mambo_iq3s_packed_bytes(int64_t n, int64_t blocks)
{
    if (n < 1 || blocks < 1)
        return 0;
    return ((n + kTileRows - 1) / kTileRows) * blocks * (int64_t)kTileBytes;
}

extern "C" int mambo_iq3s_prepare(const uint8_t *raw, int64_t n, int64_t blocks, int64_t stride_n,
                                  int64_t stride_b, int64_t stride_byte, uint16_t *d, uint32_t *qs,
                                  uint16_t *qh, int32_t *signs, uint32_t *scales, uint8_t *packed,
                                  mambo_stream_t stream)
{
    MAMBO_REQUIRE(raw != nullptr, MAMBO_ERR_VALUE, "raw must not be NULL");
    MAMBO_REQUIRE(n >= 1 && blocks >= 1, MAMBO_ERR_VALUE, "IQ3_S weight must have positive N and K");
    MAMBO_REQUIRE(d || qs || qh || signs || scales || packed, MAMBO_ERR_VALUE, "no output requested");
    MAMBO_REQUIRE(((uintptr_t)qs % 4 == 0) && ((uintptr_t)signs % 4 == 0) && ((uintptr_t)scales % 4 == 0) &&
                      ((uintptr_t)d % 2 == 0) && ((uintptr_t)qh % 2 == 0) && ((uintptr_t)packed % 16 == 0),
                  MAMBO_ERR_VALUE, "SoA fields must be naturally aligned and packed 16-byte aligned");
    const PrepareOut out{d, qs, qh, signs, scales, packed};
    const int64_t tiles = (n + kTileRows - 1) / kTileRows;
    MAMBO_REQUIRE(tiles <= 0x7FFFFFFF, MAMBO_ERR_VALUE, "N too large");
    // Contiguous blocks, fields that take the vector stores, and work for three quarters of the
    // 256 CUs: fields and tiles of 4096 x 4096 (256 workgroups) take 11.5 us here and 13.4 us a
    // tile per workgroup, those of 1024 x 8192 or 2048 x 4096 (128) 8.1 and 7.5. With one to three
    // blocks a row a workgroup has that share of its work: 19473 x 256 (305) 9.1 and 7.3, 12288 x
    // 512 (192) 8.9 and 7.6, 19473 x 512 (305) 10.3 and 11.0, 57344 x 256 (896) 10.6 and 13.1.
    const int64_t row_groups = (n + kPrepRows - 1) / kPrepRows, groups = (blocks + kPrepBlocks - 1) / kPrepBlocks;
    if (stride_byte == 1 && stride_b == kIq3sBlockBytes && row_groups * groups >= 192 && row_groups * blocks >= 600 &&
        (uintptr_t)qs % 16 == 0 && (uintptr_t)signs % 16 == 0 && (uintptr_t)qh % 8 == 0) {
        const dim3 grid((unsigned)row_groups, (unsigned)(groups < 65535 ? groups : 65535));
        MAMBO_LAUNCH(prepare_rows_kernel, grid, dim3(256), 0, (hipStream_t)stream, raw, stride_n, n, blocks, out);
    } else {
        const dim3 grid((unsigned)tiles, (unsigned)(blocks < 65535 ? blocks : 65535));
        MAMBO_LAUNCH(prepare_kernel, grid, dim3(256), 0, (hipStream_t)stream,
                     RawSrc{raw, stride_n, stride_b, stride_byte}, n, blocks, out);
    }
    return mambo_check_launch("iq3s_prepare");
}

extern "C" int mambo_iq3s_pack(const uint16_t *d, const uint32_t *qs, const uint16_t *qh, const int32_t *signs,
                               const uint32_t *scales, int64_t n, int64_t blocks, uint8_t *packed,
                               mambo_stream_t stream)
{
    MAMBO_REQUIRE(d && qs && qh && signs && scales && packed, MAMBO_ERR_VALUE, "null pointer");
    MAMBO_REQUIRE(n >= 1 && blocks >= 1, MAMBO_ERR_VALUE, "IQ3_S weight must have positive N and K");
    MAMBO_REQUIRE((uintptr_t)packed % 16 == 0, MAMBO_ERR_VALUE, "packed must be 16-byte aligned");
    const int64_t tiles = (n + kTileRows - 1) / kTileRows;
    MAMBO_REQUIRE(tiles <= 0x7FFFFFFF, MAMBO_ERR_VALUE, "N too large");
    const dim3 grid((unsigned)((tiles + 3) / 4), (unsigned)(blocks < 65535 ? blocks : 65535));
    MAMBO_LAUNCH(pack_fields_kernel, grid, dim3(256), 0, (hipStream_t)stream, SoaSrc{d, qs, qh, signs, scales}, n,
                 blocks, tiles, packed);
    return mambo_check_launch("iq3s_prepare");
}

extern "C" int mambo_iq3s_dequant(const uint16_t *d, const uint32_t *qs, const uint16_t *qh, const int32_t *signs,
                                  const uint32_t *scales, int64_t n, int64_t blocks, uint8_t *values,
                                  float *out_scales, mambo_stream_t stream)
{
    MAMBO_REQUIRE(d && qs && qh && signs && scales && values && out_scales, MAMBO_ERR_VALUE, "null pointer");
    MAMBO_REQUIRE(n >= 1 && blocks >= 1, MAMBO_ERR_VALUE, "IQ3_S weight must have positive N and K");
    MAMBO_REQUIRE((uintptr_t)values % 16 == 0, MAMBO_ERR_VALUE, "values must be 16-byte aligned");
    // 32 x 4 from 8 M weights; below, its few workgroups of long threads take longer than those of one
    // store each (us, 16 x 1 and 32 x 4, a thread per group before: 512 x 2048 2.6, 3.7 and 2.8, 1024 x
    // 4096 3.5, 4.1 and 4.1, 2048 x 4096 4.6, 4.5 and 5.6, 4096 x 4096 6.7, 6.0 and 8.8)
    const auto launch = n <= 32767 / blocks ? launch_dequant<16, 1> : launch_dequant<32, 4>;
    return launch(d, qs, qh, signs, scales, n, blocks, values, out_scales, (hipStream_t)stream);
}
