// Addresses of gemm_wide_kernel's activation copies (iq3s_wide.hip): plain constexpr functions, so
// that the host can check every lane's bytes against the tensor's end.
//
// The offset of a lane is all of its address but the block (256 * b and 8 * b, the copies' scalar
// offset) and rows past the last one are the last one again, so that no copy leaves the tensor
// whatever the buffer resource's range check counts.
#pragma once
#include <stdint.h>

// Values: copy j of a wave moves 1 KiB, rows 4 * (wave + waves * j) .. + 3 of the token tile, 16
// bytes a lane; chunk c of row i comes to slot c ^ (i & 15) of the row in LDS.
constexpr uint32_t wide_value_offset(int wave, int lane, int waves, int j, int last_row, uint32_t ldxv)
{
    const int row = 4 * (wave + waves * j) + (lane >> 4);
    return (uint32_t)(row < last_row ? row : last_row) * ldxv + 16u * (uint32_t)((lane & 15) ^ (row & 15));
}

// Scales: copy `part` moves 256 bytes, rows 32 * part .. + 31, four bytes a lane.
constexpr uint32_t wide_scale_offset(int part, int lane, int last_row, uint32_t ldxs)
{
    const int row = 32 * part + (lane >> 1);
    return (uint32_t)(row < last_row ? row : last_row) * ldxs + 4u * (uint32_t)(lane & 1);
}
