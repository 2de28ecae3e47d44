// Host interface of the 32 x 32 MFMA projection kernel (iq3s_wide.hip).
#pragma once
#include "mambo_common.h"

// Launch shape of gemm_wide_kernel for one call.
struct WidePlan {
    int mt;     // 32-token sub-tiles per workgroup
    int waves;  // per K group, 32 weight rows each
    int kg;     // K groups of waves per workgroup
    int splits; // K slices (more than one: f32 atomics into outputs zeroed beforehand)
    int bps;    // K blocks per slice
    double us;  // what the plan's cost model expects of it
};

// Whether the kernel takes the call (it can, and is the faster choice), and its plan. other: the
// configuration that takes the call otherwise.
bool mambo_wide_plan(int64_t m, const mambo_projection *proj, int count, int64_t blocks, int64_t ldxv,
                     const uint8_t *xs, int64_t ldxs, const mambo_gemm_config &other, WidePlan *plan);

// Queues the launch; the caller has checked the operands and zeroed the outputs of a plan with
// several slices.
int mambo_wide_launch(const WidePlan &plan, const uint8_t *xv, int64_t ldxv, const uint8_t *xs, int64_t ldxs, int64_t m,
                      const mambo_projection *proj, int count, int64_t blocks, hipStream_t stream);
