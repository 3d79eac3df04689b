// Launches of kernels that are compiled in a translation unit of their own (with code generation flags of their own).
#pragma once

#include <hip/hip_runtime.h>

#include "sa2_common.hpp"

namespace sa2 {

// head dimension 256 (sa2_wide.hip); dq: dQ and the dK2 rows, else the dV2 rows
void launch_fwd_wide(int grid, hipStream_t stream, const KParams &p);
void launch_bwd_wide_q(bool dq, int grid, hipStream_t stream, const KParams &p, float *ws, int halo);

// dK1/dV1 at head dimension 256 (sa2_kvr.hip); in_parts: PARTS form, kv_max_parts workgroups per key slab
void launch_bwd_kvr(bool in_parts, int grid, hipStream_t stream, const KParams &p);

// forward at head dimension 128 (sa2_fwd2.hip); split: SPLIT form, q_splits workgroups per query tile
void launch_fwd2(bool split, int grid, hipStream_t stream, const KParams &p);

}  // namespace sa2
