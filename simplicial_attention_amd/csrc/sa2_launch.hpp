// Launches of kernels that are compiled in a translation unit of their own (with code generation flags of their own).
#pragma once

#include <hip/hip_runtime.h>

#include "sa2_common.hpp"

namespace sa2 {

// forward at head dimension 128 (sa2_fwd2.hip); split: SPLIT form, q_splits workgroups per query tile
// head dimension 256 (sa2_wide.hip); dq: dQ and the dK2 rows, else the dV2 rows
void launch_fwd_wide(int grid, hipStream_t stream, const KParams &p);
void launch_bwd_wide_q(bool dq, int grid, hipStream_t stream, const KParams &p, float *ws, int halo);
void launch_bwd_wide_kv(int grid, hipStream_t stream, const KParams &p);

void launch_fwd2(bool split, int grid, hipStream_t stream, const KParams &p);

}  // namespace sa2
