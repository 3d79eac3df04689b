// Launches of kernels that are compiled in a translation unit of their own (with code generation flags of their own).
#pragma once

#include <hip/hip_runtime.h>

#include "sa2_common.hpp"

namespace sa2 {

// forward at head dimension 128 (sa2_fwd2.hip); split: SPLIT form, q_splits workgroups per query tile
void launch_fwd2(bool split, int grid, hipStream_t stream, const KParams &p);

}  // namespace sa2
