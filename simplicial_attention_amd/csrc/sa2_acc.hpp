// Register placement in kernels of one wave per SIMD (256 ordinary and 256 accumulation registers).  The translation units that
// use this header are compiled with -amdgpu-mfma-vgpr-form.
#pragma once

#include "sa2_common.hpp"

namespace sa2 {

// an MFMA operand that stays in accumulation registers, from which an MFMA reads it directly
__device__ __forceinline__ void pin_agpr(u32x4 &x) { asm volatile("" : "+a"(x)); }

// a value computed at this point of the program (the compiler would move it into the block of its first use, which may be an
// iteration away from the MFMAs it is meant to be issued behind)
__device__ __forceinline__ uint32_t here(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}

}  // namespace sa2
