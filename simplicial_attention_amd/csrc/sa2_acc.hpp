// Register placement in kernels of one wave per SIMD (256 ordinary and 256 accumulation registers).  The translation units that
// use this header are compiled with -amdgpu-mfma-vgpr-form.
#pragma once

#include "sa2_common.hpp"

namespace sa2 {

// an MFMA operand that stays in accumulation registers, from which an MFMA reads it directly
__device__ __forceinline__ void pin_agpr(u32x4 &x) { asm volatile("" : "+a"(x)); }

// An MFMA whose accumulator stays in accumulation registers, in a kernel whose other MFMA results are in ordinary ones (the
// compiler uses one form per function: 256 result registers beside 128 of operands do not fit either).  Written as assembly, so
// the wait states it needs are this code's business: two behind a VALU write of an operand are in it; nothing else touches the
// accumulator until acc_done.
__device__ __forceinline__ void mfma32_acc(f32x16 &acc, u32x4 a, u32x4 b) {
    asm volatile("s_nop 1\n\tv_mfma_f32_32x32x16_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(a), "v"(b));
}
// behind the last mfma32_acc: waits until its result is written (18 wait states behind an MFMA of 16 passes)
__device__ __forceinline__ void acc_done() { asm volatile("s_nop 15\n\ts_nop 15" ::: "memory"); }

// a value computed at this point of the program (the compiler would move it into the block of its first use, which may be an
// iteration away from the MFMAs it is meant to be issued behind)
__device__ __forceinline__ uint32_t here(uint32_t x) {
    asm volatile("" : "+v"(x));
    return x;
}

}  // namespace sa2
