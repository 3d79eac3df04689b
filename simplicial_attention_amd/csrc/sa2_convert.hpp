// Conversion of (batch, seq, heads, dim) tensors between the caller's type and head dimension and the kernels' bf16 rows of
// 32, 64, 128 or 256 elements: several tensors per launch.
//
// HBM-bound (each element is read once and written once); what it replaces is a cast, a zero fill and a copy per tensor, one
// launch each, which at small sizes cost more than the attention kernels (2 sequences of 2999 rows, 6 + 4 * 2 heads of 96 fp16
// channels: 190 us in 29 launches, 20 us in four of these).  A thread moves eight consecutive destination channels; the source
// and the destination are accessed 16 bytes at a time where their rows allow it.
#pragma once

#include "sa2_common.hpp"

namespace sa2 {

struct ConvertTensor {
    const char *src;
    char *dst;
    int64_t ssb, ssn, ssh, dsb, dsn, dsh;      // element strides
    int src_type, dst_type;                    // sa2_element
    int src_dim, dst_dim;                      // channels beyond src_dim become zero
    int N, H;
    int64_t pieces;                            // B * N * H * ceil(dst_dim / 8)
    bool src_vec, dst_vec;                     // 16-byte accesses are aligned
};

constexpr int kConvertMost = 6;
struct ConvertParams {
    ConvertTensor t[kConvertMost];
};

__device__ __forceinline__ float convert_load1(const char *p, int type, int64_t at) {
    if (type == 2) return reinterpret_cast<const float *>(p)[at];
    if (type == 1) return (float)reinterpret_cast<const _Float16 *>(p)[at];
    return as_f32((uint32_t)reinterpret_cast<const uint16_t *>(p)[at] << 16);
}
__device__ __forceinline__ void convert_store1(char *p, int type, int64_t at, float v) {
    if (type == 2) reinterpret_cast<float *>(p)[at] = v;
    else if (type == 1) reinterpret_cast<_Float16 *>(p)[at] = (_Float16)v;
    else reinterpret_cast<__bf16 *>(p)[at] = (__bf16)v;
}

static __global__ __launch_bounds__(256) void convert_kernel(ConvertParams p) {
    const ConvertTensor &t = p.t[blockIdx.y];
    typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
    const int per_row = (t.dst_dim + 7) / 8;
    for (int64_t x = (int64_t)blockIdx.x * 256 + threadIdx.x; x < t.pieces; x += (int64_t)gridDim.x * 256) {
        const int d = (int)(x % per_row) * 8;
        const int64_t row = x / per_row;
        const int h = (int)(row % t.H);
        const int64_t bn = row / t.H;
        const int n = (int)(bn % t.N);
        const int64_t b = bn / t.N;
        const int64_t s = b * t.ssb + n * t.ssn + h * t.ssh + d, o = b * t.dsb + n * t.dsn + h * t.dsh + d;
        float v[8];
        if (t.src_vec && d + 8 <= t.src_dim) {
            if (t.src_type == 2) {
                const float4 a = *reinterpret_cast<const float4 *>(t.src + s * 4), c = *reinterpret_cast<const float4 *>(t.src + s * 4 + 16);
                v[0] = a.x; v[1] = a.y; v[2] = a.z; v[3] = a.w;
                v[4] = c.x; v[5] = c.y; v[6] = c.z; v[7] = c.w;
            } else {
                const u32x4 a = ld_global16(t.src + s * 2);
                if (t.src_type == 1) {
                    const f16x8 f = __builtin_bit_cast(f16x8, a);
#pragma unroll
                    for (int e = 0; e < 8; ++e) v[e] = (float)f[e];
                } else {
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        v[2 * w] = bf16_lo(a[w]);
                        v[2 * w + 1] = bf16_hi(a[w]);
                    }
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e) v[e] = d + e < t.src_dim ? convert_load1(t.src, t.src_type, s + e) : 0.f;
        }
        if (t.dst_vec && d + 8 <= t.dst_dim) {
            if (t.dst_type == 2) {
                *reinterpret_cast<float4 *>(t.dst + o * 4) = make_float4(v[0], v[1], v[2], v[3]);
                *reinterpret_cast<float4 *>(t.dst + o * 4 + 16) = make_float4(v[4], v[5], v[6], v[7]);
            } else if (t.dst_type == 1) {
                f16x8 f;
#pragma unroll
                for (int e = 0; e < 8; ++e) f[e] = (_Float16)v[e];
                st_global16(t.dst + o * 2, __builtin_bit_cast(u32x4, f));
            } else {
                st_global16(t.dst + o * 2, (u32x4){pack_bf16(v[0], v[1]), pack_bf16(v[2], v[3]), pack_bf16(v[4], v[5]), pack_bf16(v[6], v[7])});
            }
        } else {
#pragma unroll
            for (int e = 0; e < 8; ++e)
                if (d + e < t.dst_dim) convert_store1(t.dst, t.dst_type, o + e, v[e]);
        }
    }
}

}  // namespace sa2
