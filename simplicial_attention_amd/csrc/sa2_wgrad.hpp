// Weight gradient of a linear layer: dW[m][n] = sum over rows k of dY[k][m] X[k][n], bf16 operands, fp32 sums.
//
// Both operands have the contracted index as their slow one, so both are read transposed out of LDS (ds_read_b64_tr_b16) from
// tiles that direct-to-LDS loads fill (DmaTile).  The rows are many (every token of a batch) and the result is small: a workgroup
// owns a 128 x 128 block and a share of the rows, the shares leave fp32 blocks that a second kernel adds in order.  Four waves of
// 64 x 64 (four accumulators), three buffers of 32 rows: the transfer of a tile has two steps to land.
// Bound by the latency of its steps (640 TFLOP/s at 16384 rows, 2048 x 512): 53 us, where the library's kernel, 64 x 64 blocks
// without shares, takes 104; 512 x 512: 28 against 99.
#pragma once

#include "sa2_common.hpp"
#include "sa2_lds.hpp"

namespace sa2 {

struct WgradParams {
    const char *dy, *x;
    int64_t dy_row, x_row;        // bytes between rows
    float *parts;                 // [share][M][N]
    char *dw;                     // bf16 [M][N]
    int K, M, N, shares, share_tiles;     // rows in 32-row tiles: share_tiles per share
};

struct WgradCfg {
    using T = DmaTile<128>;
    static constexpr int NBUF = 3;
    static constexpr int BUF = 2 * T::BYTES;
    static constexpr int LDS = NBUF * BUF;
};

static __global__ __launch_bounds__(256) void wgrad_kernel(WgradParams p) {
    using C = WgradCfg;
    using T = C::T;
    __shared__ __attribute__((aligned(16))) char lds[C::LDS];
    const int nb = p.N / 128, mb = p.M / 128;
    const int item = xcd_contiguous(blockIdx.x, gridDim.x);      // (blocks of one share side by side: they read the same rows)
    const int share = uniform(item / (nb * mb)), blk = item - share * (nb * mb);
    const int m0 = uniform(blk / nb) * 128, n0 = (blk - uniform(blk / nb) * nb) * 128;
    const int t0 = share * p.share_tiles, tiles = (p.K + 31) / 32;
    const int nt = tiles - t0 < p.share_tiles ? tiles - t0 : p.share_tiles;
    const int lane = threadIdx.x & 63, wave = wave_index();
    const int c = lane & 31, hf = lane >> 5;

    // wave w moves the chunks w and w + 4 of both tiles
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    const int st_row = T::st_row(wave, lane), st_col = T::st_col(lane);
    const uint32_t oy = (uint32_t)(st_row * (int)p.dy_row + st_col), ox = (uint32_t)(st_row * (int)p.x_row + st_col);
    const char *gy = p.dy + (int64_t)t0 * 32 * p.dy_row + m0 * 2, *gx = p.x + (int64_t)t0 * 32 * p.x_row + n0 * 2;
    const int rest = p.K % 32;                 // rows of the last tile, where it is not whole: the others are filled with the last row
    auto ragged = [&](int t) { return rest != 0 && t0 + t == tiles - 1; };      // ... and cleared before they are used
    auto issue = [&](int t) {                  // tile t of the share (waits for nothing)
        const uint32_t dst = uniform((int)(lds0 + (t % C::NBUF) * C::BUF + wave * T::CP));
        const char *y = uniform(gy + (int64_t)t * 32 * p.dy_row), *x = uniform(gx + (int64_t)t * 32 * p.x_row);
        if (ragged(t)) {
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int row = st_row + 16 * h < rest ? st_row + 16 * h : rest - 1;
                load_to_lds16(y, (uint32_t)(row * (int)p.dy_row + st_col), dst + 4 * h * T::CP);
                load_to_lds16(x, (uint32_t)(row * (int)p.x_row + st_col), dst + T::BYTES + 4 * h * T::CP);
            }
            return;
        }
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            load_to_lds16(uniform(y + (int64_t)(16 * h) * p.dy_row), oy, dst + 4 * h * T::CP);
            load_to_lds16(uniform(x + (int64_t)(16 * h) * p.x_row), ox, dst + T::BYTES + 4 * h * T::CP);
        }
    };
    issue(0);
    if (nt > 1) issue(1);
    f32x16 acc[2][2];                          // [m block][n block]
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[a][b] = zero16();
    const int wm = 2 * (wave >> 1), wn = 2 * (wave & 1);
    const int t_lane = T::tr_lane(lane);
    for (int t = 0; t < nt; ++t) {
        if (t + 1 < nt) wait_loads<4>();       // (the four loads of the next tile may still be under way)
        else wait_loads<0>();
        __syncthreads();                       // the tile is in, and every wave has left the one before, whose buffer is next
        if (t + 2 < nt) issue(t + 2);
        if (ragged(t)) {
            for (int n = threadIdx.x; n < 2 * (32 - rest) * 16; n += 256) {
                const int row = rest + n / 32, piece = n % 16;
                *reinterpret_cast<u32x4 *>(lds + (t % C::NBUF) * C::BUF + (n & 16 ? T::BYTES : 0) + T::off(row, 8 * piece)) = (u32x4){0, 0, 0, 0};
            }
            __syncthreads();
        }
        const char *y = lds + (t % C::NBUF) * C::BUF + t_lane, *x = y + T::BYTES;
        u32x4 fy[2][2], fx[2][2];
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int a = 0; a < 2; ++a) {
                fy[s][a] = T::tr_frag(y, s, wm + a);
                fx[s][a] = T::tr_frag(x, s, wn + a);
            }
#pragma unroll
        for (int s = 0; s < 2; ++s)
#pragma unroll
            for (int a = 0; a < 2; ++a)
#pragma unroll
                for (int b = 0; b < 2; ++b) acc[a][b] = mfma32(fx[s][b], fy[s][a], acc[a][b]);
    }
    // column c of an MFMA result is row m = dmap_row(c) of dW, register r column n = 16 hf + r
    float *out = p.parts + (int64_t)share * p.M * p.N;
#pragma unroll
    for (int a = 0; a < 2; ++a)
#pragma unroll
        for (int b = 0; b < 2; ++b) {
            float *row = out + (int64_t)(m0 + 32 * (wm + a) + dmap_row(c)) * p.N + n0 + 32 * (wn + b) + 16 * hf;
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *reinterpret_cast<float4 *>(row + 4 * r4) = make_float4(acc[a][b][4 * r4], acc[a][b][4 * r4 + 1], acc[a][b][4 * r4 + 2], acc[a][b][4 * r4 + 3]);
        }
}

// the shares added in order, eight elements per thread
static __global__ __launch_bounds__(256) void wgrad_combine_kernel(WgradParams p) {
    const int64_t at = ((int64_t)blockIdx.x * 256 + threadIdx.x) * 8, all = (int64_t)p.M * p.N;
    if (at >= all) return;
    float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const float *src = p.parts + at;
#pragma unroll 4
    for (int x = 0; x < p.shares; ++x, src += all) {
        const float4 a = *reinterpret_cast<const float4 *>(src), b = *reinterpret_cast<const float4 *>(src + 4);
        s[0] += a.x;
        s[1] += a.y;
        s[2] += a.z;
        s[3] += a.w;
        s[4] += b.x;
        s[5] += b.y;
        s[6] += b.z;
        s[7] += b.w;
    }
    st_global16(p.dw + at * 2, (u32x4){pack_bf16(s[0], s[1]), pack_bf16(s[2], s[3]), pack_bf16(s[4], s[5]), pack_bf16(s[6], s[7])});
}

}  // namespace sa2
