// Backward kernel of head dimension 256 that owns query rows: dQ and dK2 (pass DQ), dV2 by recomputation (pass DV).
//
// The passes and their mathematics are those of bwd_q_kernel (sa2_bwd_q.hpp); the split of the work is another.  A wave owns
// an offset and all 256 columns of its results, which takes all 512 registers of a SIMD's lane: the operands A and B (128,
// placed in accumulation registers by hand), the result G or T of the running offset (128), the dq rows over all the wave's
// offsets (128), the logits and dP of a tile (32).  So one workgroup of four waves runs per CU, a round has four offsets, and
// nothing is exchanged inside a step: per (offset, tile) 48 MFMAs (DV: 32) behind one barrier.  The form before it gave every
// wave a quarter of the columns of one offset: eight partial tiles went through LDS and three barriers for every 64 MFMAs,
// and 2 x 8 x 4096 rows (w1 512, w2 32) took 8.9 ms.
// Bound now: a fragment read from LDS feeds one MFMA, so LDS reads (128 B/clk) take as long as the MFMAs themselves.
//
// The rows k that the offsets scatter to live in a circular buffer of 36 fp32 rows (a round reaches 35); a round's additions
// run in four barrier-separated phases in which wave w owns the quarter (w + phase) mod 4 of the columns (fixed order, no
// atomics).  The four rows that a round completes go to the workspace block of the tile, see bwd_q_kernel.
#pragma once

#include <type_traits>

#include "sa2_acc.hpp"
#include "sa2_common.hpp"
#include "sa2_lds.hpp"

namespace sa2 {

template <int D, bool DQ>
struct WideQCfg {
    static constexpr int KS = D / 16;
    static constexpr int DT = D / 32;
    static constexpr int PPR = D / 8;                 // 16-byte pieces per row
    static constexpr int PITCH = tile_pitch<D>();
    using RT = DmaTile<D>;
    static constexpr int TB = RT::BYTES;
    static constexpr int OFF_V = TB;                  // ring buffer: a K1 tile and a V1 tile, two of them
    static constexpr int BUF = 2 * TB;
    static constexpr int RING = 2 * BUF;
    static_assert(RING - RT::CP < 65536, "the LDS address of a direct load travels in 16 bits of M0");
    static constexpr int LPT = RT::NCH / 4;           // loads per wave and tile
    static constexpr int NSLOT = 36;
    static constexpr int SPITCH = D + 4;              // floats per scatter row
    static constexpr int SC = RING;                   // scatter rows, circular
    static constexpr int QS = SC + NSLOT * SPITCH * 4;             // q rows  [32][PITCH]
    static constexpr int DOS = QS + 32 * PITCH;                    // do rows [32][PITCH]
    static constexpr int MASKS = DOS + 32 * PITCH;                 // additive masks, 3 tables [4 quarters][64 lanes][4 floats]
    static constexpr int MASK = 16 * 64 * 4;
    static constexpr int MAIN = MASKS + 3 * MASK;
    static constexpr int MERGE = 4 * 32 * SPITCH * 4;              // the waves' dq rows, at the end
    static constexpr int LDS = MAIN > MERGE ? MAIN : MERGE;
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
};

// rounds of four offsets that query tile `tile` walks
__host__ __device__ inline int wide_rounds(int tile, int w2) {
    const int n = w2 < 32 * tile + 32 ? w2 : 32 * tile + 32;
    return (n + 3) / 4;
}

template <int D, bool DQ>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_wide_q_kernel(KParams p, float *ws, int halo) {
    using C = WideQCfg<D, DQ>;
    using RT = typename C::RT;
    constexpr int KS = C::KS, DT = C::DT, PPR = C::PPR, PITCH = C::PITCH;
    __shared__ __attribute__((aligned(16))) char lds[C::LDS];

    const int N = p.N;
    const int ntile = (N + 31) / 32;
    const int item = xcd_contiguous(blockIdx.x, gridDim.x);
    const int bh = uniform(item / ntile);
    const int tile = ntile - 1 - (item - bh * ntile);
    const int b = uniform(bh / p.H), h = bh - b * p.H;
    const int hk = uniform(h / p.G);
    const int R = wide_rounds(tile, p.w2);

    const int tid = threadIdx.x;
    const int wave = wave_index(), lane = tid & 63;
    const int c = lane & 31, hf = lane >> 5;
    const int i0 = tile * 32;
    const int i = i0 + c;
    const bool row_ok = i < N;
    const int ic = row_ok ? i : N - 1;

    const char *k2g = p.k2.ptr + b * p.k2.sb + hk * p.k2.sh;
    const char *v2g = p.v2.ptr + b * p.v2.sb + hk * p.v2.sh;
    const float lse2 = p.lse[((int64_t)b * p.H + h) * N + ic] * kLog2e;
    const float dl = DQ ? p.delta[((int64_t)b * p.H + h) * N + ic] : 0.f;

    // tiles of the first window, walked in order t_lo .. t_hi; masked: the tiles below mid_lo and the diagonal one
    const int t_lo = (i0 - p.w1 + 1 > 0 ? i0 - p.w1 + 1 : 0) / 32;
    const int t_hi = i0 / 32;
    const int NT = t_hi - t_lo + 1;
    int mid_lo = (i0 + 31 - p.w1 >= 0) ? (i0 + 31 - p.w1) / 32 + 1 : t_lo;
    mid_lo = mid_lo > t_hi ? t_hi : mid_lo;
    const int n_head = mid_lo - t_lo;                 // leading steps of a round with a lower-edge mask (at most 2)

    // ---- ring staging: wave w moves the chunks w, w + 4, ... of both tiles.  The sequence of tiles runs on behind the last
    // round (into a buffer that no wave reads any more).  Only the last tile of a sequence can reach beyond its end: its rows
    // are replaced by the last one.
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds + wave * RT::CP;
    const int st_row = RT::st_row(wave, lane), st_col = RT::st_col(lane);
    const uint32_t so_k = (uint32_t)(st_row * (int)p.k1.sn + st_col), so_v = (uint32_t)(st_row * (int)p.v1.sn + st_col);
    const char *const k_low = p.k1.ptr + b * p.k1.sb + hk * p.k1.sh + (int64_t)(32 * t_lo) * p.k1.sn;
    const char *const v_low = p.v1.ptr + b * p.v1.sb + hk * p.v1.sh + (int64_t)(32 * t_lo) * p.v1.sn;
    const char *kb = k_low, *vb = v_low;
    const bool ragged = i0 + 31 >= N;                 // (then the tile t_hi is the one to clamp)
    int n_load = 0, buf_load = 0;
    auto issue_loads = [&]() {
        const int n = uniform(n_load), dst0 = uniform(buf_load);
        const char *k = uniform(kb), *v = uniform(vb);
        const bool last = n == NT - 1;
        const uint32_t dst = lds_base + dst0;
        if (ragged && last) {
#pragma unroll
            for (int x = 0; x < C::LPT; ++x) {
                int row = st_row + 4 * RT::RPC * x;
                row = i0 + row < N ? row : N - 1 - i0;
                load_to_lds16(k, (uint32_t)(row * (int)p.k1.sn + st_col), dst + 4 * x * RT::CP);
                load_to_lds16(v, (uint32_t)(row * (int)p.v1.sn + st_col), dst + C::OFF_V + 4 * x * RT::CP);
            }
        } else {
#pragma unroll
            for (int x = 0; x < C::LPT; ++x) {
                load_to_lds16(uniform(k + (int64_t)(4 * RT::RPC * x) * p.k1.sn), so_k, dst + 4 * x * RT::CP);
                load_to_lds16(uniform(v + (int64_t)(4 * RT::RPC * x) * p.v1.sn), so_v, dst + C::OFF_V + 4 * x * RT::CP);
            }
        }
        kb = uniform(last ? k_low : k + 32 * p.k1.sn);
        vb = uniform(last ? v_low : v + 32 * p.v1.sn);
        n_load = uniform(last ? 0 : n + 1);
        buf_load = uniform(dst0 ? 0 : C::BUF);
    };
    issue_loads();

    // ---- scatter rows cleared, q / do rows staged, mask tables (see bwd_q_kernel)
    float *sc = reinterpret_cast<float *>(lds + C::SC);
    for (int x = tid; x < C::NSLOT * C::SPITCH / 4; x += 256) reinterpret_cast<float4 *>(sc)[x] = make_float4(0.f, 0.f, 0.f, 0.f);
    {
        const char *qg = p.q.ptr + b * p.q.sb + h * p.q.sh;
        const char *dog = p.dout.ptr + b * p.dout.sb + h * p.dout.sh;
#pragma unroll
        for (int x = tid; x < 32 * PPR; x += 256) {
            const int row = x / PPR, col = (x % PPR) * 16;
            const int ii = i0 + row < N ? i0 + row : N - 1;
            *reinterpret_cast<u32x4 *>(lds + C::QS + row * PITCH + col) = ld_global16(qg + (int64_t)ii * p.q.sn + col);
            *reinterpret_cast<u32x4 *>(lds + C::DOS + row * PITCH + col) = ld_global16(dog + (int64_t)ii * p.dout.sn + col);
        }
    }
    for (int x = tid; x < 3 * 256; x += 256) {
        const int tab = x >> 8, qq = (x >> 6) & 3, ln = x & 63;
        const int t = tab == 0 ? t_hi : t_lo + tab - 1;
        const int rel = (ln & 31) + 32 * (t_hi - t) - 4 * (ln >> 5);
        float4 m4;
        float *mp = &m4.x;
#pragma unroll
        for (int e = 0; e < 4; ++e) mp[e] = ((unsigned)(rel - (8 * qq + e)) < (unsigned)p.w1) ? 0.f : -INFINITY;
        *reinterpret_cast<float4 *>(lds + C::MASKS + tab * C::MASK + qq * 1024 + ln * 16) = m4;
    }

    // scatter rows of this tile in the workspace: row x <-> k = i0 - halo + x
    const int srows = 32 + halo;
    const int64_t per_tensor = (int64_t)p.B * p.H * ntile * srows * D;
    float *wk = ws + (DQ ? 0 : per_tensor) + (((int64_t)b * p.H + h) * ntile + tile) * srows * D;
    auto slot_of = [&](int rel) {
        const int s = rel % C::NSLOT;
        return s < 0 ? s + C::NSLOT : s;
    };
    // rows k - i0 = lo .. lo + n - 1 go to the workspace and are cleared for reuse
    auto flush_rows = [&](int lo, int n) {
        for (int x = tid; x < n * (D / 4); x += 256) {
            const int rel = lo + x / (D / 4), col = (x % (D / 4)) * 4;
            float4 *src = reinterpret_cast<float4 *>(sc + (slot_of(rel) * C::SPITCH + col));
            *reinterpret_cast<float4 *>(wk + (int64_t)(rel + halo) * D + col) = *src;
            *src = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };

    f32x16 acc[DT];            // G^T (DQ) or T^T (DV) of the running offset
    f32x16 dq[DQ ? DT : 1];
    u32x4 A[KS], B[DQ ? KS : 1];
    if constexpr (DQ) {
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) dq[dt] = zero16();
    }
    // the k2 (and v2) rows i - dlt, in the operands' layout
    auto load_rows = [&](int dlt) {
        int kr = i - dlt;
        kr = kr < 0 ? 0 : (kr < N ? kr : N - 1);
        const char *k2r = k2g + (int64_t)kr * p.k2.sn + 16 * hf, *v2r = v2g + (int64_t)kr * p.v2.sn + 16 * hf;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            A[kk] = ld_global16(k2r + 32 * kk);
            if constexpr (DQ) B[kk] = ld_global16(v2r + 32 * kk);
        }
    };
    load_rows(wave);
    __syncthreads();

    const int r_lane = RT::row_lane(lane), t_lane = RT::tr_lane(lane);
    const f32x2 ndl2 = {-dl, -dl};
    int buf = 0;
    // a step's tiles are in (all waves have left the step before, whose buffer the next ones take)
    auto open_step = [&] {
        wait_loads<0>();
        __syncthreads();
        issue_loads();
    };
    for (int r = 0; r < R; ++r) {
        const int dlt = 4 * r + wave;
        const bool col_ok = row_ok && i - dlt >= 0 && dlt < p.w2;
        const bool wave_on = wave_any(col_ok);
        {
            const char *qr = lds + C::QS + c * PITCH + 16 * hf, *dor = lds + C::DOS + c * PITCH + 16 * hf;
            const float c2 = p.scale_log2e;
#pragma unroll
            for (int kk = 0; kk < KS; ++kk) {
                const u32x4 fq = ld_lds16(qr + 32 * kk), fk = A[kk];
#pragma unroll
                for (int w = 0; w < 4; ++w) A[kk][w] = pack_bf16(bf16_lo(fq[w]) * c2 * bf16_lo(fk[w]), bf16_hi(fq[w]) * c2 * bf16_hi(fk[w]));
                pin_agpr(A[kk]);
                if constexpr (DQ) {
                    B[kk] = mul_bf16x8(ld_lds16(dor + 32 * kk), B[kk]);
                    pin_agpr(B[kk]);
                }
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16_pairs();
        }
        const float nl = col_ok ? -lse2 : -INFINITY;  // where the logit chains start
        const f32x2 nl2 = {nl, nl};

        if (!wave_on)              // (a wave that is off stays off: later rounds have larger offsets)
            for (int n = 0; n < NT; ++n) open_step();
        else
            for (int n = 0; n < NT; ++n) {
                open_step();
                const char *sub = lds + buf;
                // One stream of fragments, a window of W in flight (see bwd_q_kernel): the K1 row fragments of the logit chain,
                // (DQ) the V1 row fragments of the dP chain, the transposed fragments of the accumulating products
                constexpr int W = 6;
                constexpr int NROW = DQ ? 2 * KS : KS, NFR = NROW + 2 * DT;
                const char *kf = sub + r_lane, *vf = sub + C::OFF_V + r_lane;
                const char *tf = sub + (DQ ? 0 : C::OFF_V) + t_lane;
                auto fragment = [&](auto idx) {
                    constexpr int s = decltype(idx)::value;
                    if constexpr (s < KS) return RT::row_frag(kf, s);
                    else if constexpr (s < NROW) return RT::row_frag(vf, s - KS);
                    else return RT::tr_frag(tf, (s - NROW) / DT, (s - NROW) % DT);
                };
                u32x4 f[W];
                static_for<0, W>([&](auto s) { f[s] = fragment(s); });
                f32x16 X = splat16_pairs(nl2);
                const bool diag = n == NT - 1;
                if (diag || n < n_head) {
                    const char *mk = lds + C::MASKS + (diag ? 0 : 1 + n) * C::MASK + lane * 16;
    #pragma unroll
                    for (int qq = 0; qq < 4; ++qq) {
                        const float4 m4 = *reinterpret_cast<const float4 *>(mk + qq * 1024);
                        X[4 * qq] += m4.x;
                        X[4 * qq + 1] += m4.y;
                        X[4 * qq + 2] += m4.z;
                        X[4 * qq + 3] += m4.w;
                    }
                }
                f32x16 dP = splat16_pairs(ndl2);
                u32x4 pb[2];
                // (DQ: the exponentials are issued between the MFMAs of the dP chain, dS needs its end)
                auto weights = [&](int rr) {
                    float p0 = DQ ? X[rr] : fast_exp2(X[rr]), p1 = DQ ? X[rr + 1] : fast_exp2(X[rr + 1]);
                    if constexpr (DQ) {
                        p0 *= dP[rr];
                        p1 *= dP[rr + 1];
                    }
                    pb[rr >> 3][(rr & 7) >> 1] = pack_bf16(p0, p1);
                };
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, NROW>([&](auto s_) {
                    constexpr int s = decltype(s_)::value;
                    if constexpr (s < KS) X = mfma32(f[s % W], A[s], X);
                    else dP = mfma32(f[s % W], B[DQ ? s - KS : 0], dP);
                    if constexpr (s + W < NFR) f[s % W] = fragment(std::integral_constant<int, s + W>{});
                    if constexpr (DQ && s > KS) {
                        constexpr int e = s - KS - 1;           // (one behind each, the last two together)
                        X[e] = fast_exp2(X[e]);
                        if constexpr (s == NROW - 1) X[e + 1] = fast_exp2(X[e + 1]);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
    #pragma unroll
                for (int rr = 0; rr < 8; rr += 2) weights(rr);
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, 2 * DT>([&](auto s_) {
                    constexpr int s = decltype(s_)::value;      // k-slice s / DT, d tile s % DT
                    acc[s % DT] = mfma32(f[(NROW + s) % W], pb[s / DT], acc[s % DT]);
                    if constexpr (NROW + s + W < NFR) f[(NROW + s) % W] = fragment(std::integral_constant<int, NROW + s + W>{});
                    if constexpr (s < 4) weights(8 + 2 * s);
                    __builtin_amdgcn_sched_barrier(0);
                });
                buf = uniform(buf ? 0 : C::BUF);
            }

        // ---- round end: dq_i += k2_{i-dlt} * G in registers, scatter row i - dlt += q_i * G (times scale log2(e): the combine
        // kernel multiplies by ln 2) or do_i * T in LDS, one quarter of the columns per wave and phase
        {
            u32x4 kx[DQ ? 2 * DT : 1];
            if constexpr (DQ) {
                int kr = i - dlt;
                kr = kr < 0 ? 0 : (kr < N ? kr : N - 1);
                const char *k2r = k2g + (int64_t)kr * p.k2.sn + 32 * hf;
#pragma unroll
                for (int x = 0; x < 2 * DT; ++x) kx[x] = ld_global16(k2r + (x >> 1) * 64 + (x & 1) * 16);
            }
            const char *xr = lds + (DQ ? C::QS : C::DOS) + c * PITCH + 32 * hf;
            float *srow = sc + slot_of(c - dlt) * C::SPITCH + 16 * hf;
            const float xs = DQ ? p.scale_log2e : 1.f;
            // (a column without a key row holds zeros: its logits started from -inf)
            auto add_quarter = [&](auto quarter_tag) {
                constexpr int Q = decltype(quarter_tag)::value;
#pragma unroll
                for (int x = 2 * DT / 4 * Q; x < 2 * DT / 4 * (Q + 1); ++x) {
                    const int dt = x >> 1, r0 = 8 * (x & 1);
                    const u32x4 xq = ld_lds16(xr + dt * 64 + r0 * 2);
                    float4 *dst = reinterpret_cast<float4 *>(srow + 32 * dt + r0);
                    float4 a0 = dst[0], a1 = dst[1];
                    a0.x += bf16_lo(xq[0]) * xs * acc[dt][r0];
                    a0.y += bf16_hi(xq[0]) * xs * acc[dt][r0 + 1];
                    a0.z += bf16_lo(xq[1]) * xs * acc[dt][r0 + 2];
                    a0.w += bf16_hi(xq[1]) * xs * acc[dt][r0 + 3];
                    a1.x += bf16_lo(xq[2]) * xs * acc[dt][r0 + 4];
                    a1.y += bf16_hi(xq[2]) * xs * acc[dt][r0 + 5];
                    a1.z += bf16_lo(xq[3]) * xs * acc[dt][r0 + 6];
                    a1.w += bf16_hi(xq[3]) * xs * acc[dt][r0 + 7];
                    dst[0] = a0;
                    dst[1] = a1;
                }
            };
            for (int ph = 0; ph < 4; ++ph) {
                if (wave_on) with_slice<4>(wave + ph, add_quarter);
                __syncthreads();
            }
            if constexpr (DQ) {
#pragma unroll
                for (int x = 0; x < 2 * DT; ++x)
#pragma unroll
                    for (int w = 0; w < 4; ++w) {
                        dq[x >> 1][8 * (x & 1) + 2 * w] += bf16_lo(kx[x][w]) * acc[x >> 1][8 * (x & 1) + 2 * w];
                        dq[x >> 1][8 * (x & 1) + 2 * w + 1] += bf16_hi(kx[x][w]) * acc[x >> 1][8 * (x & 1) + 2 * w + 1];
                    }
            }
            if (r + 1 < R) load_rows(dlt + 4);
            // the rows k - i0 = 28 - 4 r .. 31 - 4 r are complete: no later round reaches them
            if (r + 1 < R) flush_rows(28 - 4 * r, 4);
        }
    }
    wait_loads<0>();           // (the transfer issued behind the last tile still writes into the ring)
    // ---- the rows that the last round leaves, k - i0 = -4 (R - 1) - 3 .. 31 - 4 (R - 1), and zeros in those below that the
    // block has room for
    const int low = -4 * (R - 1) - 3;
    flush_rows(low, 35);
    for (int x = tid; x < (low + halo) * (D / 4); x += 256) reinterpret_cast<float4 *>(wk)[x] = make_float4(0.f, 0.f, 0.f, 0.f);

    // ---- dq rows: the sum over the waves, in their order
    if constexpr (DQ) {
        __syncthreads();
        float *rows = reinterpret_cast<float *>(lds);
        store_row_f32(rows + (wave * 32 + c) * C::SPITCH + 16 * hf, dq, p.scale);
        __syncthreads();
        const int row = tid >> 3, seg = tid & 7;
        const int ir = i0 + row;
        if (ir >= N) return;
        char *orow = p.dq.ptr + b * p.dq.sb + (int64_t)ir * p.dq.sn + h * p.dq.sh;
#pragma unroll
        for (int x = 0; x < D / 32; ++x) {
            const int d = 4 * (seg + 8 * x);
            float4 a = *reinterpret_cast<const float4 *>(rows + row * C::SPITCH + d);
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                const float4 e = *reinterpret_cast<const float4 *>(rows + (w * 32 + row) * C::SPITCH + d);
                a.x += e.x;
                a.y += e.y;
                a.z += e.z;
                a.w += e.w;
            }
            *reinterpret_cast<u32x2 *>(orow + d * 2) = (u32x2){pack_bf16(a.x, a.y), pack_bf16(a.z, a.w)};
        }
    }
}

}  // namespace sa2
