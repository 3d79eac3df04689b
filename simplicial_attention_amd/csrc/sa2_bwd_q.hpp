// Backward kernels that own query rows: dQ and dK2 (pass DQ), dV2 by recomputation (pass DV).
//
// Same shape as the forward: one workgroup owns 32 query rows i of one (batch, head), in round r
// wave w handles the offset dlt = i - k = 8r + w (any second window), and all waves walk the same
// K1/V1 tiles through a double-buffered LDS ring, one tile and one barrier per step.  A fused
// kernel (S, dP, T and G accumulators together) needs more than 256 registers per wave, which
// forces one wave per SIMD; so the work is split into two passes that each fit two waves per SIMD:
//
//   pass DQ, with A = q_i * k2_{i-dlt} * scale * log2(e), B = do_i * v2_{i-dlt}:
//       S^T = K1 A^T,  dP^T = V1 B^T,  dS = P (dP - delta_i),  G^T += K1^T dS^T
//       dq_i += k2_{i-dlt} * G_i,   dk2_{i-dlt} += q_i * G_i
//   pass DV:
//       S^T = K1 A^T,  T^T += V1^T P^T,   dv2_{i-dlt} += do_i * T_i
//
// with P = exp2(S - lse_i log2(e)).  The logit chain starts from -lse_i log2(e) (from -inf in lanes
// without a valid (row, offset)) plus an additive 0 / -inf mask from an LDS table on the diagonal tile
// and on the tiles that the window's lower edge crosses, so its result is the exponent; the dP chain
// starts from -delta_i.  No mask, subtraction or scaling code follows the chains.
// Sums over offsets go to fp32 LDS rows shared by the workgroup; a round's additions run in eight
// barrier-separated phases in which wave w owns the d-slice (w + phase) mod 8, so no two waves touch
// one element at a time and the order is fixed (bitwise reproducible, no atomics).  The rows k that
// the offsets scatter to live in a 64-row circular buffer (row k in slot (k - i0) mod 64); the eight
// rows that a round completes go to the fp32 workspace:
// [tensor 0: dk2, 1: dv2][b][h][tile][32 + halo][D], row x of a tile <-> k = i0 - halo + x, with
// halo = 8 ceil(w2 / 8) - 1.  combine_rows reduces it, in dk2_dv2_combine_kernel or, on small grids with
// saved forward partials, in small_grid_merge_kernel, beside dV2.
#pragma once

#include <type_traits>

#include "sa2_common.hpp"
#include "sa2_fwd.hpp"
#include "sa2_lds.hpp"

namespace sa2 {

template <int D, bool DQ>
struct QCfg {
    static constexpr int PITCH = tile_pitch<D>();     // staged q / do / k2 / v2 rows
    static constexpr int TILE = 32 * PITCH;
    // ring buffer: a K1 tile and a V1 tile, written by direct-to-LDS loads (layout: DmaTile; DQ reads K1 both ways)
    using RT = DmaTile<D>;
    static constexpr int OFF_V = RT::BYTES;
    static constexpr int BUF = 2 * RT::BYTES;
    static constexpr int RING = 2 * BUF;
    static constexpr int SPITCH = D + 4;              // floats per row of the fp32 rows
    static constexpr int DQS = RING;                  // dq rows [32][SPITCH]            (DQ only)
    static constexpr int SC = RING + (DQ ? 32 * SPITCH * 4 : 0);   // scatter rows, circular [64][SPITCH]
    static constexpr int QS = SC + 64 * SPITCH * 4;                // q rows times scale log2(e), fp32 [32][QPITCH bytes]
    static constexpr int QPITCH = D * 4 + 16;
    static constexpr int DOS = QS + 32 * QPITCH;                   // do rows  [32][PITCH]
    static constexpr int K2S = DOS + TILE;                         // k2 rows, circular [64][PITCH]
    static constexpr int V2S = K2S + 64 * PITCH;                   // v2 rows, circular [64][PITCH]  (DQ only)
    static constexpr int MASKS = DQ ? V2S + 64 * PITCH : V2S;      // additive masks, 3 tables [4 quarters][64 lanes][4 floats]
    static constexpr int MASK = 16 * 64 * 4;
    static constexpr int LDS = MASKS + 3 * MASK;
    static constexpr int PPR = D / 8;                 // 16-byte pieces per row
    static constexpr int PIECES = 32 * PPR;           // ... per tile
    // dQ pass at D = 64: the start values of the logit chains stay in 16 registers for a round (198 of 256; at D = 128 none are
    // left) instead of being copied together at every step.  A step has 12 MFMAs there, and what it issues beside them is the
    // bound: 919 -> 890 us at 8 x 8 (4 kv) x 2048 rows, w1 512, w2 32.  At D = 32 it is no gain: 694 us there either way, and 2533 us
    // copied, 2580 kept at 2 x 4 x 30000 rows, w1 200, w2 100, where many rounds have few steps each.
    static constexpr bool KEEP_NL = DQ && D == 64;
};

// SPLIT: the rounds of a query tile are shared by p.q_splits workgroups (fwd_split_round); each leaves its dq rows in
// p.q_parts as fp32 and its scatter rows in a workspace block of its own, which the combine kernel adds in split order.
//
// workspace layout (floats): [split][tensor 0: dk2, 1: dv2 (not with saved forward partials)][b][h][tile][srows][D], srows = 32 + halo
__host__ __device__ inline int64_t qk2_ws_floats(int B, int H, int N, int D, int srows) {   // of one split
    return 2ll * B * H * ((N + 31) / 32) * srows * D;
}

// CH < D: the channels from CH on are zero in every operand (rows of narrower heads padded to D), and the products over them
// are left out: their k-slots add zeros to S and dP, their rows of G are zero.  2 x 6 (2 kv) x 2999 rows of 96 channels,
// w1 300, w2 20: 243 -> 204 us.
template <int D, bool DQ, bool SPLIT = false, int CH = D>
__global__ __launch_bounds__(512) void bwd_q_kernel(KParams p, float *ws, int halo) {
    using C = QCfg<D, DQ>;
    constexpr int KS = CH / 16, DT = CH / 32, PPR = C::PPR, PITCH = C::PITCH;
    static_assert(CH % 32 == 0, "whole tiles of channels");
    constexpr bool KEEP_NL = C::KEEP_NL || CH < D;    // (218 registers at CH = 96 without them)
    __shared__ __attribute__((aligned(16))) char lds[C::LDS];

    const int N = p.N;
    const int ntile = (N + 31) / 32;
    const int item_all = xcd_contiguous(blockIdx.x, gridDim.x);
    const int item = SPLIT ? uniform(item_all / p.q_splits) : item_all;
    const int split = SPLIT ? item_all - item * p.q_splits : 0;
    const int bh = uniform(item / ntile);
    const int tile = ntile - 1 - (item - bh * ntile);
    const int b = uniform(bh / p.H), h = bh - b * p.H;
    const int hk = uniform(h / p.G);
    // rounds r_first .. R - 1 of eight offsets each
    const int rounds = fwd_rounds(tile, p.w2);
    const int r_first = SPLIT ? uniform(fwd_split_round(split, p.q_splits, rounds)) : 0;
    const int R = SPLIT ? uniform(fwd_split_round(split + 1, p.q_splits, rounds)) : rounds;
    if (SPLIT && r_first >= R) return;

    const int tid = threadIdx.x;
    const int wave = wave_index(), lane = tid & 63;
    const int c = lane & 31, hf = lane >> 5;
    const int i0 = tile * 32;
    const int i = i0 + c;
    const bool row_ok = i < N;
    const int ic = row_ok ? i : N - 1;

    const char *k1g = p.k1.ptr + b * p.k1.sb + hk * p.k1.sh;
    const char *v1g = p.v1.ptr + b * p.v1.sb + hk * p.v1.sh;
    const char *k2g = p.k2.ptr + b * p.k2.sb + hk * p.k2.sh;
    const char *v2g = p.v2.ptr + b * p.v2.sb + hk * p.v2.sh;
    const float lse2 = p.lse[((int64_t)b * p.H + h) * N + ic] * kLog2e;
    // delta of the tile's rows: read, or, in a split grid that is given the out rows, formed here and left for the dK1/dV1
    // kernel (small grids only: there a launch less counts, while the kernel of its own is 1/2 % of a large backward)
    __shared__ float delta_s[SPLIT ? 32 : 1];
    float dl = 0.f;
    if constexpr (DQ && !SPLIT) dl = p.delta[((int64_t)b * p.H + h) * N + ic];

    // tiles of the first window, walked in order t_lo .. t_hi; masked: the tiles below mid_lo and the diagonal one
    const int t_lo = (i0 - p.w1 + 1 > 0 ? i0 - p.w1 + 1 : 0) / 32;
    const int t_hi = i0 / 32;
    const int NT = t_hi - t_lo + 1;
    int mid_lo = (i0 + 31 - p.w1 >= 0) ? (i0 + 31 - p.w1) / 32 + 1 : t_lo;   // first tile that no row masks at the window's lower edge
    mid_lo = mid_lo > t_hi ? t_hi : mid_lo;
    const int n_head = mid_lo - t_lo;                 // leading steps of a round with a lower-edge mask (at most 2)

    // ---- ring staging: direct-to-LDS loads, wave w moves chunk w of the K1 tile and of the V1 tile (D = 64: four
    // chunks per tile, waves 0-3 stage)
    using RT = typename C::RT;
    const bool stager = RT::NCH >= 8 || wave < RT::NCH;
    const int st_row = RT::st_row(wave % RT::NCH, lane), st_col = RT::st_col(lane);
    int n_load = 0, u_load = 0;
    // address = tile base (uniform) + this lane's row and column (32 bits); only the diagonal tile can
    // reach past the last row, so only it needs a clamped row
    const int st_row_diag = i0 + st_row < N ? st_row : N - 1 - i0;
    const uint32_t so_k = (uint32_t)(st_row * (int)p.k1.sn + st_col), so_v = (uint32_t)(st_row * (int)p.v1.sn + st_col);
    const uint32_t so_k_diag = (uint32_t)(st_row_diag * (int)p.k1.sn + st_col), so_v_diag = (uint32_t)(st_row_diag * (int)p.v1.sn + st_col);
    const uint32_t lds_chunk = (uint32_t)(uintptr_t)lds + (wave % RT::NCH) * RT::CP;
    // tile bases as running pointers (t_lo, t_lo + 1, ..., t_hi, then t_lo again: no multiplications in the step).
    // Loads are issued at every step, also behind the last tile (the sequence runs on into a buffer that no wave
    // reads any more), so the step has no branch on its position; the kernel waits for the last ones before it ends.
    const char *const k_low = k1g + (int64_t)(32 * t_lo) * p.k1.sn, *const v_low = v1g + (int64_t)(32 * t_lo) * p.v1.sn;
    const int64_t k_step = 32 * p.k1.sn, v_step = 32 * p.v1.sn;
    const char *kb = k_low, *vb = v_low;
    auto issue_loads = [&]() {
        const bool diag = n_load == NT - 1;           // the diagonal tile t_hi closes the sequence
        if (stager) {
            const uint32_t dst = lds_chunk + (u_load & 1) * C::BUF;
            load_to_lds16(kb, diag ? so_k_diag : so_k, dst);
            load_to_lds16(vb, diag ? so_v_diag : so_v, dst + C::OFF_V);
        }
        ++u_load;
        kb = diag ? k_low : kb + k_step;
        vb = diag ? v_low : vb + v_step;
        n_load = diag ? 0 : n_load + 1;
    };
    const int r_lane = RT::row_lane(lane);            // row fragment: row c, pieces 2*kk + hf
    const int t_lane = RT::tr_lane(lane);             // transposed fragment, per-lane part

    // ---- fp32 rows shared by the workgroup, zeroed; q/do rows and the k2/v2 rows of the first round staged
    float *dqs = reinterpret_cast<float *>(lds + C::DQS);
    float *sc = reinterpret_cast<float *>(lds + C::SC);
    {
        float4 *z = reinterpret_cast<float4 *>(lds + C::RING);
        constexpr int NZ = (C::QS - C::RING) / 16;
        for (int x = tid; x < NZ; x += 512) z[x] = make_float4(0.f, 0.f, 0.f, 0.f);
        const char *qg = p.q.ptr + b * p.q.sb + h * p.q.sh;
        const char *dog = p.dout.ptr + b * p.dout.sb + h * p.dout.sh;
        for (int x = tid; x < 32 * PPR; x += 512) {
            const int row = x / PPR, col = (x % PPR) * 16;
            int ii = i0 + row;
            ii = ii < N ? ii : N - 1;
            // q unpacked and scaled once per workgroup (the operand build of every offset and the dK2 rows multiply by it)
            const u32x4 fq = ld_global16(qg + (int64_t)ii * p.q.sn + col);
            const float c2 = p.scale_log2e;
            float4 *qdst = reinterpret_cast<float4 *>(lds + C::QS + row * C::QPITCH + col * 2);
            qdst[0] = make_float4(bf16_lo(fq[0]) * c2, bf16_hi(fq[0]) * c2, bf16_lo(fq[1]) * c2, bf16_hi(fq[1]) * c2);
            qdst[1] = make_float4(bf16_lo(fq[2]) * c2, bf16_hi(fq[2]) * c2, bf16_lo(fq[3]) * c2, bf16_hi(fq[3]) * c2);
            const u32x4 fd = ld_global16(dog + (int64_t)ii * p.dout.sn + col);
            *reinterpret_cast<u32x4 *>(lds + C::DOS + row * PITCH + col) = fd;
            if constexpr (DQ && SPLIT) {
                const u32x4 fo = ld_global16(p.o.ptr + b * p.o.sb + (int64_t)ii * p.o.sn + h * p.o.sh + col);
                const float part = delta_piece(fo, fd, p.o_lo.ptr ? p.o_lo.ptr + b * p.o_lo.sb + (int64_t)ii * p.o_lo.sn + h * p.o_lo.sh + col : nullptr);
                const float dsum = delta_row_sum<PPR>(part);
                if (col == 0) {
                    delta_s[row] = dsum;
                    if (split == 0 && i0 + row < N) p.delta[((int64_t)b * p.H + h) * N + i0 + row] = dsum;
                }
            }
        }
        for (int x = tid; x < 39 * PPR; x += 512) {
            const int row = x / PPR, col = (x % PPR) * 16;
            int kk2 = i0 - 7 - 8 * r_first + row;
            kk2 = kk2 < 0 ? 0 : (kk2 < N ? kk2 : N - 1);
            const int slot = (row - 7 - 8 * r_first) & 63;
            *reinterpret_cast<u32x4 *>(lds + C::K2S + slot * PITCH + col) = ld_global16(k2g + (int64_t)kk2 * p.k2.sn + col);
            if constexpr (DQ)
                *reinterpret_cast<u32x4 *>(lds + C::V2S + slot * PITCH + col) = ld_global16(v2g + (int64_t)kk2 * p.v2.sn + col);
        }
    }
    // additive masks: table 0 for the diagonal tile, tables 1, 2 for the tiles the lower window edge
    // crosses.  Entry (lane, rr) is 0 if query row i0 + c attends key row 32 t + 4 hf + e(rr), else -inf
    for (int x = tid; x < 3 * 256; x += 512) {
        const int tab = x >> 8, qq = (x >> 6) & 3, ln = x & 63;
        const int t = tab == 0 ? t_hi : t_lo + tab - 1;
        const int rel = (ln & 31) + 32 * (t_hi - t) - 4 * (ln >> 5);
        float4 m4;
        float *mp = &m4.x;
#pragma unroll
        for (int e = 0; e < 4; ++e) mp[e] = ((unsigned)(rel - (8 * qq + e)) < (unsigned)p.w1) ? 0.f : -INFINITY;
        *reinterpret_cast<float4 *>(lds + C::MASKS + tab * C::MASK + qq * 1024 + ln * 16) = m4;
    }
    // the 8 k2 (and v2) rows that round r + 1 adds (k - i0 = -8r - 15 .. -8r - 8), one 16-byte piece per thread
    const bool row_stager = tid < (DQ ? 2 : 1) * 8 * PPR;
    const int rs_sel = tid / (8 * PPR), rs_row = (tid / PPR) % 8, rs_col = (tid % PPR) * 16;
    u32x4 st_r = {0u, 0u, 0u, 0u};
    auto issue_rows = [&](int r) {
        if (row_stager) {
            int kk2 = i0 - 8 * r - 15 + rs_row;
            kk2 = kk2 < 0 ? 0 : (kk2 < N ? kk2 : N - 1);
            st_r = ld_global16((rs_sel ? v2g + (int64_t)kk2 * p.v2.sn : k2g + (int64_t)kk2 * p.k2.sn) + rs_col);
        }
    };
    auto write_rows = [&](int r) {
        if (row_stager) {
            const int slot = (-8 * r - 15 + rs_row) & 63;
            *reinterpret_cast<u32x4 *>(lds + (rs_sel ? C::V2S : C::K2S) + slot * PITCH + rs_col) = st_r;
        }
    };
    // scatter rows of this tile in the workspace: row x <-> k = i0 - halo + x
    const int srows = 32 + halo;
    const int64_t per_tensor = (int64_t)p.B * p.H * ntile * srows * D;
    float *wk = ws + split * p.q_ws_stride + (DQ ? 0 : per_tensor) + (((int64_t)b * p.H + h) * ntile + tile) * srows * D;
    // rows k - i0 = lo .. lo + n - 1 of the circular buffer go to the workspace and are cleared for reuse
    auto flush_rows = [&](int lo, int n) {
        for (int x = tid; x < n * (D / 4); x += 512) {
            const int rel = lo + x / (D / 4), col = (x % (D / 4)) * 4;
            float4 *src = reinterpret_cast<float4 *>(sc + ((rel & 63) * C::SPITCH + col));
            *reinterpret_cast<float4 *>(wk + (int64_t)(rel + halo) * D + col) = *src;
            *src = make_float4(0.f, 0.f, 0.f, 0.f);
        }
    };

    // ring protocol: step u lives in buffer u & 1.  Its transfer starts behind the barrier of step u - 1 (every
    // wave has then finished step u - 2, the last reader of that buffer) and is awaited before the barrier of step u.
    issue_loads();
    int u = 0;
    auto open_step = [&]() {
        if (stager) wait_loads<0>();
        __syncthreads();
        issue_loads();
    };

    f32x16 acc[DT];            // G^T (DQ) or T^T (DV) of the running offset
    u32x4 A[KS];
    u32x4 Bv[DQ ? KS : 1];

    __syncthreads();
    if constexpr (DQ && SPLIT) dl = delta_s[c];
    const f32x16 neg_delta = splat16(-dl);      // DQ: -delta_i in every element (one query row per lane column)
    for (int r = r_first; r < R; ++r) {
        const int dlt = 8 * r + wave;
        const int kr = i - dlt;
        const bool col_ok = row_ok && kr >= 0 && dlt < p.w2;
        const bool wave_on = wave_any(col_ok);
        const int slot = (c - dlt) & 63;              // slot of row k = i - dlt in the circular rows
        {
            const char *qr = lds + C::QS + c * C::QPITCH + 32 * hf;
            const char *k2r = lds + C::K2S + slot * PITCH + 16 * hf;
#pragma unroll
            for (int kk = 0; kk < KS; ++kk) {
                const float4 qa = *reinterpret_cast<const float4 *>(qr + 64 * kk), qb = *reinterpret_cast<const float4 *>(qr + 64 * kk + 16);
                const u32x4 fk = ld_lds16(k2r + 32 * kk);
                A[kk][0] = pack_bf16(qa.x * bf16_lo(fk[0]), qa.y * bf16_hi(fk[0]));
                A[kk][1] = pack_bf16(qa.z * bf16_lo(fk[1]), qa.w * bf16_hi(fk[1]));
                A[kk][2] = pack_bf16(qb.x * bf16_lo(fk[2]), qb.y * bf16_hi(fk[2]));
                A[kk][3] = pack_bf16(qb.z * bf16_lo(fk[3]), qb.w * bf16_hi(fk[3]));
            }
            if constexpr (DQ) {
                const char *dor = lds + C::DOS + c * PITCH + 16 * hf;
                const char *v2r = lds + C::V2S + slot * PITCH + 16 * hf;
#pragma unroll
                for (int kk = 0; kk < KS; ++kk) Bv[kk] = mul_bf16x8(ld_lds16(dor + 32 * kk), ld_lds16(v2r + 32 * kk));
            }
#pragma unroll
            for (int dt = 0; dt < DT; ++dt) acc[dt] = zero16_pairs();
        }
        const float nl = col_ok ? -lse2 : -INFINITY;  // where the logit chains start
        const f32x2 nl2 = {nl, nl};
        f32x16 nl_reg;                                // (KEEP_NL)
        if constexpr (KEEP_NL) nl_reg = splat16(nl);

        for (int n = 0; n < NT; ++n) {
            open_step();
            if (wave_on) {
                const char *sub = lds + (u & 1) * C::BUF;
                const int t = t_lo + n;
                // The operand fragments of the step form one stream: the K1 row fragments of the logit chain, (DQ) the
                // V1 row fragments of the dP chain, then the transposed fragments of the accumulating products.  A
                // window of W fragments is kept in flight: behind every MFMA the fragment W places further down the
                // stream is requested (a scheduling fence keeps it there), so a read has W MFMAs of time to
                // arrive and no chain waits for LDS.
                constexpr int W = 4;
                constexpr int NROW = DQ ? 2 * KS : KS;          // row fragments
                constexpr int NFR = NROW + 2 * DT;              // ... and transposed ones
                const char *kb = sub + r_lane, *vb = sub + C::OFF_V + r_lane;
                const char *tb = sub + (DQ ? 0 : C::OFF_V) + t_lane;      // DQ: G^T += K1^T dS^T;  DV: T^T += V1^T P^T
                auto fragment = [&](auto idx) {
                    constexpr int s = decltype(idx)::value;
                    if constexpr (s < KS) return RT::row_frag(kb, s);
                    else if constexpr (s < NROW) return RT::row_frag(vb, s - KS);
                    else return RT::tr_frag(tb, (s - NROW) / DT, (s - NROW) % DT);
                };
                // (the step's first fragment reads are requested first: the start values of the chains are then set up
                // while they are in flight, not in front of them)
                u32x4 f[W];
                static_for<0, (W < NFR ? W : NFR)>([&](auto s) { f[s] = fragment(s); });
                f32x16 X;
                if constexpr (!KEEP_NL) X = splat16_pairs(nl2);
                const bool masked = t == t_hi || n < n_head;
                if (masked) {
                    if constexpr (KEEP_NL) X = nl_reg;
                    const char *mk = lds + C::MASKS + (t == t_hi ? 0 : 1 + n) * C::MASK + lane * 16;
#pragma unroll
                    for (int qq = 0; qq < 4; ++qq) {
                        const float4 m4 = *reinterpret_cast<const float4 *>(mk + qq * 1024);
                        X[4 * qq] += m4.x;
                        X[4 * qq + 1] += m4.y;
                        X[4 * qq + 2] += m4.z;
                        X[4 * qq + 3] += m4.w;
                    }
                }
                if constexpr (KEEP_NL) {
                    // (the first product in both branches: an unmasked one takes the start values from where they are)
                    if (masked) X = mfma32(f[0], A[0], X);
                    else X = mfma32(f[0], A[0], nl_reg);
                }
                f32x16 dP = neg_delta;      // DQ: the chain starts from -delta_i, so dP - delta costs no VALU work
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, NROW>([&](auto sc_) {
                    constexpr int s = decltype(sc_)::value;
                    if constexpr (s < KS) {
                        if constexpr (s > 0 || !KEEP_NL) X = mfma32(f[s % W], A[s], X);
                    }
                    else dP = mfma32(f[s % W], Bv[DQ ? s - KS : 0], dP);
                    if constexpr (s + W < NFR) f[s % W] = fragment(std::integral_constant<int, s + W>{});
                    __builtin_amdgcn_sched_barrier(0);
                });
                // weights of the first 16 tile rows, their products, the weights of the other 16 rows between them
                u32x4 pb[2];
                auto weights = [&](int rr) {
                    float p0 = fast_exp2(X[rr]), p1 = fast_exp2(X[rr + 1]);
                    if constexpr (DQ) {
                        p0 *= dP[rr];
                        p1 *= dP[rr + 1];
                    }
                    pb[rr >> 3][(rr & 7) >> 1] = pack_bf16(p0, p1);
                };
#pragma unroll
                for (int rr = 0; rr < 8; rr += 2) weights(rr);
                __builtin_amdgcn_sched_barrier(0);
                static_for<0, 2 * DT>([&](auto sc_) {
                    constexpr int s = decltype(sc_)::value;     // k2s = s / DT, dt = s % DT
                    acc[s % DT] = mfma32(f[(NROW + s) % W], pb[s / DT], acc[s % DT]);
                    if constexpr (NROW + s + W < NFR) f[(NROW + s) % W] = fragment(std::integral_constant<int, NROW + s + W>{});
                    if constexpr (s < DT) {
                        // (four pairs of weights behind the first DT MFMAs)
#pragma unroll
                        for (int x = 4 * s / DT; x < 4 * (s + 1) / DT; ++x) weights(8 + 2 * x);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                });
            }
            ++u;
        }

        // ---- round end: add into the shared fp32 rows, one d-slice per wave and phase
        {
            if (r + 1 < R) issue_rows(r);      // the rows that the next round adds arrive behind the phases below
            // factor of the scattered rows: DQ the fp32 q rows (times scale log2(e): the combine kernel multiplies by ln 2), DV the dO rows
            const char *qr = DQ ? lds + C::QS + c * C::QPITCH + 16 * hf * 4 : lds + C::DOS + c * PITCH + 16 * hf * 2;
            const char *k2r = lds + C::K2S + slot * PITCH + 16 * hf * 2;
            float *srow_p = sc + slot * C::SPITCH + 16 * hf;
            float *drow_p = dqs + c * C::SPITCH + 16 * hf;
            auto add_slice = [&](auto slice_tag) {
                constexpr int S = decltype(slice_tag)::value;     // slice: dt = S / 2, registers 8*(S%2) .. +7
                constexpr int dt = S >> 1, r0 = 8 * (S & 1);
                float4 x0, x1;
                if constexpr (DQ) {
                    x0 = *reinterpret_cast<const float4 *>(qr + (32 * dt + r0) * 4);
                    x1 = *reinterpret_cast<const float4 *>(qr + (32 * dt + r0) * 4 + 16);
                } else {
                    const u32x4 xq = ld_lds16(qr + dt * 64 + r0 * 2);
                    x0 = make_float4(bf16_lo(xq[0]), bf16_hi(xq[0]), bf16_lo(xq[1]), bf16_hi(xq[1]));
                    x1 = make_float4(bf16_lo(xq[2]), bf16_hi(xq[2]), bf16_lo(xq[3]), bf16_hi(xq[3]));
                }
                float *dst = srow_p + 32 * dt + r0;
                float4 a0 = *reinterpret_cast<float4 *>(dst), a1 = *reinterpret_cast<float4 *>(dst + 4);
                a0.x += x0.x * acc[dt][r0];
                a0.y += x0.y * acc[dt][r0 + 1];
                a0.z += x0.z * acc[dt][r0 + 2];
                a0.w += x0.w * acc[dt][r0 + 3];
                a1.x += x1.x * acc[dt][r0 + 4];
                a1.y += x1.y * acc[dt][r0 + 5];
                a1.z += x1.z * acc[dt][r0 + 6];
                a1.w += x1.w * acc[dt][r0 + 7];
                *reinterpret_cast<float4 *>(dst) = a0;
                *reinterpret_cast<float4 *>(dst + 4) = a1;
                if constexpr (DQ) {
                    const u32x4 xk = ld_lds16(k2r + dt * 64 + r0 * 2);
                    float *dd = drow_p + 32 * dt + r0;
                    float4 b0 = *reinterpret_cast<float4 *>(dd), b1 = *reinterpret_cast<float4 *>(dd + 4);
                    b0.x += bf16_lo(xk[0]) * acc[dt][r0];
                    b0.y += bf16_hi(xk[0]) * acc[dt][r0 + 1];
                    b0.z += bf16_lo(xk[1]) * acc[dt][r0 + 2];
                    b0.w += bf16_hi(xk[1]) * acc[dt][r0 + 3];
                    b1.x += bf16_lo(xk[2]) * acc[dt][r0 + 4];
                    b1.y += bf16_hi(xk[2]) * acc[dt][r0 + 5];
                    b1.z += bf16_lo(xk[3]) * acc[dt][r0 + 6];
                    b1.w += bf16_hi(xk[3]) * acc[dt][r0 + 7];
                    *reinterpret_cast<float4 *>(dd) = b0;
                    *reinterpret_cast<float4 *>(dd + 4) = b1;
                }
            };
            auto add_slice_of = [&](auto slice_tag) {     // (CH < D: nothing to add to the slices of the zero channels)
                if constexpr (decltype(slice_tag)::value < 2 * DT) add_slice(slice_tag);
            };
            for (int ph = 0; ph < 8; ++ph) {
                // D / 16 slices: the waves form 8 / (D / 16) groups that take turns, group g owns the phases D / 16 g ..
                // D / 16 g + D / 16 - 1 (D = 128: one group, every wave works in every phase)
                constexpr int SL = D / 16;
                if (SL == 8 || ph / SL == wave / SL) with_slice<SL>(wave + ph, add_slice_of);
                if (ph == 7 && r + 1 < R) write_rows(r);    // (their slots are not in use in this round)
                __syncthreads();
            }
            // the rows k - i0 = 24 - 8r .. 31 - 8r are complete: no later round reaches them
            if (r + 1 < R) flush_rows(24 - 8 * r, 8);
        }
    }
    wait_loads<0>();           // (the transfer issued behind the last tile still writes into the ring)
    // ---- the rows that the last round leaves: k - i0 = -8 (R - 1) - 7 .. 31 - 8 (R - 1)
    flush_rows(-8 * (R - 1) - 7, 39);

    // ---- dq rows to global memory (bf16, scaled)
    if constexpr (DQ) {
        constexpr int SEG = D / 16;
        const int row = tid >> 4, seg = tid & 15;
        const int ir = i0 + row;
        if (ir < N) {
            const float *src = dqs + row * C::SPITCH + seg * SEG;
            if constexpr (SPLIT) {
                float *dst = p.q_parts + ((((int64_t)split * p.B + b) * p.H + h) * N + ir) * D + seg * SEG;
#pragma unroll
                for (int x = 0; x < SEG; x += 2) *reinterpret_cast<float2 *>(dst + x) = *reinterpret_cast<const float2 *>(src + x);
                return;
            }
            char *orow = p.dq.ptr + b * p.dq.sb + (int64_t)ir * p.dq.sn + h * p.dq.sh + seg * SEG * 2;
            if constexpr (SEG == 8) {
                float4 a = *reinterpret_cast<const float4 *>(src);
                float4 bq = *reinterpret_cast<const float4 *>(src + 4);
                u32x4 ov = {pack_bf16(a.x * p.scale, a.y * p.scale), pack_bf16(a.z * p.scale, a.w * p.scale),
                            pack_bf16(bq.x * p.scale, bq.y * p.scale), pack_bf16(bq.z * p.scale, bq.w * p.scale)};
                st_global16(orow, ov);
            } else if constexpr (SEG == 4) {
                float4 a = *reinterpret_cast<const float4 *>(src);
                u32x2 ov = {pack_bf16(a.x * p.scale, a.y * p.scale), pack_bf16(a.z * p.scale, a.w * p.scale)};
                *reinterpret_cast<u32x2 *>(orow) = ov;
            } else {
                static_assert(SEG == 2, "head dimension 32, 64 or 128");
                float2 a = *reinterpret_cast<const float2 *>(src);
                *reinterpret_cast<uint32_t *>(orow) = pack_bf16(a.x * p.scale, a.y * p.scale);
            }
        }
    }
}

// dV2 from the forward's saved per-offset T:
//     dv2[b,k,hk,:] = sum_g sum_dlt do[b,k+dlt,h,:] * T[b,h,dlt,k+dlt,:] * 2^(m[b,h,dlt,k+dlt] - lse2[b,h,k+dlt])
// (h = hk*G + g).  Streams T once from HBM.  A workgroup owns 32 rows k, a thread 8 d of one row; consecutive
// threads own consecutive rows, whose pieces are consecutive in the blocked layout of T (saved_t_offset).  The do
// rows k0 .. k0 + 62 that 32 offsets reach and the 32 x 32 weights are staged in LDS per block of 32 offsets.
// GROUPS (small_grid_merge_kernel): at D = 32 and 64 the threads of a workgroup form OG groups that take every OG-th offset and meet
// through LDS.  The loop over the offsets is a chain of loads, which few workgroups do not hide; a large grid does
// and loses by the larger workgroups (152 us instead of 130 at 8 x 8 x 2048 rows of 64).
template <int D, bool GROUPS>
struct Dv2Cfg {
    static constexpr int LP = D / 8;                 // 16-byte pieces per row
    static constexpr int OG = GROUPS ? 16 / LP : 1;  // offset groups
    static constexpr int THREADS = 32 * LP * OG;
    static constexpr int PITCH = tile_pitch<D>();
};

template <int D, bool GROUPS>
__device__ __forceinline__ void dv2_from_saved_block(const KParams &p, const int block) {
    using C = Dv2Cfg<D, GROUPS>;
    constexpr int LP = C::LP, NTH = C::THREADS, PITCH = C::PITCH, OG = C::OG;
    __shared__ __attribute__((aligned(16))) char dos[63 * PITCH];
    __shared__ float wsh[32 * 32];
    __shared__ float4 red[OG > 1 ? (OG - 1) * 32 * LP * 2 : 1];
    const int N = p.N;
    const int ntile = (N + 31) / 32;
    const int kt = block % ntile;
    const int bh = block / ntile;
    const int hk = bh % p.HK, b = bh / p.HK;
    const int tid = threadIdx.x;
    const int og = GROUPS ? tid / (32 * LP) : 0, t_in = GROUPS ? tid % (32 * LP) : tid;
    const int c = t_in & 31, piece = t_in >> 5;       // d = 8 piece .. 8 piece + 7
    const int k0 = 32 * kt, k = k0 + c;
    const int t_piece = saved_t_offset(0, (piece >> 1) & 1, piece >> 2, piece & 1);
    float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
    const int nd = p.w2 < N - k0 ? p.w2 : N - k0;     // offsets that reach a row of the sequence from row k0
    for (int g = 0; g < p.G; ++g) {
        const int h = hk * p.G + g;
        const int64_t bh_row = ((int64_t)b * p.H + h);
        const char *dog = p.dout.ptr + b * p.dout.sb + h * p.dout.sh;
        const float *lse = p.lse + bh_row * N;
        for (int d0 = 0; d0 < nd; d0 += 32) {
            // (rows past the end have weight 0; their T is read from the last row, which every offset has written)
            auto t_of = [&](int dl) {
                const int i = k + d0 + dl < N ? k + d0 + dl : N - 1;
                const int64_t sbh = bh_row * p.w2 + d0 + dl;
                return ld_global16(p.t_save + (sbh * ntile + (i >> 5)) * saved_t_block<D>() + t_piece + (i & 31) * 16);
            };
            const int nl = nd - d0 < 32 ? nd - d0 : 32;
            // GROUPS: the first eight T pieces of the block are requested in front of the staging, whose latency they then share
            // (offsets past the last one are read from it and not used)
            u32x4 ahead[GROUPS ? 8 : 1];
            auto request = [&](int x0) {
#pragma unroll
                for (int x = 0; x < 8; ++x) ahead[GROUPS ? x : 0] = t_of(og + (x0 + x) * OG < nl ? og + (x0 + x) * OG : nl - 1);
            };
            if constexpr (GROUPS) request(0);
            __syncthreads();
            for (int x = tid; x < 63 * LP; x += NTH) {
                const int row = x / LP, pc = x % LP;
                int i = k0 + d0 + row;
                i = i < N ? i : N - 1;
                *reinterpret_cast<u32x4 *>(dos + row * PITCH + pc * 16) = ld_global16(dog + (int64_t)i * p.dout.sn + pc * 16);
            }
            for (int x = tid; x < 32 * 32; x += NTH) {
                const int dl = x >> 5, dlt = d0 + dl, i = k0 + dlt + (x & 31);
                float w = 0.f;
                if (dlt < p.w2 && i < N) w = fast_exp2(p.m_save[(bh_row * p.w2 + dlt) * N + i] - lse[i] * kLog2e);
                wsh[x] = w;
            }
            __syncthreads();
            auto add = [&](int dl, const u32x4 &t) {
                const u32x4 o = ld_lds16(dos + (c + dl) * PITCH + piece * 16);
                const float w = wsh[dl * 32 + c];
#pragma unroll
                for (int x = 0; x < 4; ++x) {
                    acc[2 * x] += bf16_lo(o[x]) * bf16_lo(t[x]) * w;
                    acc[2 * x + 1] += bf16_hi(o[x]) * bf16_hi(t[x]) * w;
                }
            };
            if constexpr (GROUPS) {
#pragma unroll
                for (int x0 = 0; x0 < 32 / OG; x0 += 8) {
                    if (x0 > 0) {
                        if (x0 * OG >= nl) break;         // (D = 64, up to 16 offsets: there are no second eight)
                        request(x0);
                    }
#pragma unroll
                    for (int x = 0; x < 8; ++x)
                        if (og + (x0 + x) * OG < nl) add(og + (x0 + x) * OG, ahead[x]);
                }
            } else {
#pragma unroll 8
                for (int dl = 0; dl < nl; ++dl) add(dl, t_of(dl));
            }
        }
    }
    if constexpr (OG > 1) {
        if (og > 0) {
            float4 *dst = red + ((og - 1) * 32 * LP + t_in) * 2;
            dst[0] = make_float4(acc[0], acc[1], acc[2], acc[3]);
            dst[1] = make_float4(acc[4], acc[5], acc[6], acc[7]);
        }
        __syncthreads();
        if (og > 0) return;
#pragma unroll
        for (int x = 0; x < OG - 1; ++x) {
            const float4 a = red[(x * 32 * LP + t_in) * 2], e = red[(x * 32 * LP + t_in) * 2 + 1];
            acc[0] += a.x;
            acc[1] += a.y;
            acc[2] += a.z;
            acc[3] += a.w;
            acc[4] += e.x;
            acc[5] += e.y;
            acc[6] += e.z;
            acc[7] += e.w;
        }
    }
    if (k >= N) return;
    u32x4 r = {pack_bf16(acc[0], acc[1]), pack_bf16(acc[2], acc[3]), pack_bf16(acc[4], acc[5]), pack_bf16(acc[6], acc[7])};
    st_global16(p.dv2.ptr + b * p.dv2.sb + (int64_t)k * p.dv2.sn + hk * p.dv2.sh + piece * 16, r);
}

template <int D>
__global__ __launch_bounds__((Dv2Cfg<D, false>::THREADS)) void dv2_from_saved_kernel(KParams p) {
    dv2_from_saved_block<D, false>(p, blockIdx.x);
}

// dK2 / dV2 from the partial rows of the workspace: sums the tiles that reach a row and the query heads of a group.
// Workspace rows of a tile with first query row i0: index x <-> k = i0 - halo + x, so
// rows 0..halo-1 are the halo below the tile and rows halo..halo+31 its own rows.
// With split query tiles (p.q_splits > 1) the shares of a tile are added in split order (a share has written the rows its
// rounds reach, k - i0 = -8 R + 1 .. 31 - 8 r_first); dq_from_shares forms dq from the shares' fp32 rows.  One chain of sums per
// element, whichever kernel runs it: dK2 has the same bits with saved partials and without.
template <int D, int NTH>
__device__ __forceinline__ void combine_rows(const KParams &p, const float *ws, const int srows, const int with_dv2, const int block) {
    constexpr int LP = D / 8;   // threads per row, 8 d each
    const int N = p.N, ntile = (N + 31) / 32;
    const int halo = srows - 32;
    const int piece = threadIdx.x % LP;
    const int64_t row = (int64_t)block * (NTH / LP) + threadIdx.x / LP;
    const int64_t rows = (int64_t)p.B * p.HK * N;
    if (row >= rows) return;
    const int k = (int)(row % N);
    const int hk = (int)((row / N) % p.HK);
    const int b = (int)(row / ((int64_t)N * p.HK));
    const int tile = k / 32, kl = k % 32;
    const int64_t per_tensor = (int64_t)p.B * p.H * ntile * srows * D;
    float ak[8], av[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) ak[x] = av[x] = 0.f;
    for (int g = 0; g < p.G; ++g) {
        const int h = hk * p.G + g;
        const float *base = ws + (((int64_t)b * p.H + h) * ntile) * srows * D;
        for (int m = 0; tile + m < ntile && kl + halo - 32 * m >= 0; ++m) {
            const float *src = base + ((int64_t)(tile + m) * srows + (kl + halo - 32 * m)) * D + piece * 8;
            if (p.q_splits > 1) {
                // the shares whose rounds r0 .. r1 - 1 reach the row: 1 - 8 r1 <= rel <= 31 - 8 r0
                const int rounds = fwd_rounds(tile + m, p.w2), rel = kl - 32 * m;
                const int r_lo = rel >= 0 ? 0 : (-rel) / 8, r_hi = (31 - rel) / 8;        // rounds that reach it
                int s = fwd_split_of(r_lo, p.q_splits, rounds);
                for (int r0 = fwd_split_round(s, p.q_splits, rounds), r1; s < p.q_splits; ++s, r0 = r1) {
                    r1 = fwd_split_round(s + 1, p.q_splits, rounds);
                    if (r0 >= r1 || r0 > r_hi) break;
                    if (rel < 1 - 8 * r1) continue;
                    const float *ss = src + s * p.q_ws_stride;
#pragma unroll
                    for (int x = 0; x < 8; ++x) {
                        ak[x] += ss[x];
                        if (with_dv2) av[x] += ss[per_tensor + x];
                    }
                }
                continue;
            }
#pragma unroll
            for (int x = 0; x < 8; ++x) {
                ak[x] += src[x];
                if (with_dv2) av[x] += src[per_tensor + x];
            }
        }
    }
    u32x4 ok, ov;
#pragma unroll
    for (int w = 0; w < 4; ++w) {
        ok[w] = pack_bf16(ak[2 * w] * kLn2, ak[2 * w + 1] * kLn2);   // the partial rows carry q * scale * log2(e)
        ov[w] = pack_bf16(av[2 * w], av[2 * w + 1]);
    }
    st_global16(p.dk2.ptr + b * p.dk2.sb + (int64_t)k * p.dk2.sn + hk * p.dk2.sh + piece * 16, ok);
    if (with_dv2) st_global16(p.dv2.ptr + b * p.dv2.sb + (int64_t)k * p.dv2.sn + hk * p.dv2.sh + piece * 16, ov);
}

// dq from the fp32 rows that the shares of split query tiles leave
template <int D, int NTH>
__device__ __forceinline__ void dq_from_shares(const KParams &p, const int block) {
    constexpr int LP = D / 8;
    const int N = p.N, piece = threadIdx.x % LP;
    const int64_t row = (int64_t)block * (NTH / LP) + threadIdx.x / LP;
    const int64_t rows = (int64_t)p.B * p.H * N;
    if (row >= rows) return;
    const int i = (int)(row % N), h = (int)((row / N) % p.H), b = (int)(row / ((int64_t)N * p.H));
    const int rounds = fwd_rounds(i / 32, p.w2);
    const int splits = p.q_splits < rounds ? p.q_splits : rounds;
    float a[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll 4
    for (int s = 0; s < splits; ++s) {
        const float *src = p.q_parts + (s * rows + row) * D + piece * 8;
#pragma unroll
        for (int x = 0; x < 8; ++x) a[x] += src[x];
    }
    u32x4 o;
#pragma unroll
    for (int w = 0; w < 4; ++w) o[w] = pack_bf16(a[2 * w] * p.scale, a[2 * w + 1] * p.scale);
    st_global16(p.dq.ptr + b * p.dq.sb + (int64_t)i * p.dq.sn + h * p.dq.sh + piece * 16, o);
}

// (grid row 1, with split query tiles: dq)
template <int D>
__global__ __launch_bounds__(256) void dk2_dv2_combine_kernel(KParams p, const float *ws, int srows, int with_dv2) {
    if (blockIdx.y == 1) dq_from_shares<D, 256>(p, blockIdx.x);
    else combine_rows<D, 256>(p, ws, srows, with_dv2, blockIdx.x);
}

// Small grids with saved forward partials: dV2, dK2 and, of split query tiles, dQ in one launch.  Blocks 0 .. dv2_blocks - 1 form dV2,
// the next dk2_blocks dK2, the rest dQ.  Each is a chain of dependent loads in a few workgroups, so one behind the other they cost
// the sum of their latencies, side by side the longest.  As two launches; as one; as one with the first T pieces of dV2 requested
// ahead of the staging (GROUPS), in us between events around the launches (a kernel trace has 3 us less for the last of each): 1 x 4 x 128
// rows of 32, w2 128: 40.9, 22.7, 15.9; 1 x 8 (4 kv) x 1000 rows of 64, w2 32: 27.5, 20.7, 16.9; 2 x 6 (2 kv) x 2999 rows of 128, w2 20
// (nothing ahead at D = 128): 71, 54.  (dK2's shares dealt out to four groups of threads that meet through LDS: 15.9, 16.9, 58, and
// 30.0 instead of 22.5 at 1 x 16 (4 kv) x 4096 rows of 64, w2 2.)
template <int D>
struct MergeCfg {
    static constexpr int THREADS = 512, ROWS = THREADS / (D / 8);      // rows of dK2 or dQ per block
    static_assert(Dv2Cfg<D, (D < 128)>::THREADS == THREADS, "one block size");
};
template <int D>
__global__ __launch_bounds__(512) void small_grid_merge_kernel(KParams p, const float *ws, int srows, int dv2_blocks, int dk2_blocks) {
    using C = MergeCfg<D>;
    const int x = blockIdx.x;
    if (x < dv2_blocks) dv2_from_saved_block<D, (D < 128)>(p, x);
    else if (x < dv2_blocks + dk2_blocks) combine_rows<D, C::THREADS>(p, ws, srows, 0, x - dv2_blocks);
    else dq_from_shares<D, C::THREADS>(p, x - dv2_blocks - dk2_blocks);
}

}  // namespace sa2
