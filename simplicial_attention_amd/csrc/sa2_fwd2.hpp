// Forward kernel in which a wave owns two offsets: four waves per workgroup, every K1/V1 fragment feeds two MFMAs.
//
// One workgroup owns 32 query rows of one (batch, head).  In round r wave w handles the offsets dlt = i - k = 8 r + 2 w and
// 8 r + 2 w + 1; the waves walk the same 32-row K1/V1 tiles, which stream through LDS rings (direct-to-LDS loads, layout DmaTile
// of sa2_lds.hpp), one tile and one barrier per step.  Per (offset, tile), as in fwd_kernel (sa2_fwd.hpp):
//     S^T = K1 A^T,  A = q_i * k2_{i-dlt} * scale * log2(e),   P^T = exp2(S^T - M_i),   T^T += V1^T P^T
// and per round, in registers:  O_i += v2_{i-dlt} * T  for both offsets.
//
// What bounded the eight-wave form (one offset per wave, an output accumulator in LDS): neither the MFMA pipe (46 % busy at
// D = 128) nor the VALU (46 %) nor LDS (32 %) but the lockstep of its waves and the ends of its rounds (nine barriers each, a
// quarter of the time).  Here
//   - a fragment read from LDS is used twice, so there are half as many of them;
//   - the output sum is the wave's own: nothing is shared between the waves but the tiles, and they meet once, at the end;
//   - a wave overlaps its own work: the exponentials of tile u are issued behind the single MFMAs of the value products of
//     tile u - 1 (a scheduling fence behind each), fragments run through rolling windows, the first ones of a step are
//     requested before its barrier.
// That takes about 450 registers: one wave per SIMD.  4 x 8 x 8192 rows, w1 512, w2 32: 2.39 -> 2.23 ms.
// A microbenchmark of the mix (4 fma, 1 exp2, 1 LDS fragment per MFMA) runs at 21-24 ns per MFMA with one wave per SIMD as with
// two: the second wave is not needed to fill the pipe, registers are worth more.
//
// Registers: the operands A are placed in accumulation registers by hand (pin_agpr), everything else is left to the
// compiler, which is told to keep MFMA results in ordinary registers (-amdgpu-mfma-vgpr-form: the VALU reads the logits at
// once; left to itself it puts the results of every MFMA of a kernel of this size in accumulation registers and moves the
// logits).  A row's
// softmax reference M is fixed by the wave's first tile (the diagonal one, which every valid row attends).  Where a row sum
// says at the end that weights outgrew 2^90 (rare), the workgroup walks its rounds twice more: once for the largest logits of
// the rows, once for the result.  Lanes without a valid key row (k < 0, a row beyond the sequence) compute on clamped rows;
// their sums are never taken.
#pragma once

#include "sa2_acc.hpp"
#include "sa2_common.hpp"
#include "sa2_fwd.hpp"
#include "sa2_lds.hpp"

namespace sa2 {

template <int D>
struct Fwd2Cfg {
    static_assert(D == 128, "at D = 64 and 32 two eight-wave workgroups per CU are faster (612 us, this form 710 us, at 8 x 8 x 2048 rows of 64)");
    static constexpr int KS = D / 16;
    static constexpr int DT = D / 32;
    static constexpr int PITCH = tile_pitch<D>();     // staged q / k2 / v2 rows
    using RT = DmaTile<D>;
    static constexpr int TB = RT::BYTES;
    // rings: K1 tile u + 1 is published with barrier u, V1 tile u with it (its products run in step u + 1, at the latest), tiles
    // u + 3 and u + 2 are being loaded
    static constexpr int NBUF = 4;
    static constexpr int VRING = NBUF * TB;
    static constexpr int RING = 2 * NBUF * TB;
    static_assert(RING - RT::CP < 65536, "the LDS address of a direct load travels in 16 bits of M0");
    static constexpr int LPW = RT::NCH / 2;           // loads per wave and step
    static constexpr int QS = RING;                   // q rows as fp32 times scale log2(e)
    static constexpr int QPITCH = D * 4 + 16;
    static constexpr int K2S = QS + 32 * QPITCH;      // 64-row circular buffers, row k in slot (k - i0) mod 64
    static constexpr int V2S = K2S + 64 * PITCH;
    static constexpr int MASKS = V2S + 64 * PITCH;    // additive masks (0 / -inf) of the diagonal tile and of up to two lower-edge tiles
    static constexpr int MASK = 16 * 64 * 4;
    static constexpr int VOTE = MASKS + 3 * MASK;     // one word per wave
    static constexpr int MAIN = VOTE + 16;
    // the waves' merge: [4][32][D + 4] fp32 rows, references and row sums
    static constexpr int APITCH = D + 4;
    static constexpr int XM = 4 * 32 * APITCH * 4;
    static constexpr int MERGE = XM + 2 * 4 * 32 * 4;
    static constexpr int LDS = MAIN > MERGE ? MAIN : MERGE;
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
    static constexpr int PPR = D / 8;                 // 16-byte pieces per row
};

template <int D, bool SPLIT = false>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void fwd2_kernel(KParams p) {
    using C = Fwd2Cfg<D>;
    using RT = typename C::RT;
    constexpr int KS = C::KS, DT = C::DT, PPR = C::PPR, PITCH = C::PITCH;
    constexpr float kBig = 1.2379400392853803e27f;    // 2^90: row sums beyond it move the reference
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

    const char *k1g = p.k1.ptr + b * p.k1.sb + hk * p.k1.sh;
    const char *v1g = p.v1.ptr + b * p.v1.sb + hk * p.v1.sh;
    const char *k2g = p.k2.ptr + b * p.k2.sb + hk * p.k2.sh;
    const char *v2g = p.v2.ptr + b * p.v2.sb + hk * p.v2.sh;

    // tiles of the first window; sequence of a round: the diagonal tile first, then t_lo .. t_hi - 1
    const int t_lo = (i0 - p.w1 + 1 > 0 ? i0 - p.w1 + 1 : 0) / 32;
    const int t_hi = i0 / 32;
    const int NT = t_hi - t_lo + 1;
    int mid_lo = (i0 + 31 - p.w1 >= 0) ? (i0 + 31 - p.w1) / 32 + 1 : t_lo;   // first tile below the diagonal that no row masks
    mid_lo = mid_lo > t_hi ? t_hi : mid_lo;
    const int n_masked = 1 + (mid_lo - t_lo);         // leading steps of a round that need a mask (at most 3)

    // ---- ring staging: load l = wave + 4 x moves chunk l % NCH of the K1 (l < NCH) or of the V1 tile.  The two sequences of tiles
    // run on behind the last round (into buffers that no wave reads any more), so that every step issues and awaits the
    // same number of transfers; the kernel waits for the last ones before it ends.
    const uint32_t lds_base = (uint32_t)(uintptr_t)lds;
    const int st_col = RT::st_col(lane);
    constexpr int LPT = RT::NCH / 4;                  // loads per wave and tile (chunks wave and wave + 4)
    // Address = tile base (uniform) + this lane's row and column (32 bits); rows of the diagonal tile beyond the sequence are
    // replaced by its last one.  The bases are running pointers: the diagonal tile, then t_lo, t_lo + 1, ...
    struct Seq {
        const char *base, *diag, *low;
        int n;                                        // place in the round of the next tile
        uint32_t so[LPT], so_diag[LPT];
    };
    auto make_seq = [&](const char *g, int64_t sn) {
        Seq s;
        s.diag = g + (int64_t)(32 * t_hi) * sn;
        s.low = g + (int64_t)(32 * t_lo) * sn;
        s.base = s.diag;
        s.n = 0;
#pragma unroll
        for (int x = 0; x < LPT; ++x) {
            const int row = RT::st_row(wave, lane) + 4 * RT::RPC * x;
            s.so[x] = (uint32_t)(row * (int)sn + st_col);
            s.so_diag[x] = (uint32_t)((i0 + row < N ? row : N - 1 - i0) * (int)sn + st_col);
        }
        return s;
    };
    Seq sk = make_seq(k1g, p.k1.sn), sv = make_seq(v1g, p.v1.sn);
    // (the loop-carried places are kept on the scalar unit by hand: left to itself the compiler moves their arithmetic to the
    // VALU)
    auto issue_tile = [&](Seq &s, int64_t sn, int buf) {
        const int n = uniform(s.n);
        const char *base = uniform(s.base);
        const uint32_t dst = lds_base + buf + wave * RT::CP;
#pragma unroll
        for (int x = 0; x < LPT; ++x) load_to_lds16(base, n == 0 ? s.so_diag[x] : s.so[x], dst + 4 * x * RT::CP);
        const bool wrap = n == NT - 1;
        s.base = uniform(wrap ? s.diag : (n == 0 ? s.low : base + 32 * sn));
        s.n = uniform(wrap ? 0 : n + 1);
    };
    auto issue_k = [&](int buf) { issue_tile(sk, p.k1.sn, buf); };
    auto issue_v = [&](int buf) { issue_tile(sv, p.v1.sn, C::VRING + buf); };

    // ---- the q rows of the tile and the k2/v2 rows k - i0 = -32 .. 31 (less 8 per round that other workgroups walk), which fill
    // the 64 slots and are the rows of the first four rounds: all loads in flight at once (nothing else runs on the CU meanwhile)
    constexpr int RPT = 64 * PPR / 256, QPT = (32 * PPR + 255) / 256;
    const int s_row = tid / PPR, s_col = (tid % PPR) * 16;
    u32x4 sk2[RPT], sv2[RPT];
    auto load_first_rows = [&] {
#pragma unroll
        for (int x = 0; x < RPT; ++x) {
            int kk2 = i0 - 32 - 8 * r_first + s_row + x * (256 / PPR);
            kk2 = kk2 < 0 ? 0 : (kk2 < N ? kk2 : N - 1);
            sk2[x] = ld_global16(k2g + (int64_t)kk2 * p.k2.sn + s_col);
            sv2[x] = ld_global16(v2g + (int64_t)kk2 * p.v2.sn + s_col);
        }
    };
    auto store_first_rows = [&] {
#pragma unroll
        for (int x = 0; x < RPT; ++x) {
            const int slot = (s_row + x * (256 / PPR) - 32 - 8 * r_first) & 63;
            *reinterpret_cast<u32x4 *>(lds + C::K2S + slot * PITCH + s_col) = sk2[x];
            *reinterpret_cast<u32x4 *>(lds + C::V2S + slot * PITCH + s_col) = sv2[x];
        }
    };
    u32x4 sq[QPT];
    {
        const char *qg = p.q.ptr + b * p.q.sb + h * p.q.sh;
#pragma unroll
        for (int x = 0; x < QPT; ++x) {
            int ii = i0 + (s_row + x * (256 / PPR)) % 32;
            ii = ii < N ? ii : N - 1;
            sq[x] = ld_global16(qg + (int64_t)ii * p.q.sn + s_col);
        }
    }
    load_first_rows();
    // K1 tiles 0, 1, 2 and V1 tiles 0, 1 before the first step
    issue_k(0);
    issue_v(0);
    issue_k(C::TB);
    issue_v(C::TB);
    issue_k(2 * C::TB);
    // additive masks: table 0 for the diagonal tile, tables 1, 2 for the tiles the lower window edge
    // crosses.  Entry (lane, rr) is 0 if query row i0 + c attends key row 32 t + 4 hf + e(rr), else -inf
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
    // rows that round r + 1 adds beyond those (k - i0 = -8 r - 15 .. -8 r - 8), stored at the end of round r
    auto adds_rows = [&](int r) { return r + 1 < R && r + 1 >= r_first + 4; };
    auto stage_rows = [&](int r) {
        for (int x = tid; x < 2 * 8 * PPR; x += 256) {
            const int sel = x / (8 * PPR), row = (x / PPR) % 8, col = (x % PPR) * 16;
            int kk2 = i0 - 8 * r - 15 + row;
            kk2 = kk2 < 0 ? 0 : (kk2 < N ? kk2 : N - 1);
            const int slot = (-8 * r - 15 + row) & 63;
            *reinterpret_cast<u32x4 *>(lds + (sel ? C::V2S : C::K2S) + slot * PITCH + col) =
                ld_global16((sel ? v2g + (int64_t)kk2 * p.v2.sn : k2g + (int64_t)kk2 * p.k2.sn) + col);
        }
    };

    // ---- this wave's state
    f32x16 T[2][DT];           // value accumulators of the two offsets
    u32x4 A[2][KS];            // logit operands
    f32x16 O[DT];              // sum over the offsets
    f32x16 X[2];               // logits of the running tile
    f32x16 NM;                 // -M in every element: where the logit chains start
    u32x4 pa[2][2], pb[2][2];  // packed weights of the tile before / the running one
    float M = 0.f;             // softmax reference of the row (log2 domain); meaningless while `fresh`
    bool fresh = true;         // the row has not met an attended entry yet
    float l = 0.f;             // this lane's part of the row sum, relative to M, of the rounds that are complete
    float l0 = 0.f, l1 = 0.f;  // ... and of the running round, per offset
    constexpr int FW = KS < 4 ? KS : 4;
    u32x4 kf[FW], vf[FW];
    const int k_lane = RT::row_lane(lane), v_lane = RT::tr_lane(lane);

    int bk = 0;                // ring buffer of the running tile (step u: tile u in buffer u mod 4)
    int pending = 0;           // steps whose transfers are older than the stores of the last round's end (saved partials)
    int n_stores = 0;
    auto close_step = [&] {
        bk = uniform(bk == (C::NBUF - 1) * C::TB ? 0 : bk + C::TB);
    };
    auto next_k = [&] { return bk == (C::NBUF - 1) * C::TB ? 0 : bk + C::TB; };
    auto opposite = [&] { return bk >= 2 * C::TB ? bk - 2 * C::TB : bk + 2 * C::TB; };
    auto prev = [&] { return bk == 0 ? (C::NBUF - 1) * C::TB : bk - C::TB; };
    // A step begins: everything but the transfers that the step before issued has landed (the stores of a round's end are younger
    // than the transfers that the two steps behind it await).  Its own transfers are issued behind the first MFMAs of its
    // logit chain (issue), where the scalar work of their addresses costs nothing.
    auto open_step = [&](bool may_pend) {
        if (may_pend && pending > 0) {
            pending = uniform(pending - 1);
            if (uniform(n_stores) == 2 * (D / 16)) wait_loads<C::LPW + 2 * (D / 16)>();
            else wait_loads<C::LPW + D / 16>();
        } else {
            wait_loads<C::LPW>();
        }
        __syncthreads();
    };
    // (K1 tile u + 3 replaces tile u - 1, V1 tile u + 2 tile u - 2)
    auto issue = [&] {
        issue_k(prev());
        issue_v(opposite());
    };
    auto load_kf = [&](int buf) {
#pragma unroll
        for (int f = 0; f < FW; ++f) kf[f] = RT::row_frag(lds + buf + k_lane, f);
    };
    auto read_vf = [&](const char *vbase, int f) { vf[f % FW] = RT::tr_frag(vbase, f / DT, f % DT); };
    auto first_vf = [&](int vb) {
        const char *vbase = lds + C::VRING + vb + v_lane;
#pragma unroll
        for (int f = 0; f < FW; ++f) read_vf(vbase, f);
    };
    // operands of the offsets d0 and d0 + 1
    auto build_operands = [&](int d0) {
        const char *ka = lds + C::K2S + ((c - d0) & 63) * PITCH + 16 * hf, *kb = lds + C::K2S + ((c - d0 - 1) & 63) * PITCH + 16 * hf;
        const char *qr = lds + C::QS + c * C::QPITCH + 32 * hf;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            const float4 x = *reinterpret_cast<const float4 *>(qr + 64 * kk), y = *reinterpret_cast<const float4 *>(qr + 64 * kk + 16);
            const float q8[8] = {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w};
            const u32x4 fa = ld_lds16(ka + 32 * kk), fb = ld_lds16(kb + 32 * kk);
            u32x4 a0, a1;
#pragma unroll
            for (int w = 0; w < 4; ++w) {
                a0[w] = pack_bf16(q8[2 * w] * bf16_lo(fa[w]), q8[2 * w + 1] * bf16_hi(fa[w]));
                a1[w] = pack_bf16(q8[2 * w] * bf16_lo(fb[w]), q8[2 * w + 1] * bf16_hi(fb[w]));
            }
            A[0][kk] = a0;
            A[1][kk] = a1;
            pin_agpr(A[0][kk]);
            pin_agpr(A[1][kk]);
        }
    };
    auto add_mask = [&](int n) {
        const char *mk = lds + C::MASKS + n * C::MASK + lane * 16;
#pragma unroll
        for (int qq = 0; qq < 4; ++qq) {
            const float4 m4 = *reinterpret_cast<const float4 *>(mk + qq * 1024);
#pragma unroll
            for (int u = 0; u < 2; ++u) {
                X[u][4 * qq] += m4.x;
                X[u][4 * qq + 1] += m4.y;
                X[u][4 * qq + 2] += m4.z;
                X[u][4 * qq + 3] += m4.w;
            }
        }
    };
    // logits of the tile in bk; they start from NM, or (masked) from what X holds
    auto logit_chain = [&](auto masked, auto with_loads) {
        const char *kbase = lds + bk + k_lane;
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, KS>([&](auto kk_) {
            constexpr int kk = decltype(kk_)::value;
            if constexpr (kk == 0 && !decltype(masked)::value) {
                X[0] = mfma32(kf[0], A[0][0], NM);
                X[1] = mfma32(kf[0], A[1][0], NM);
            } else {
                X[0] = mfma32(kf[kk % FW], A[0][kk], X[0]);
                X[1] = mfma32(kf[kk % FW], A[1][kk], X[1]);
            }
            if constexpr (kk == 0 && decltype(with_loads)::value) issue_k(prev());
            if constexpr (kk == 1 && decltype(with_loads)::value) issue_v(opposite());
            if constexpr (kk + FW < KS) kf[kk % FW] = RT::row_frag(kbase, kk + FW);
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    // The weights of the running tile in 17 pieces: piece k takes the exponentials of elements 2 k', 2 k' + 1 of X[u] (k = 8 u + k')
    // in place and sums and packs those of piece k - 1 (a transcendental result is not ready for the next instruction)
    auto exp_piece = [&](u32x4 (&w)[2][2], auto k_) {
        constexpr int k = decltype(k_)::value;
        if constexpr (k < 16) {
            X[k / 8][2 * (k % 8)] = fast_exp2(X[k / 8][2 * (k % 8)]);
            X[k / 8][2 * (k % 8) + 1] = fast_exp2(X[k / 8][2 * (k % 8) + 1]);
        }
        if constexpr (k > 0) {
            constexpr int j = k - 1;
            const float a = X[j / 8][2 * (j % 8)], e = X[j / 8][2 * (j % 8) + 1];
            if constexpr (j < 8) l0 += a + e;
            else l1 += a + e;
            w[j / 8][(j % 8) >> 2][j & 3] = here(pack_bf16(a, e));
        }
    };
    // T += V1^T P^T of the tile before the running one, with the weights w; beside the products the weights of X (into fresh_w)
    auto value_products = [&](const u32x4 (&w)[2][2], u32x4 (&fresh_w)[2][2], int kb, auto with_exps) {
        const char *vbase = lds + C::VRING + prev() + v_lane;
        const char *kbase = lds + kb + k_lane;
        constexpr int S = 2 * KS;
        static_for<0, KS>([&](auto m_) {
            constexpr int m = decltype(m_)::value, k2s = m / DT, dt = m % DT;
            const u32x4 v = vf[m % FW];
            T[0][dt] = mfma32(v, w[0][k2s], T[0][dt]);
            if constexpr (decltype(with_exps)::value) static_for<17 * (2 * m) / S, 17 * (2 * m + 1) / S>([&](auto k) { exp_piece(fresh_w, k); });
            __builtin_amdgcn_sched_barrier(0);
            T[1][dt] = mfma32(v, w[1][k2s], T[1][dt]);
            if constexpr (m + FW < KS) read_vf(vbase, m + FW);
            else kf[m - (KS - FW)] = RT::row_frag(kbase, m - (KS - FW));
            if constexpr (decltype(with_exps)::value) static_for<17 * (2 * m + 1) / S, 17 * (2 * m + 2) / S>([&](auto k) { exp_piece(fresh_w, k); });
            __builtin_amdgcn_sched_barrier(0);
        });
    };
    using Yes = std::true_type;
    using No = std::false_type;

    // (the mask tables above were formed while the rows were on their way)
#pragma unroll
    for (int x = 0; x < QPT; ++x) {
        const int row = s_row + x * (256 / PPR);
        if (row >= 32) break;
        const float c2 = p.scale_log2e;
        float4 *dst = reinterpret_cast<float4 *>(lds + C::QS + row * C::QPITCH + s_col * 2);
        dst[0] = make_float4(bf16_lo(sq[x][0]) * c2, bf16_hi(sq[x][0]) * c2, bf16_lo(sq[x][1]) * c2, bf16_hi(sq[x][1]) * c2);
        dst[1] = make_float4(bf16_lo(sq[x][2]) * c2, bf16_hi(sq[x][2]) * c2, bf16_lo(sq[x][3]) * c2, bf16_hi(sq[x][3]) * c2);
    }
    store_first_rows();
    wait_loads<0>();
    __syncthreads();           // the staged rows, the mask tables and the first tiles are visible

    for (int attempt = 0;; ++attempt) {
        // ---- the softmax reference: the largest logit of the wave's first tile, which every valid row attends an entry of; if a
        // row's weights outgrow 2^90 on it (rare), all is done once more with the largest logit of all the wave's tiles
        {
            float tmax = -INFINITY;
            for (int r = r_first; r < (attempt ? R : r_first + 1); ++r) {
                const int d0 = 8 * r + 2 * wave;
                const bool ok0 = row_ok && i - d0 >= 0 && d0 < p.w2, ok1 = row_ok && i - d0 - 1 >= 0 && d0 + 1 < p.w2;
                // (lanes without a valid key row hold logits of clamped rows: left out)
                const float s0 = ok0 ? 0.f : -INFINITY, s1 = ok1 ? 0.f : -INFINITY;
                if (attempt && adds_rows(r - 1)) {
                    stage_rows(r - 1);
                    __syncthreads();
                }
                build_operands(d0);
                for (int n = 0; n < (attempt ? NT : 1); ++n) {
                    if (attempt) {
                        open_step(true);
                        issue();
                    }
                    load_kf(bk);
#pragma unroll
                    for (int rr = 0; rr < 16; ++rr) {
                        X[0][rr] = s0;
                        X[1][rr] = s1;
                    }
                    if (n < n_masked) add_mask(n);
                    logit_chain(Yes{}, No{});
#pragma unroll
                    for (int rr = 0; rr < 16; ++rr) tmax = fmaxf(tmax, fmaxf(X[0][rr], X[1][rr]));
                    if (attempt) close_step();
                }
            }
            auto sw = __builtin_amdgcn_permlane32_swap(as_u32(tmax), as_u32(tmax), false, false);
            tmax = fmaxf(as_f32(sw[0]), as_f32(sw[1]));
            fresh = tmax == -INFINITY;
            M = fresh ? 0.f : tmax;
            NM = splat16(-M);
            if (attempt && R > r_first + 4) {
                // (the k2/v2 rows of the first rounds again)
                __syncthreads();
                load_first_rows();
                store_first_rows();
                __syncthreads();
            }
        }
        l = 0.f;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt) O[dt] = zero16();
        load_kf(bk);

        for (int r = r_first; r < R; ++r) {
            const int d0 = 8 * r + 2 * wave;
            const bool ok0 = row_ok && i - d0 >= 0 && d0 < p.w2, ok1 = row_ok && i - d0 - 1 >= 0 && d0 + 1 < p.w2;
            const bool wave_on = wave_any(ok0);          // (a wave that is off stays off: later rounds have larger offsets)
            if (!wave_on) {
                for (int n = 0; n < NT; ++n) {
                    open_step(true);
                    issue();
                    close_step();
                }
            } else {
                build_operands(d0);
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) T[u][dt] = zero16_pairs();
                l0 = l1 = 0.f;
                // ---- the diagonal tile
                open_step(true);
                X[0] = X[1] = NM;
                add_mask(0);
                logit_chain(Yes{}, Yes{});
                load_kf(next_k());
                static_for<0, 17>([&](auto k) { exp_piece(pa, k); });
                first_vf(bk);
                close_step();
                // ---- the other tiles: logits of tile n, then the products of tile n - 1 with the weights of tile n beside them
                auto step = [&](int n, const u32x4 (&old)[2][2], u32x4 (&cur)[2][2]) {
                    open_step(n == 1);
                    if (__builtin_expect(n < n_masked, 0)) {
                        X[0] = X[1] = NM;
                        add_mask(n);
                        logit_chain(Yes{}, Yes{});
                    } else {
                        logit_chain(No{}, Yes{});
                    }
                    value_products(old, cur, next_k(), Yes{});
                    first_vf(bk);
                    close_step();
                };
                for (int n = 1; n < NT; n += 2) {
                    step(n, pa, pb);
                    if (n + 1 < NT) {
                        step(n + 1, pb, pa);
                    } else {
#pragma unroll
                        for (int u = 0; u < 2; ++u)
#pragma unroll
                            for (int x = 0; x < 2; ++x) pa[u][x] = pb[u][x];
                    }
                }
                value_products(pa, pb, bk, No{});        // (requests the fragments of the next round's first tile once more)

                // ---- end of the round: O += v2_{i-dlt} * T (in the lanes that have a key row); T and its reference kept for the
                // backward
                l += (ok0 ? l0 : 0.f) + (ok1 ? l1 : 0.f);
                n_stores = 0;
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int dlt = d0 + u;
                    if (p.t_save && dlt < p.w2) {
                        const int64_t sbh = ((int64_t)b * p.H + h) * p.w2 + dlt;
                        if (row_ok) {
                            char *trow = p.t_save + (sbh * ntile + tile) * saved_t_block<D>() + saved_t_offset(c, hf, 0, 0);
#pragma unroll
                            for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                                for (int half = 0; half < 2; ++half) {
                                    u32x4 pk;
#pragma unroll
                                    for (int w = 0; w < 4; ++w) pk[w] = pack_bf16(T[u][dt][8 * half + 2 * w], T[u][dt][8 * half + 2 * w + 1]);
                                    st_global16(trow + saved_t_offset(0, 0, dt, half), pk);
                                }
                            if (hf == 0) p.m_save[sbh * N + i] = M;
                        }
                        n_stores += D / 16;
                    }
                    if (u == 0 ? ok0 : ok1) {
                        const char *v2row = lds + C::V2S + ((c - dlt) & 63) * PITCH + 32 * hf;
#pragma unroll
                        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
                            for (int half = 0; half < 2; ++half) {
                                const u32x4 xv = ld_lds16(v2row + dt * 64 + half * 16);
#pragma unroll
                                for (int w = 0; w < 4; ++w) {
                                    O[dt][8 * half + 2 * w] += bf16_lo(xv[w]) * T[u][dt][8 * half + 2 * w];
                                    O[dt][8 * half + 2 * w + 1] += bf16_hi(xv[w]) * T[u][dt][8 * half + 2 * w + 1];
                                }
                            }
                    }
                }
                pending = n_stores ? 2 : 0;
            }
            if (adds_rows(r)) {
                stage_rows(r);
                __syncthreads();
            }
        }
        // did a row sum of this workgroup outgrow the safe range?
        if (attempt) break;
        uint32_t *vote = reinterpret_cast<uint32_t *>(lds + C::VOTE);
        const bool outgrown = wave_any(!(l < kBig));
        if (lane == 0) vote[wave] = outgrown;
        __syncthreads();
        if (!uniform((int)(vote[0] | vote[1] | vote[2] | vote[3]))) break;
        if (R > r_first + 4) {
            load_first_rows();
            store_first_rows();
            __syncthreads();
        }
    }

    // ---- the waves meet: O = sum_w O_w 2^(M_w - Mc), L = sum_w l_w 2^(M_w - Mc), Mc = max_w M_w
    wait_loads<0>();           // (transfers issued behind the last tile still write into the rings)
    __syncthreads();
    float *rows = reinterpret_cast<float *>(lds);
    float *xm = reinterpret_cast<float *>(lds + C::XM), *xl = xm + 4 * 32;
    if (hf == 0) xm[wave * 32 + c] = fresh ? -INFINITY : M;
    __syncthreads();
    float Mc = xm[c];
#pragma unroll
    for (int w = 1; w < 4; ++w) Mc = fmaxf(Mc, xm[w * 32 + c]);
    {
        const float g = fresh ? 0.f : fast_exp2(M - Mc);
        auto sw = __builtin_amdgcn_permlane32_swap(as_u32(l), as_u32(l), false, false);
        if (hf == 0) xl[wave * 32 + c] = fresh ? 0.f : (as_f32(sw[0]) + as_f32(sw[1])) * g;
        float *dst = rows + (wave * 32 + c) * C::APITCH + 16 * hf;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r4 = 0; r4 < 4; ++r4)
                *reinterpret_cast<float4 *>(dst + 32 * dt + 4 * r4) =
                    make_float4(O[dt][4 * r4] * g, O[dt][4 * r4 + 1] * g, O[dt][4 * r4 + 2] * g, O[dt][4 * r4 + 3] * g);
    }
    __syncthreads();
    {
        constexpr int SEG = D / 8;              // d values per thread (256 threads, 32 rows), in groups of four
        const int row = tid >> 3, seg = tid & 7;
        const int ir = i0 + row;
        if (ir >= N) return;
        float L = 0.f, mc = -INFINITY;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            L += xl[w * 32 + row];
            mc = fmaxf(mc, xm[w * 32 + row]);
        }
        const float inv = SPLIT ? 1.f : 1.f / L;
        const int64_t prows = (int64_t)p.B * p.H * N, prow = (int64_t)split * prows + ((int64_t)b * p.H + h) * N + ir;
        char *orow = p.o.ptr + b * p.o.sb + (int64_t)ir * p.o.sn + h * p.o.sh;
        char *rrow = p.o_lo.ptr ? p.o_lo.ptr + b * p.o_lo.sb + (int64_t)ir * p.o_lo.sn + h * p.o_lo.sh : nullptr;
#pragma unroll
        for (int x = 0; x < SEG / 4; ++x) {
            const int d = 4 * (seg + 8 * x);
            float4 a = *reinterpret_cast<const float4 *>(rows + row * C::APITCH + d);
#pragma unroll
            for (int w = 1; w < 4; ++w) {
                const float4 e = *reinterpret_cast<const float4 *>(rows + (w * 32 + row) * C::APITCH + d);
                a.x += e.x;
                a.y += e.y;
                a.z += e.z;
                a.w += e.w;
            }
            if constexpr (SPLIT) {
                // (a share that attends nothing of a row leaves zeros with the reference -inf)
                *reinterpret_cast<float4 *>(p.q_parts + prow * D + d) = a;
            } else {
                a.x *= inv;
                a.y *= inv;
                a.z *= inv;
                a.w *= inv;
                const u32x2 ov = {pack_bf16(a.x, a.y), pack_bf16(a.z, a.w)};
                *reinterpret_cast<u32x2 *>(orow + d * 2) = ov;
                if (rrow)
                    *reinterpret_cast<u32x2 *>(rrow + d * 2) =
                        (u32x2){pack_bf16(a.x - bf16_lo(ov[0]), a.y - bf16_hi(ov[0])), pack_bf16(a.z - bf16_lo(ov[1]), a.w - bf16_hi(ov[1]))};
            }
        }
        if (seg == 0) {
            if constexpr (SPLIT) *reinterpret_cast<float2 *>(p.q_parts + (int64_t)p.q_splits * prows * D + 2 * prow) = make_float2(mc, L);
            else p.lse[((int64_t)b * p.H + h) * N + ir] = (mc + __builtin_amdgcn_logf(L)) * kLn2;
        }
    }
}

}  // namespace sa2
