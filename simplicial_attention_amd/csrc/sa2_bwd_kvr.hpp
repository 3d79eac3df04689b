// Backward kernel that owns key rows, all results in registers: dK1 and dV1, one wave per SIMD.
//
// A wave owns 32 key rows j and walks the (query tile, offset dlt = i - k) pairs that reach them; per tile and offset
//     X[i][j] = A K1^T - lse,  P = exp2(X),  Y[i][j] = B V1^T - delta,  dS = P * Y
//     dV1^T += B^T P,   dK1^T += A^T dS        with A = q_i * k2_{i-dlt} * scale * log2(e),  B = do_i * v2_{i-dlt}
// (triton_two_simplicial_attention.py:298-503 of the reference; the mathematics of bwd_kv8_kernel, sa2_bwd_kv8.hpp).  Its K1 and
// V1 rows (128 registers at D = 256), both results (256), the logits and dP of a tile (32) and a window of fragments take all
// 512 registers of a lane: nothing is exchanged between the waves but the operand tiles, 64 MFMAs stand behind one barrier.
// The operand tiles of the next step are built between the MFMAs of this one, eight 16-byte products per thread.  The rows they
// are built from are staged in LDS per query tile: q pieces by direct-to-LDS loads that only their own wave reads, do pieces
// (whose place is beyond the reach of such a load) through registers, k2 and v2 rows in circular buffers of 48 rows.
// The form before it gave every wave a quarter of the columns of one slab: four partial tiles went through LDS and three
// barriers for every 64 MFMAs of a workgroup, and 2 x 8 x 4096 rows (w1 512, w2 32) took 6.9 ms; now 2.6.
// Bound now (66 cycles per MFMA): a fragment read from LDS feeds one MFMA, and with one wave per SIMD its latency shows at the
// start of every step.
#pragma once

#include <type_traits>

#include "sa2_acc.hpp"
#include "sa2_common.hpp"
#include "sa2_bwd_kv8.hpp"
#include "sa2_lds.hpp"

namespace sa2 {

template <int D>
struct KvrCfg {
    static_assert(D == 256, "two waves per SIMD are faster at smaller head dimensions (bwd_kv8_kernel)");
    static constexpr int KS = D / 16, DT = D / 32;
    using T = DmaTile<D>;
    static constexpr int CPW = T::NCH / 4;             // chunks of a tile that a wave builds
    static constexpr int NPROD = 2 * CPW;              // products per thread and step
    static constexpr int NSLOT = 48;                   // k2 / v2 rows, circular
    static constexpr int NRC = NSLOT / T::RPC;         // their chunks
    // staging in the first 64 KiB (direct loads): q pieces, k2 rows, v2 rows; do pieces beyond it
    static constexpr int QS = 0;
    static constexpr int RK = QS + T::NCH * 1024;
    static constexpr int RV = RK + NRC * 1024;
    static constexpr int DOS = RV + NRC * 1024;
    static constexpr int OPS = DOS + T::NCH * 1024;    // operand tiles A, B; two buffers
    static_assert(DOS <= 65536, "the LDS address of a direct load travels in 16 bits of M0");
    static constexpr int STEP = 2 * T::BYTES;
    static constexpr int TAB = OPS + 2 * STEP;         // -lse log2(e) [32], -delta [32]
    static constexpr int LDS = TAB + 256;
    static_assert(LDS <= 160 * 1024, "LDS of a CU");
};

template <int D, bool PARTS>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1))) void bwd_kvr_kernel(KParams p) {
    using C = KvrCfg<D>;
    using T = typename C::T;
    constexpr int KS = C::KS, DT = C::DT, RPC = T::RPC, CPW = C::CPW;
    __shared__ __attribute__((aligned(16))) char lds[C::LDS];

    const int N = p.N;
    const int nslab = (N + 127) / 128;
    const int item_all = xcd_contiguous(blockIdx.x, gridDim.x);
    const int item = PARTS ? uniform(item_all / p.kv_max_parts) : item_all;
    const int part = PARTS ? item_all - item * p.kv_max_parts : 0;
    const int bh = uniform(item / nslab);
    const int slab = item - bh * nslab;
    const int b = uniform(bh / p.HK), hk = bh - b * p.HK;
    // this workgroup's share of the slab's walk, in pairs of offsets (see bwd_kv8_kernel)
    const int head_pairs = uniform(kv8_walk_pairs(slab, N, p.w1, p.w2));
    int pair0 = 0, npairs = head_pairs * p.G;
    if constexpr (PARTS) {
        const int64_t all = (int64_t)head_pairs * p.G;
        const int parts = uniform(kv8_parts_of(all, p.kv_chunk, p.kv_max_parts));
        if (part >= parts) return;                     // (a slab with a short walk: the combine kernel knows)
        pair0 = uniform((int)(all * part / parts));
        npairs = uniform((int)(all * (part + 1) / parts)) - pair0;
    }

    const int tid = threadIdx.x;
    const int wave = wave_index(), lane = tid & 63;
    const int c = lane & 31, hf = lane >> 5;
    const int j0 = slab * 128, jw = j0 + 32 * wave;
    const int j = jw + c;
    const bool j_ok = j < N;
    const int jc = j_ok ? j : N - 1;
    const int it_begin = j0 / 32, it_end = kv8_last_tile(slab, N, p.w1);       // query tiles that reach the workgroup's rows
    const int w1 = p.w1 < N ? p.w1 : N;
    const int last_i = jw + 31 + w1 - 1 < N - 1 ? jw + 31 + w1 - 1 : N - 1;
    const int wit_lo = jw / 32, wit_hi = jw < N ? last_i / 32 : -1;            // ... this wave's
    auto last_offset = [&](int it) { return p.w2 - 1 < 32 * it + 31 ? p.w2 - 1 : 32 * it + 31; };

    const char *k2g = p.k2.ptr + b * p.k2.sb + hk * p.k2.sh;
    const char *v2g = p.v2.ptr + b * p.v2.sb + hk * p.v2.sh;

    u32x4 kf[KS], vf[KS];
    {
        const char *krow = p.k1.ptr + b * p.k1.sb + hk * p.k1.sh + (int64_t)jc * p.k1.sn + 16 * hf;
        const char *vrow = p.v1.ptr + b * p.v1.sb + hk * p.v1.sh + (int64_t)jc * p.v1.sn + 16 * hf;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            kf[kk] = ld_global16(krow + 32 * kk);
            vf[kk] = ld_global16(vrow + 32 * kk);
        }
    }
    f32x16 dK[DT], dV[DT];                             // (dK1 in accumulation registers)
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) {
        dK[dt] = dV[dt] = zero16();
        pin_acc(dK[dt]);
    }

    // ---- the walk: query heads of the group, query tiles, offsets
    struct Step {
        int g, it, dlt;
    };
    int pairs_left = npairs;
    // to the next step; false behind the last one of this workgroup's share
    auto advance = [&](Step &s) {
        const int top = last_offset(s.it);
        if ((s.dlt & 1) || s.dlt == top) {
            if (--pairs_left == 0) return false;
        }
        if (++s.dlt > top) {
            s.dlt = 0;
            if (++s.it > it_end) {
                s.it = it_begin;
                ++s.g;
            }
        }
        return true;
    };

    // ---- staging
    const int l_row = (lane >> 2) % RPC, l_col = T::st_col(lane);              // a lane's place in a chunk
    const int l_seg = lane / (4 * RPC) * (RPC * 64) + (lane & 3) * 16;
    const uint32_t lds0 = (uint32_t)(uintptr_t)lds;
    auto clamp_row = [&](int r) { return r < 0 ? 0 : (r < N ? r : N - 1); };
    // the rows first .. first + RPC - 1 of k2 or v2 into a chunk of the circular buffer
    auto load_ring = [&](const char *g, int64_t sn, int ring, int first) {
        const int base = clamp_row(first);
        int chunk = first / RPC % C::NRC;                                      // (first is a multiple of RPC)
        chunk = chunk < 0 ? chunk + C::NRC : chunk;
        load_to_lds16(uniform(g + (int64_t)base * sn), (uint32_t)((clamp_row(first + l_row) - base) * (int)sn + l_col),
                      uniform((int)(lds0 + ring + chunk * 1024)));
    };
    // what the builds of query tile s.it from offset s.dlt on read: q pieces, 48 rows of k2 and v2 (no build may be
    // reading); the start values of its chains on their way to LDS
    float start = 0.f;
    auto stage = [&](const Step &s) {
        const int h = hk * p.G + s.g, i0 = 32 * s.it;
        const char *qg = p.q.ptr + b * p.q.sb + h * p.q.sh;
        const int base = clamp_row(i0);
#pragma unroll
        for (int n = 0; n < CPW; ++n) {
            const int ch = wave + 4 * n;
            load_to_lds16(uniform(qg + (int64_t)base * p.q.sn), (uint32_t)((clamp_row(i0 + ch * RPC + l_row) - base) * (int)p.q.sn + l_col),
                          uniform((int)(lds0 + C::QS + ch * 1024)));
        }
        if (tid < 64) {
            const int64_t row = ((int64_t)b * p.H + h) * N + clamp_row(i0 + c);
            start = hf ? -p.delta[row] : -p.lse[row] * kLog2e;
            if (!hf && i0 + c >= N) start = -INFINITY;
        }
        const int top = i0 + 32 - RPC * (s.dlt / RPC);                         // behind the highest row needed
        for (int x = wave; x < C::NRC; x += 4) {
            load_ring(k2g, p.k2.sn, C::RK, top - RPC * (x + 1));
            load_ring(v2g, p.v2.sn, C::RV, top - RPC * (x + 1));
        }
    };
    // the rest of it (every wave has left the tile before)
    auto stage_rest = [&](const Step &s) {
        const int h = hk * p.G + s.g, i0 = 32 * s.it;
        const char *dog = p.dout.ptr + b * p.dout.sb + h * p.dout.sh;
        u32x4 x[CPW];
#pragma unroll
        for (int n = 0; n < CPW; ++n) x[n] = ld_global16(dog + (int64_t)clamp_row(i0 + (wave + 4 * n) * RPC + l_row) * p.dout.sn + l_col);
#pragma unroll
        for (int n = 0; n < CPW; ++n) *reinterpret_cast<u32x4 *>(lds + C::DOS + (wave + 4 * n) * 1024 + lane * 16) = x[n];
        if (tid < 64) reinterpret_cast<float *>(lds + C::TAB)[tid] = start;
    };
    // a step is built: the k2 / v2 rows that no later offset of the tile reaches make room for those 48 below
    auto refill = [&](const Step &s) {
        if ((s.dlt + 1) % RPC != 0 || wave > 1) return;
        const int first = 32 * s.it + 32 - (s.dlt + 1) - C::NSLOT;
        if (wave == 0) load_ring(k2g, p.k2.sn, C::RK, first);
        else load_ring(v2g, p.v2.sn, C::RV, first);
    };

    // ---- operand build: product x of a thread is a piece of A (even x) or B (odd x), chunk wave + 4 (x / 2)
    const float c2 = p.scale_log2e;
    u32x4 bx, by, bz;
    // place of the lane's piece of chunk `wave`, row - offset, in a circular buffer (chunk wave + 4 n: 4096 n bytes on)
    int shift = 0;                                     // slot of row 0 of the offset being built
    uint32_t at = 0;
    auto build_begin = [&](const Step &s) {
        shift = (32 * s.it - s.dlt) % C::NSLOT;
        shift = uniform(shift < 0 ? shift + C::NSLOT : shift);
    };
    auto build_read = [&](auto x_) {
        constexpr int x = decltype(x_)::value, n = x / 2;
        constexpr uint32_t ring = C::NRC * 1024;
        if constexpr (x == 0) {
            const int slot = wave * RPC + shift + l_row;      // (below 2 * NSLOT)
            at = (uint32_t)(slot / RPC * 1024 + slot % RPC * 64 + l_seg);
            at = at < at - ring ? at : at - ring;
        }
        const uint32_t far = at + 4096 * n, wrapped = far < far - ring ? far : far - ring;
        bx = ld_lds16(lds + (x & 1 ? C::DOS : C::QS) + (wave + 4 * n) * 1024 + lane * 16);
        by = ld_lds16(lds + (x & 1 ? C::RV : C::RK) + (n ? wrapped : at));
    };
    auto build_word = [&](auto x_, int w) {
        constexpr bool is_a = (decltype(x_)::value & 1) == 0;
        if constexpr (is_a) bz[w] = pack_bf16(bf16_lo(bx[w]) * c2 * bf16_lo(by[w]), bf16_hi(bx[w]) * c2 * bf16_hi(by[w]));
        else bz[w] = pack_bf16(bf16_lo(bx[w]) * bf16_lo(by[w]), bf16_hi(bx[w]) * bf16_hi(by[w]));
    };
    auto build_write = [&](auto x_, char *dst) {
        constexpr int x = decltype(x_)::value, n = x / 2;
        *reinterpret_cast<u32x4 *>(dst + (x & 1) * T::BYTES + (wave + 4 * n) * T::CP + lane * 16) = bz;
    };
    auto build = [&](char *dst) {
        static_for<0, C::NPROD>([&](auto x) {
            build_read(x);
#pragma unroll
            for (int w = 0; w < 4; ++w) build_word(x, w);
            build_write(x, dst);
        });
    };

    const int r_lane = T::row_lane(lane), t_lane = T::tr_lane(lane);
    // one step; `dst`: where the operand tiles of the next one are built meanwhile
    auto compute = [&](const Step &s, const char *ops, char *dst) {
        constexpr int W = 6, NROW = 2 * KS, TRA = NROW + 2 * DT, NFR = TRA + 2 * DT;
        constexpr int EVERY = NFR / C::NPROD;
        static_assert(EVERY == 8 && NFR == C::NPROD * EVERY, "a product rides behind eight MFMAs");
        const char *ra = ops + r_lane, *rb = ra + T::BYTES, *ta = ops + t_lane, *tb = ta + T::BYTES;
        // A rows, B rows, B transposed, A transposed
        auto fragment = [&](auto idx) {
            constexpr int x = decltype(idx)::value;
            if constexpr (x < KS) return T::row_frag(ra, x);
            else if constexpr (x < NROW) return T::row_frag(rb, x - KS);
            else if constexpr (x < TRA) return T::tr_frag(tb, (x - NROW) / DT, (x - NROW) % DT);
            else return T::tr_frag(ta, (x - TRA) / DT, (x - TRA) % DT);
        };
        u32x4 f[W];
        f32x16 X, Y;
#pragma unroll
        for (int kk = 0; kk < KS; ++kk) {
            pin_agpr(kf[kk]);
            pin_agpr(vf[kk]);
        }
        const char *tab = lds + C::TAB + 16 * hf;
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 a = *reinterpret_cast<const float4 *>(tab + 32 * q4);
            X[4 * q4] = a.x;
            X[4 * q4 + 1] = a.y;
            X[4 * q4 + 2] = a.z;
            X[4 * q4 + 3] = a.w;
            const float4 d = *reinterpret_cast<const float4 *>(tab + 128 + 32 * q4);
            Y[4 * q4] = d.x;
            Y[4 * q4 + 1] = d.y;
            Y[4 * q4 + 2] = d.z;
            Y[4 * q4 + 3] = d.w;
        }
        static_for<0, W>([&](auto x) { f[x] = fragment(x); });
        const int i0 = 32 * s.it, dlt = s.dlt;
        if (!(i0 >= jw + 31 && i0 + 31 - jw < w1 && i0 >= dlt)) {
            // attended rows i: max(j, dlt) <= i < j + w1 (register e holds row i0 + 4 hf + 8 (e / 4) + e % 4)
            const int from = j > dlt ? j : dlt, span = j + w1 > from ? j + w1 - from : 0;
            int rel = i0 + 4 * hf - from;
            asm volatile("" : "+v"(rel));
#pragma unroll
            for (int e = 0; e < 16; ++e) X[e] = (unsigned)(rel + 8 * (e >> 2) + (e & 3)) < (unsigned)span ? X[e] : -INFINITY;
        }
        u32x4 pb[2], sb[2];
        auto weights = [&](int e) {            // X becomes P, packed
            X[e] = fast_exp2(X[e]);
            X[e + 1] = fast_exp2(X[e + 1]);
            pb[e >> 3][(e & 7) >> 1] = pack_bf16(X[e], X[e + 1]);
        };
        auto slopes = [&](int e) { sb[e >> 3][(e & 7) >> 1] = pack_bf16(X[e] * Y[e], X[e + 1] * Y[e + 1]); };
        __builtin_amdgcn_sched_barrier(0);
        static_for<0, NFR>([&](auto x_) {
            constexpr int x = decltype(x_)::value;
            if constexpr (x < KS) X = mfma32(f[x % W], kf[x], X);
            else if constexpr (x < NROW) Y = mfma32(f[x % W], vf[x - KS], Y);
            else if constexpr (x < TRA) dV[(x - NROW) % DT] = mfma32(f[x % W], pb[(x - NROW) / DT], dV[(x - NROW) % DT]);
            else mfma32_acc(dK[(x - TRA) % DT], f[x % W], sb[(x - TRA) / DT]);
            if constexpr (x + W < NFR) f[x % W] = fragment(std::integral_constant<int, x + W>{});
            // the exponentials behind the chain of Y, dS behind the products of dV
            if constexpr (x >= KS + 2 && x < KS + 10) weights(2 * (x - KS - 2));
            if constexpr (x >= NROW + 2 && x < NROW + 10) slopes(2 * (x - NROW - 2));
            constexpr std::integral_constant<int, x / EVERY> prod{};
            if constexpr (x % EVERY == 0) build_read(prod);
            if constexpr (x % EVERY >= 4) build_word(prod, x % EVERY - 4);
            if constexpr (x % EVERY == 7) build_write(prod, dst);
            __builtin_amdgcn_sched_barrier(0);
        });
    };

    // ---- the walk
    Step nb = {0, it_begin, 0};
    if constexpr (PARTS) {
        nb.g = uniform(pair0 / head_pairs);
        int left = pair0 - nb.g * head_pairs;
        for (int n; left >= (n = kv8_pairs_of(nb.it, p.w2)); ++nb.it) left -= n;
        nb.dlt = 2 * left;
    }
    stage(nb);
    stage_rest(nb);
    wait_loads<0>();
    __syncthreads();
    build_begin(nb);
    build(lds + C::OPS);
    __syncthreads();
    int buf = 0;
    bool more = true;
    // one step, with this wave's MFMAs (ON) or without
    auto step = [&](auto on_, const Step &cur) {
        const bool turn = more && nb.dlt == 0;
        if (turn) stage(nb);
        else if (more) refill(cur);
        build_begin(nb);
        const char *ops = lds + C::OPS + (buf ? C::STEP : 0);
        char *dst = lds + C::OPS + (buf ? 0 : C::STEP);
        // (behind the last step and where the tile changes, what is built here is of no use: it is built again or not read)
        if constexpr (decltype(on_)::value) compute(cur, ops, dst);
        else build(dst);
        if (!more) return;
        wait_loads<0>();
        __syncthreads();
        if (turn) {
            stage_rest(nb);
            __syncthreads();
            build(dst);
            __syncthreads();
        }
        buf ^= 1;
    };
    // (two loops, entered in turn: a branch inside one loop makes the compiler move the results where its arms meet)
    auto on_at = [&](const Step &s) { return s.it >= wit_lo && s.it <= wit_hi; };
    while (more) {
        if (on_at(nb)) {
            do {
                const Step cur = nb;
                more = advance(nb);
                step(std::true_type{}, cur);
            } while (more && on_at(nb));
        } else {
            do {
                const Step cur = nb;
                more = advance(nb);
                step(std::false_type{}, cur);
            } while (more && !on_at(nb));
        }
    }

    acc_done();
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) pin_acc(dK[dt]);
    if (!j_ok) return;
    // (A carried scale log2(e): times ln 2 gives the softmax scale)
    if constexpr (PARTS) {
        const int64_t rows = (int64_t)p.B * p.HK * N;
        float *row = p.kv_parts + ((int64_t)(2 * part) * rows + ((int64_t)b * p.HK + hk) * N + j) * D + 16 * hf;
        store_row_f32<DT>(row, dK, kLn2);
        store_row_f32<DT>(row + rows * D, dV, 1.f);
    } else {
        store_row<DT>(p.dk1.ptr + b * p.dk1.sb + (int64_t)j * p.dk1.sn + hk * p.dk1.sh + 32 * hf, dK, kLn2);
        store_row<DT>(p.dv1.ptr + b * p.dv1.sb + (int64_t)j * p.dv1.sn + hk * p.dv1.sh + 32 * hf, dV, 1.f);
    }
}

}  // namespace sa2
