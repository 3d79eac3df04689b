// C ABI of libsa2: argument validation and kernel launches (see include/sa2.h).
#include "sa2.h"

#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <mutex>

#include "sa2_bwd.hpp"
#include "sa2_bwd_kv8.hpp"
#include "sa2_bwd_q.hpp"
#include "sa2_common.hpp"
#include "sa2_convert.hpp"
#include "sa2_lds.hpp"
#include "sa2_qkv_norm.hpp"
#include "sa2_wgrad.hpp"
#include "sa2_fwd.hpp"
#include "sa2_launch.hpp"
#ifdef SA2_PROFILING
#include "sa2_prof_mix.hpp"
#endif

namespace {

thread_local char g_err[256] = "";

int fail(int code, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_err, sizeof(g_err), fmt, ap);
    va_end(ap);
    return code;
}

int check_problem(const sa2_problem *p) {
    if (!p) return fail(SA2_ERR_NULL_POINTER, "problem is NULL");
    if (p->batch < 1 || p->seq_len < 1 || p->heads < 1 || p->kv_heads < 1)
        return fail(SA2_ERR_BAD_SHAPE, "batch=%d seq_len=%d heads=%d kv_heads=%d must all be >= 1", p->batch, p->seq_len,
                    p->heads, p->kv_heads);
    if (p->heads % p->kv_heads != 0)
        return fail(SA2_ERR_BAD_SHAPE, "heads=%d is not a multiple of kv_heads=%d", p->heads, p->kv_heads);
    if (p->w1 < 1 || p->w2 < 1) return fail(SA2_ERR_BAD_SHAPE, "windows w1=%d w2=%d must be >= 1", p->w1, p->w2);
    if (p->causal != 1) return fail(SA2_ERR_UNSUPPORTED, "only causal=1 is defined for the sliding windows");
    if (p->dtype != SA2_BF16) return fail(SA2_ERR_UNSUPPORTED, "dtype %d is not supported (bf16 only)", p->dtype);
    if (p->dim_head != 32 && p->dim_head != 64 && p->dim_head != 128 && p->dim_head != 256)
        return fail(SA2_ERR_UNSUPPORTED, "dim_head=%d is not supported (32, 64, 128 or 256)", p->dim_head);
    if (!(p->scale > 0.f) || !std::isfinite(p->scale)) return fail(SA2_ERR_BAD_SHAPE, "scale must be positive and finite");
    if ((int64_t)p->batch * p->heads * ((p->seq_len + 31) / 32) > 0x7fffffffll)
        return fail(SA2_ERR_BAD_SHAPE, "problem too large for a 1-D grid");
    return SA2_OK;
}

int check_tensor(const sa2_tensor *t, const char *name) {
    if (!t || !t->ptr) return fail(SA2_ERR_NULL_POINTER, "tensor %s is NULL", name);
    if ((reinterpret_cast<uintptr_t>(t->ptr) & 15) != 0 || (t->stride_b & 7) != 0 || (t->stride_n & 7) != 0 ||
        (t->stride_h & 7) != 0)
        return fail(SA2_ERR_ALIGNMENT, "tensor %s: base pointer must be 16-byte aligned and strides multiples of 8 elements",
                    name);
    return SA2_OK;
}

// The kernels address a row inside a 32-row tile of an operand by 32 bits: its stride is bounded (by 64 MiB)
int check_operand(const sa2_problem *p, const sa2_tensor *t, const char *name) {
    const int rc = check_tensor(t, name);
    if (rc == SA2_OK && p->seq_len > 1 && (t->stride_n < 0 || t->stride_n > SA2_MOST_STRIDE_N))
        return fail(SA2_ERR_BAD_SHAPE, "tensor %s: rows are %lld elements apart, 0 to %lld are supported", name, (long long)t->stride_n,
                    (long long)SA2_MOST_STRIDE_N);
    return rc;
}

sa2::DevTensor dev(const sa2_tensor *t) {
    sa2::DevTensor d;
    d.ptr = static_cast<char *>(t->ptr);
    d.sb = t->stride_b * 2;
    d.sn = t->stride_n * 2;
    d.sh = t->stride_h * 2;
    return d;
}

sa2::KParams base_params(const sa2_problem *p) {
    sa2::KParams k{};
    k.B = p->batch;
    k.N = p->seq_len;
    k.H = p->heads;
    k.HK = p->kv_heads;
    k.G = p->heads / p->kv_heads;
    k.w1 = p->w1;
    k.w2 = p->w2;
    k.scale = p->scale;
    k.scale_log2e = p->scale * sa2::kLog2e;
    k.q_splits = 1;
    return k;
}

int after_launch(const char *what) {
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return fail(SA2_ERR_LAUNCH, "%s launch failed: %s", what, hipGetErrorString(e));
    return SA2_OK;
}

#define SA2_TRY(expr)                  \
    do {                               \
        int rc_ = (expr);              \
        if (rc_ != SA2_OK) return rc_; \
    } while (0)

// Head dimension 256 runs kernels of its own (sa2_wide.hpp), which keep no forward partials.
constexpr int kWideDimHead = 256;

// Runs the statement with the compile-time constant DH set to the problem's head dimension (validated by
// check_problem): the kernels built for head dimensions 32, 64 and 128 ...
#define SA2_FOR_DIM_HEAD(dim_head, ...)         \
    do {                                        \
        if ((dim_head) == 128) {                \
            constexpr int DH = 128;             \
            __VA_ARGS__;                        \
        } else if ((dim_head) == 64) {          \
            constexpr int DH = 64;              \
            __VA_ARGS__;                        \
        } else {                                \
            constexpr int DH = 32;              \
            __VA_ARGS__;                        \
        }                                       \
    } while (0)

// ... and the kernels that every head dimension shares
#define SA2_FOR_ANY_DIM_HEAD(dim_head, ...)             \
    do {                                                \
        if ((dim_head) == kWideDimHead) {               \
            constexpr int DH = kWideDimHead;            \
            __VA_ARGS__;                                \
        } else {                                        \
            SA2_FOR_DIM_HEAD(dim_head, __VA_ARGS__);    \
        }                                               \
    } while (0)

// Scratch of sa2_bwd_noalloc: delta rows followed by the dK2/dV2 partial rows.  A file-scope device
// array: every GPU the library runs on holds its own copy, at its own address, until the process
// ends.  In host code the array's name is only a handle for hipGetSymbolAddress; kernels and
// runtime calls get the address that call returns for the current device.
constexpr int64_t kNoallocScratchBytes = SA2_NOALLOC_SCRATCH_BYTES;
static __device__ __align__(256) unsigned char g_noalloc_scratch[kNoallocScratchBytes];

constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
unsigned char *g_scratch_ptr[kMaxDevices] = {};

// device address of the scratch array on the current device (looked up once per device)
int noalloc_scratch(unsigned char **out) {
    int device = -1;
    hipError_t e = hipGetDevice(&device);
    if (e != hipSuccess) return fail(SA2_ERR_LAUNCH, "hipGetDevice failed: %s", hipGetErrorString(e));
    if (device < 0 || device >= kMaxDevices) return fail(SA2_ERR_UNSUPPORTED, "device index %d is not supported (at most %d)", device, kMaxDevices);
    std::lock_guard<std::mutex> guard(g_scratch_mutex);
    if (!g_scratch_ptr[device]) {
        void *ptr = nullptr;
        e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(g_noalloc_scratch));
        if (e != hipSuccess || !ptr) return fail(SA2_ERR_LAUNCH, "hipGetSymbolAddress(scratch) failed: %s", hipGetErrorString(e));
        g_scratch_ptr[device] = static_cast<unsigned char *>(ptr);
    }
    *out = g_scratch_ptr[device];
    return SA2_OK;
}

}  // namespace

extern "C" {

int sa2_version(void) { return SA2_VERSION; }

const char *sa2_last_error(void) { return g_err; }

int sa2_supported(int32_t dim_head, int32_t w1, int32_t w2, int32_t dtype) {
    return (dim_head == 32 || dim_head == 64 || dim_head == 128 || dim_head == kWideDimHead) && w1 >= 1 && w2 >= 1 && dtype == SA2_BF16;
}

static int check_saved(const sa2_problem *prob, const sa2_saved *saved) {
    if (prob->dim_head == kWideDimHead) return fail(SA2_ERR_UNSUPPORTED, "dim_head=%d keeps no forward partials: pass saved = NULL", prob->dim_head);
    if (!saved->t || !saved->m) return fail(SA2_ERR_NULL_POINTER, "saved->t or saved->m is NULL");
    if ((reinterpret_cast<uintptr_t>(saved->t) & 15) != 0) return fail(SA2_ERR_ALIGNMENT, "saved->t must be 16-byte aligned");
    return SA2_OK;
}

int64_t sa2_saved_t_bytes(const sa2_problem *prob) {
    if (check_problem(prob) != SA2_OK) return -1;
    if (prob->dim_head == kWideDimHead) return 0;
    return (int64_t)prob->batch * prob->heads * prob->w2 * ((prob->seq_len + 31) / 32) * 32 * prob->dim_head * 2;
}

int64_t sa2_saved_m_bytes(const sa2_problem *prob) {
    if (check_problem(prob) != SA2_OK) return -1;
    if (prob->dim_head == kWideDimHead) return 0;
    return (int64_t)prob->batch * prob->heads * prob->w2 * prob->seq_len * 4;
}

// ---- splitting the work of small grids.  The rules are functions of the problem alone (the library is built for this one
// chip), so workspace sizes and the kernels that run do not depend on the device or on which thread asked first.
static constexpr int kComputeUnits = 256;

// Estimated finish time of `groups` workgroups of at most `longest` units each (their sum: `total`) that the CUs take one
// at a time: one round of the longest while they fit the chip, else an even share and a ragged end, but no less than
// the whole rounds that workgroups of equal length would take (list schedules of the shapes of the tests and the benchmark
// end within 5 % of this).
static double finish_time(double groups, double longest, double total) {
    if (groups <= kComputeUnits) return longest;
    const double full = std::ceil(groups / kComputeUnits) * longest, even = total / kComputeUnits + 0.2 * longest;
    return full > even ? full : even;
}

// Query-stationary kernels: the rounds (eight offsets each) of a query tile over several workgroups.  A unit is one step
// (a K1/V1 tile of one round, 0.7 us); a round end takes kRoundEnd of them, a workgroup's start and end kQueryCost, and
// the partial rows are written and read once.  Two sequences of 128 rows and 4 heads at D = 64 (32 workgroups of 4 rounds)
// took 29 us unsplit.
static constexpr int kRoundEnd = 3, kQueryCost = 6;
static constexpr int64_t kQueryPartBytes = 128ll << 20;
// Every split of the backward has scatter rows of its own, as many as the second window is long even where the sequence is shorter
// (2 heads of 96 rows, w2 = 10^6, D = 64: 3 GiB each); splits that would take more than this together are not made.
static constexpr int64_t kScatterPartBytes = 1ll << 30;

// rows below a 32-row query tile that its offsets reach (offsets run in rounds of eight)
static int q_halo(int w2) { return 8 * ((w2 + 7) / 8) - 1; }

// partial rows of dK2 and dV2 (the dV2 half is not needed with saved forward partials)
static int64_t partial_rows_bytes(const sa2_problem *prob) {
    return sa2::qk2_ws_floats(prob->batch, prob->heads, prob->seq_len, prob->dim_head, 32 + q_halo(prob->w2)) * 4;
}

static int64_t q_parts_bytes(const sa2_problem *prob, int splits) {
    return (int64_t)splits * prob->batch * prob->heads * prob->seq_len * prob->dim_head * 4;
}

// `shared`: two workgroups of the kernel fit a CU and together finish 1.4 times the work of one (the forward at D = 32
// and 64), so up to two workgroups per CU run at once and each takes 1.45 times as long.
// `scatter_bytes`: scatter rows of one split
static int q_splits(const sa2_problem *prob, int merge_cost, bool shared, int64_t scatter_bytes) {
    if (prob->dim_head == kWideDimHead) return 1;
    const int ntile = (prob->seq_len + 31) / 32;
    const double heads = (double)prob->batch * prob->heads;
    if (heads * ntile > 4 * kComputeUnits) return 1;       // (fills the chip many times over: nothing to gain)
    const int rounds = sa2::fwd_rounds(ntile - 1, prob->w2);
    // tiles of equal rounds and steps, as (rounds, steps per round, how many)
    struct Class {
        int rounds, steps, count;
    };
    Class cls[68];
    int ncls = 0;
    for (int t = 0; t < ntile; ++t) {
        const int lo = 32 * t - prob->w1 + 1 > 0 ? (32 * t - prob->w1 + 1) / 32 : 0;
        const int r = sa2::fwd_rounds(t, prob->w2), n = t - lo + 1;
        if (ncls && cls[ncls - 1].rounds == r && cls[ncls - 1].steps == n) ++cls[ncls - 1].count;
        else if (ncls < 68) cls[ncls++] = {r, n, 1};
        else ++cls[ncls - 1].count;                        // (windows of over 2000 rows: the last class stands for the rest)
    }
    int best = 1;
    double best_cost = 0;
    for (int splits = 1; splits <= rounds; ++splits) {
        if (splits > 1 && (q_parts_bytes(prob, splits) > kQueryPartBytes || splits * scatter_bytes > kScatterPartBytes)) break;
        double total = 0, longest = 0, groups = 0;
        for (int x = 0; x < ncls; ++x) {
            const int r = cls[x].rounds, n = splits < r ? splits : r;
            const double step = cls[x].steps + kRoundEnd, one = (r + n - 1) / n * step + kQueryCost;
            longest = one > longest ? one : longest;
            total += cls[x].count * (r * step + n * kQueryCost);
            groups += (double)cls[x].count * n;
        }
        groups *= heads;
        total *= heads;
        const double merge = splits > 1 ? merge_cost + 2.0 * (double)q_parts_bytes(prob, splits) / 3.5e6 : 0;
        const double time = shared && groups > kComputeUnits ? finish_time(0.5 * groups, 1.45 * longest, 0.73 * total) : finish_time(groups, longest, total);
        if (splits == 1 || time + merge < 0.95 * best_cost) {
            best = splits;
            best_cost = time + merge;
        }
    }
    return best;
}

static int fwd_splits(const sa2_problem *prob) { return q_splits(prob, 8, prob->dim_head != 128, 0); }   // (the merge is a launch of its own)
static int bwd_splits(const sa2_problem *prob) { return q_splits(prob, 2, false, partial_rows_bytes(prob)); }

// dim_head 64 and 32: two workgroups of eight waves per CU, an offset per wave.  128: one wave per SIMD with two offsets each, unless the second
// window leaves so many waves of the last round without one that eight waves are faster.  4 x 8 x 8192 rows, w1 512, the eight-wave form
// and the other (us): w2 2 506, 613; 4 511, 620; 9 971, 1028; 12 1032, 1050; 32 2253, 2107.  (Shared rounds are another matter: kernels there are
// short of workgroups, not of waves, and one form serves.)
static constexpr int kShortWindow = 12;
static void launch_fwd(int dim_head, bool split, int grid, hipStream_t s, const sa2::KParams &k) {
    if (dim_head == 128) {
        if (!split && k.w2 <= kShortWindow) hipLaunchKernelGGL((sa2::fwd_kernel<128>), dim3(grid), dim3(512), 0, s, k);
        else sa2::launch_fwd2(split, grid, s, k);
    } else if (dim_head == 64) {
        if (split) hipLaunchKernelGGL((sa2::fwd_kernel<64, true>), dim3(grid), dim3(512), 0, s, k);
        else hipLaunchKernelGGL((sa2::fwd_kernel<64>), dim3(grid), dim3(512), 0, s, k);
    } else {
        if (split) hipLaunchKernelGGL((sa2::fwd_kernel<32, true>), dim3(grid), dim3(512), 0, s, k);
        else hipLaunchKernelGGL((sa2::fwd_kernel<32>), dim3(grid), dim3(512), 0, s, k);
    }
}

int64_t sa2_fwd_workspace_bytes(const sa2_problem *prob) {
    if (check_problem(prob) != SA2_OK) return -1;
    const int splits = fwd_splits(prob);
    return splits > 1 ? q_parts_bytes(prob, splits) + 8ll * splits * prob->batch * prob->heads * prob->seq_len : 0;
}

int sa2_fwd_ws(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
               const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *out, const sa2_tensor *out_residual,
               float *lse, const sa2_saved *saved, void *workspace, int64_t workspace_bytes, void *hip_stream) {
    SA2_TRY(check_problem(prob));
    if (out_residual) SA2_TRY(check_tensor(out_residual, "out_residual"));
    SA2_TRY(check_operand(prob, q, "q"));
    SA2_TRY(check_operand(prob, k1, "k1"));
    SA2_TRY(check_operand(prob, k2, "k2"));
    SA2_TRY(check_operand(prob, v1, "v1"));
    SA2_TRY(check_operand(prob, v2, "v2"));
    SA2_TRY(check_tensor(out, "out"));
    if (!lse) return fail(SA2_ERR_NULL_POINTER, "lse is NULL");
    if ((reinterpret_cast<uintptr_t>(workspace) & 15) != 0) return fail(SA2_ERR_ALIGNMENT, "workspace must be 16-byte aligned");
    sa2::KParams k = base_params(prob);
    k.q = dev(q);
    k.k1 = dev(k1);
    k.k2 = dev(k2);
    k.v1 = dev(v1);
    k.v2 = dev(v2);
    k.o = dev(out);
    if (out_residual) k.o_lo = dev(out_residual);
    k.lse = lse;
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    if (saved) {
        SA2_TRY(check_saved(prob, saved));
        k.t_save = static_cast<char *>(saved->t);
        k.m_save = saved->m;
    }
    const int grid = prob->batch * prob->heads * ((prob->seq_len + 31) / 32);
    if (prob->dim_head == kWideDimHead) {
        const int wgrid = prob->batch * prob->heads * ((prob->seq_len + 127) / 128);
        sa2::launch_fwd_wide(wgrid, s, k);
        return after_launch("forward");
    }
    const int64_t need = workspace ? sa2_fwd_workspace_bytes(prob) : 0;
    if (need == 0 || workspace_bytes < need) {
        launch_fwd(prob->dim_head, false, grid, s, k);
        return after_launch("forward");
    }
    k.q_splits = fwd_splits(prob);
    k.q_parts = static_cast<float *>(workspace);
    launch_fwd(prob->dim_head, true, k.q_splits * grid, s, k);
    SA2_TRY(after_launch("forward in splits"));
    const int64_t rows = (int64_t)prob->batch * prob->heads * prob->seq_len;
    const int rows_per_block = 256 / (prob->dim_head / 8);
    const int cgrid = (int)((rows + rows_per_block - 1) / rows_per_block);
    SA2_FOR_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL(sa2::fwd_combine_kernel<DH>, dim3(cgrid), dim3(256), 0, s, k));
    return after_launch("forward combine");
}

int sa2_fwd(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
            const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *out, const sa2_tensor *out_residual,
            float *lse, const sa2_saved *saved, void *hip_stream) {
    return sa2_fwd_ws(prob, q, k1, k2, v1, v2, out, out_residual, lse, saved, nullptr, 0, hip_stream);
}

int sa2_bwd_delta(const sa2_problem *prob, const sa2_tensor *out, const sa2_tensor *out_residual,
                  const sa2_tensor *dout, float *delta, void *hip_stream) {
    SA2_TRY(check_problem(prob));
    if (out_residual) SA2_TRY(check_tensor(out_residual, "out_residual"));
    SA2_TRY(check_tensor(out, "out"));
    SA2_TRY(check_tensor(dout, "dout"));
    if (!delta) return fail(SA2_ERR_NULL_POINTER, "delta is NULL");
    sa2::KParams k = base_params(prob);
    k.o = dev(out);
    if (out_residual) k.o_lo = dev(out_residual);
    k.dout = dev(dout);
    k.delta = delta;
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    int64_t rows = (int64_t)prob->batch * prob->heads * prob->seq_len;
    int lanes_per_row = prob->dim_head / 8;
    int rows_per_block = 256 / lanes_per_row;
    int grid = (int)((rows + rows_per_block - 1) / rows_per_block);
    SA2_FOR_ANY_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL(sa2::delta_kernel<DH>, dim3(grid), dim3(256), 0, s, k));
    return after_launch("delta");
}

static int bwd_common(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                      const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *dout, const float *lse,
                      const float *delta, sa2::KParams *k) {
    SA2_TRY(check_problem(prob));
    SA2_TRY(check_operand(prob, q, "q"));
    SA2_TRY(check_operand(prob, k1, "k1"));
    SA2_TRY(check_operand(prob, k2, "k2"));
    SA2_TRY(check_operand(prob, v1, "v1"));
    SA2_TRY(check_operand(prob, v2, "v2"));
    SA2_TRY(check_operand(prob, dout, "dout"));
    if (!lse) return fail(SA2_ERR_NULL_POINTER, "lse is NULL");
    if (!delta) return fail(SA2_ERR_NULL_POINTER, "delta is NULL");
    *k = base_params(prob);
    k->q = dev(q);
    k->k1 = dev(k1);
    k->k2 = dev(k2);
    k->v1 = dev(v1);
    k->v2 = dev(v2);
    k->dout = dev(dout);
    k->lse = const_cast<float *>(lse);
    k->delta = const_cast<float *>(delta);
    return SA2_OK;
}

// Profiling builds only (-DSA2_PROFILING, libsa2_prof.so): SA2_BWD_PASS=first launches only the
// MFMA kernel of the dQ/dK2/dV2 entry point, so that it can be timed alone; the results of such a
// call are incomplete.  The product library does not read the environment.
static int bwd_pass_filter() {
#ifdef SA2_PROFILING
    const char *v = std::getenv("SA2_BWD_PASS");
    if (v && std::strcmp(v, "first") == 0) return 1;
#endif
    return 0;
}

static int64_t max64(int64_t a, int64_t b) { return a > b ? a : b; }

// dK1/dV1 with the walk of a key slab split over several workgroups (fp32 partial results, summed by a second kernel).
// One workgroup runs per CU, so a small grid leaves CUs idle (at 1 sequence of 1000 rows and 4 key/value heads 32
// workgroups took 695 us where the work of 256 CUs is 60 us) and a middle one ends on a ragged tail (512 workgroups of
// unequal length at 8 sequences of 2048 rows).  The rule estimates the finish time of every part count in units of one
// pair (a query tile and two offsets, 1.3 us at D = 64, 1.9 us at D = 128); a part costs kPartCost pairs on top of its share
// (its K1/V1 rows, the first rows and operand tiles, 2 * 128 * D fp32 values written and read again).
static constexpr int kPartCost = 12;
static constexpr int kMaxParts = 64;

struct Kv8Plan {
    int chunk, parts;      // parts == 1: one workgroup per slab, no partial results
};

static int64_t kv_part_bytes(const sa2_problem *prob) {
    return 2ll * prob->batch * prob->kv_heads * prob->seq_len * prob->dim_head * 4;
}

// Partial results of dK1/dV1 may take what the scatter rows of dK2 and dV2 take, or this much where those are small.
static constexpr int64_t kPartBytes = 192ll << 20;

// The plan of sa2_bwd, whose workspace leaves room for two parts: for grids of one to four workgroups per CU on short
// sequences, where the slabs at the sequence's end (those within w1 + 128 rows of it) meet fewer query tiles than the others.
static Kv8Plan two_part_plan(const sa2_problem *prob) {
    if (prob->dim_head == kWideDimHead) return {0, 1};
    const int nslab = (prob->seq_len + 127) / 128;
    const int64_t grid = (int64_t)prob->batch * prob->kv_heads * nslab;
    const int64_t ragged = (prob->w1 + 127) / 128 + 1;          // slabs per sequence with a shortened range of query tiles
    if (grid <= kComputeUnits || grid >= 4 * kComputeUnits || 8 * ragged < nslab) return {0, 1};
    int64_t longest = 0;
    for (int t = 0; t < nslab; ++t)
        longest = max64(longest, (int64_t)sa2::kv8_walk_pairs(t, prob->seq_len, prob->w1, prob->w2) * (prob->heads / prob->kv_heads));
    return {(int)((longest + 1) / 2), 2};
}

static Kv8Plan kv8_plan(const sa2_problem *prob) {
    const int nslab = (prob->seq_len + 127) / 128, G = prob->heads / prob->kv_heads;
    const int64_t heads = (int64_t)prob->batch * prob->kv_heads;
    const int64_t budget = max64(kPartBytes, partial_rows_bytes(prob));
    // slabs of equal length, as (pairs, how many): those at a sequence's ends differ from the others
    struct Class {
        int64_t pairs;
        int count;
    };
    Class cls[24];
    int ncls = 0;
    int64_t longest = 0, total = 0;
    for (int t = 0; t < nslab; ++t) {
        const int64_t n = (int64_t)sa2::kv8_walk_pairs(t, prob->seq_len, prob->w1, prob->w2) * G;
        longest = n > longest ? n : longest;
        total += n;
        if (ncls && (cls[ncls - 1].pairs == n || ncls == 24)) ++cls[ncls - 1].count;
        else cls[ncls++] = {n, 1};
    }
    total *= heads;
    Kv8Plan best = {0, 1};
    double best_cost = 0;
    for (int parts = 1; parts <= kMaxParts && parts <= longest && (parts == 1 || parts * kv_part_bytes(prob) <= budget); ++parts) {
        const int64_t chunk = (longest + parts - 1) / parts;
        const double extra = parts > 1 ? kPartCost : 0;
        double groups = 0;
        for (int x = 0; x < ncls; ++x) groups += (double)cls[x].count * sa2::kv8_parts_of(cls[x].pairs, (int)chunk, parts);
        groups *= heads;
        // (the combine kernel: a launch, and the partial rows read at 5.8 TB/s; a pair is worth 1.3 us of it)
        const double merge = parts > 1 ? 2 + (double)(parts * kv_part_bytes(prob)) / 7.5e6 : 0;
        const double cost = finish_time(groups, chunk + extra, (double)total + extra * groups) + merge;
        if (parts == 1 || cost < 0.995 * best_cost) {
            best = {(int)chunk, parts};
            best_cost = cost;
        }
    }
    // (where the estimate sees no gain, slabs are divided as sa2_bwd divides them, so that both entry points give the same bits there.  Not
    // for speed: 8 sequences of 2048 rows, 4 key/value heads, D = 64, forward and backward take 3.04 ms in halves and 3.06 undivided, which is
    // less than two runs differ by)
    return best.parts == 1 ? two_part_plan(prob) : best;
}

static int64_t two_parts_bytes(const sa2_problem *prob) { return two_part_plan(prob).parts > 1 ? 2 * kv_part_bytes(prob) : 0; }

int64_t sa2_bwd_workspace_bytes(const sa2_problem *prob) {
    if (check_problem(prob) != SA2_OK) return -1;
    return max64(partial_rows_bytes(prob), two_parts_bytes(prob));
}

int64_t sa2_bwd_workspace_bytes_with_saved(const sa2_problem *prob) {
    if (check_problem(prob) != SA2_OK) return -1;
    return max64(partial_rows_bytes(prob) / 2, two_parts_bytes(prob));
}

// workspace of the dQ/dK2/dV2 pass in `splits`: scatter rows per split, fp32 dq rows per split behind them
static int64_t q_workspace_bytes(const sa2_problem *prob, int splits, bool with_saved) {
    const int64_t scatter = partial_rows_bytes(prob) / (with_saved ? 2 : 1);
    return splits > 1 ? splits * scatter + q_parts_bytes(prob, splits) : scatter;
}

int64_t sa2_bwd_split_workspace_bytes(const sa2_problem *prob, int with_saved) {
    if (check_problem(prob) != SA2_OK) return -1;
    const Kv8Plan plan = kv8_plan(prob);
    const int64_t parts = plan.parts > 1 ? plan.parts * kv_part_bytes(prob) : 0;
    return max64(q_workspace_bytes(prob, bwd_splits(prob), with_saved != 0), parts);
}

// The launches behind sa2_bwd_dq_dkv2, in order on one stream: the MFMA kernel(s) (launch_q_mfma), then dV2 from the forward's
// saved partials and the reduction of the partial rows (launch_q_merge).
struct QLaunch {
    sa2::KParams k;
    float *ws;
    int grid, halo;
    bool use_saved;
    int channels = 256;      // channels of a head that are not zero padding, at most
};

static int prepare_dq_dkv2(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                           const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *dout, const float *lse,
                           const float *delta, const sa2_saved *saved, const sa2_tensor *dq, const sa2_tensor *dk2,
                           const sa2_tensor *dv2, void *workspace, int64_t workspace_bytes, bool may_split, QLaunch *out) {
    sa2::KParams &k = out->k;
    SA2_TRY(bwd_common(prob, q, k1, k2, v1, v2, dout, lse, delta, &k));
    SA2_TRY(check_tensor(dq, "dq"));
    SA2_TRY(check_tensor(dk2, "dk2"));
    SA2_TRY(check_tensor(dv2, "dv2"));
    if (!workspace) return fail(SA2_ERR_NULL_POINTER, "workspace is NULL");
    if ((reinterpret_cast<uintptr_t>(workspace) & 15) != 0) return fail(SA2_ERR_ALIGNMENT, "workspace must be 16-byte aligned");
    // the dK2 partial rows are the first half of the workspace, the dV2 partial rows the second: with saved
    // forward partials dV2 needs none
    const bool saved_given = saved != nullptr;
    const int splits = may_split ? bwd_splits(prob) : 1;
    const int64_t need = q_workspace_bytes(prob, splits, saved_given);
    if (workspace_bytes < need)
        return fail(SA2_ERR_BAD_SHAPE, "workspace of %lld bytes is smaller than the %lld bytes this call needs (sa2_bwd_%sworkspace_bytes%s())",
                    (long long)workspace_bytes, (long long)need, may_split ? "split_" : "", saved_given && !may_split ? "_with_saved" : "");
    k.dq = dev(dq);
    k.dk2 = dev(dk2);
    k.dv2 = dev(dv2);
    out->ws = static_cast<float *>(workspace);
    out->grid = prob->batch * prob->heads * ((prob->seq_len + 31) / 32);
    out->halo = q_halo(prob->w2);
    // with the forward's saved per-offset T the dv2 pass (a recomputation of S and T) is
    // replaced by a kernel that streams T once
    out->use_saved = saved_given;
    out->k.q_ws_stride = partial_rows_bytes(prob) / (saved_given ? 2 : 1) / 4;
    if (splits > 1) {
        k.q_splits = splits;
        k.q_parts = out->ws + splits * k.q_ws_stride;
    }
    if (saved) {
        SA2_TRY(check_saved(prob, saved));
        k.t_save = static_cast<char *>(saved->t);
        k.m_save = saved->m;
    }
    return SA2_OK;
}

static int launch_q_mfma(const sa2_problem *prob, const QLaunch &L, int pass, hipStream_t s) {
    if (prob->dim_head == kWideDimHead) {
        sa2::launch_bwd_wide_q(true, L.grid, s, L.k, L.ws, L.halo);
        if (pass != 1) sa2::launch_bwd_wide_q(false, L.grid, s, L.k, L.ws, L.halo);
        return after_launch("dq/dk2/dv2");
    }
    // At most 96 channels that are not padding (the package: heads of 65 to 96), with partials saved for dV2.  2 x 6 (2 kv) x 2999
    // rows of 96 channels, w1 300, w2 20: 243 us with the general instance, 204 with this one.  Without partials both passes are general.
    const bool narrow = prob->dim_head == 128 && L.channels <= 96 && L.use_saved;
    if (narrow) {
        if (L.k.q_splits > 1) hipLaunchKernelGGL((sa2::bwd_q_kernel<128, true, true, 96>), dim3(L.k.q_splits * L.grid), dim3(512), 0, s, L.k, L.ws, L.halo);
        else hipLaunchKernelGGL((sa2::bwd_q_kernel<128, true, false, 96>), dim3(L.grid), dim3(512), 0, s, L.k, L.ws, L.halo);
        return after_launch("dq/dk2 of narrow heads");
    }
    if (L.k.q_splits > 1) {
        const dim3 sgrid(L.k.q_splits * L.grid);
        SA2_FOR_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL((sa2::bwd_q_kernel<DH, true, true>), sgrid, dim3(512), 0, s, L.k, L.ws, L.halo));
        if (!L.use_saved)
            SA2_FOR_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL((sa2::bwd_q_kernel<DH, false, true>), sgrid, dim3(512), 0, s, L.k, L.ws, L.halo));
        return after_launch("dq/dk2/dv2 in splits");
    }
    SA2_FOR_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL((sa2::bwd_q_kernel<DH, true>), dim3(L.grid), dim3(512), 0, s, L.k, L.ws, L.halo));
    if (pass != 1 && !L.use_saved)
        SA2_FOR_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL((sa2::bwd_q_kernel<DH, false>), dim3(L.grid), dim3(512), 0, s, L.k, L.ws, L.halo));
    return after_launch("dq/dk2/dv2");
}

static int dv2_blocks(const sa2_problem *prob) { return prob->batch * prob->kv_heads * ((prob->seq_len + 31) / 32); }

static int launch_dv2_from_saved(const sa2_problem *prob, const QLaunch &L, hipStream_t s) {
    SA2_FOR_DIM_HEAD(prob->dim_head,
                     hipLaunchKernelGGL(sa2::dv2_from_saved_kernel<DH>, dim3(dv2_blocks(prob)), dim3((sa2::Dv2Cfg<DH, false>::THREADS)), 0, s, L.k));
    return after_launch("dv2 from saved partials");
}

// Up to two dV2 blocks per CU the chains of loads of single workgroups are what dV2, dK2 and dQ take: one launch.  Measured against
// two at 1 to 512 dV2 blocks, 1 to 16 query heads per key/value head, w2 1 to 500 and D = 32, 64, 128, it takes 0.4 to 0.9 of their time; at
// 512 blocks (1 x 16 (4 kv) x 4096 rows), us in a trace, two and one: D = 32 w2 2 17.6, 15.0; D = 64 w2 2 28.2, 16.2; w2 16 48.2, 33.5; w2 128
// 328, 254; D = 128 w2 2 39.2, 21.3; w2 128 493, 448.  The line lies on the safe side: at 2048 blocks one launch of D = 32 and 64 loses at the
// shortest second windows (w2 2, 1 x 4 x 16384 rows of 32: 17.3, 19.8), at 1024 it does not (13.8, 13.0; D = 128 w2 32, 1 x 16 (4 kv) x 8192
// rows: 292, 253).
static int launch_small_grid_merge(const sa2_problem *prob, const QLaunch &L, hipStream_t s) {
    const int64_t k_rows = (int64_t)prob->batch * prob->kv_heads * prob->seq_len, q_rows = (int64_t)prob->batch * prob->heads * prob->seq_len;
    SA2_FOR_DIM_HEAD(prob->dim_head, {
        using C = sa2::MergeCfg<DH>;
        const int k_blocks = (int)((k_rows + C::ROWS - 1) / C::ROWS);
        const int q_blocks = L.k.q_splits > 1 ? (int)((q_rows + C::ROWS - 1) / C::ROWS) : 0;
        hipLaunchKernelGGL(sa2::small_grid_merge_kernel<DH>, dim3(dv2_blocks(prob) + k_blocks + q_blocks), dim3(C::THREADS), 0, s, L.k, L.ws, 32 + L.halo, dv2_blocks(prob), k_blocks);
    });
    return after_launch("dv2, dk2 and dq of a small grid");
}

static int launch_q_combine(const sa2_problem *prob, const QLaunch &L, hipStream_t s) {
    // (split query tiles: a second grid row forms dq)
    const bool dq_too = L.k.q_splits > 1;
    const int64_t rows = (int64_t)prob->batch * (dq_too ? prob->heads : prob->kv_heads) * prob->seq_len;
    const int rows_per_block = 256 / (prob->dim_head / 8);
    const int cgrid = (int)((rows + rows_per_block - 1) / rows_per_block);
    const int with_dv2 = L.use_saved ? 0 : 1;
    SA2_FOR_ANY_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL(sa2::dk2_dv2_combine_kernel<DH>, dim3(cgrid, dq_too ? 2 : 1), dim3(256), 0, s, L.k, L.ws, 32 + L.halo, with_dv2));
    return after_launch("dk2/dv2 combine");
}

static int launch_q_merge(const sa2_problem *prob, const QLaunch &L, hipStream_t s) {
    if (L.use_saved && dv2_blocks(prob) <= 2 * kComputeUnits) return launch_small_grid_merge(prob, L, s);
    if (L.use_saved) SA2_TRY(launch_dv2_from_saved(prob, L, s));
    return launch_q_combine(prob, L, s);
}

int sa2_bwd_dq_dkv2(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                    const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *dout, const float *lse,
                    const float *delta, const sa2_saved *saved, const sa2_tensor *dq, const sa2_tensor *dk2,
                    const sa2_tensor *dv2, void *workspace, int64_t workspace_bytes, void *hip_stream) {
    QLaunch L;
    SA2_TRY(prepare_dq_dkv2(prob, q, k1, k2, v1, v2, dout, lse, delta, saved, dq, dk2, dv2, workspace, workspace_bytes, false, &L));
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    const int pass = bwd_pass_filter();
    SA2_TRY(launch_q_mfma(prob, L, pass, s));
    if (pass == 1) return SA2_OK;    // profiling build, one pass: leave the reductions out of its timing
    return launch_q_merge(prob, L, s);
}

static int launch_dkv1(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                       const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *dout, const float *lse,
                       const float *delta, const sa2_tensor *dk1, const sa2_tensor *dv1, const Kv8Plan &plan, float *parts, void *hip_stream) {
    sa2::KParams k;
    SA2_TRY(bwd_common(prob, q, k1, k2, v1, v2, dout, lse, delta, &k));
    SA2_TRY(check_tensor(dk1, "dk1"));
    SA2_TRY(check_tensor(dv1, "dv1"));
    k.dk1 = dev(dk1);
    k.dv1 = dev(dv1);
    k.kv_parts = parts;
    k.kv_chunk = plan.chunk;
    k.kv_max_parts = plan.parts;
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    const int grid = prob->batch * prob->kv_heads * ((prob->seq_len + 127) / 128);
    // dim_head 256: one wave per SIMD with everything in registers; 128: the two waves of a slab split the contractions (everything
    // in registers takes 6.0 ms there, 4.9 this way); 64 and 32: each wave forms both outputs
    const bool in_parts = plan.parts > 1;
    const dim3 kgrid(in_parts ? plan.parts * grid : grid), block(512);
    if (prob->dim_head == kWideDimHead) {
        sa2::launch_bwd_kvr(in_parts, kgrid.x, s, k);
    } else if (prob->dim_head == 128) {
        if (in_parts) hipLaunchKernelGGL((sa2::bwd_kv8_kernel<128, sa2::kKvSplit, true>), kgrid, block, 0, s, k);
        else hipLaunchKernelGGL((sa2::bwd_kv8_kernel<128, sa2::kKvSplit>), kgrid, block, 0, s, k);
    } else if (prob->dim_head == 64) {
        if (in_parts) hipLaunchKernelGGL((sa2::bwd_kv8_kernel<64, sa2::kKvBoth, true>), kgrid, block, 0, s, k);
        else hipLaunchKernelGGL((sa2::bwd_kv8_kernel<64, sa2::kKvBoth>), kgrid, block, 0, s, k);
    } else {
        if (in_parts) hipLaunchKernelGGL((sa2::bwd_kv8_kernel<32, sa2::kKvBoth, true>), kgrid, block, 0, s, k);
        else hipLaunchKernelGGL((sa2::bwd_kv8_kernel<32, sa2::kKvBoth>), kgrid, block, 0, s, k);
    }
    SA2_TRY(after_launch("dk1/dv1"));
    if (!in_parts) return SA2_OK;
    const int64_t rows = (int64_t)prob->batch * prob->kv_heads * prob->seq_len;
    const int rows_per_block = 256 / (prob->dim_head / 8);
    const int cgrid = (int)((rows + rows_per_block - 1) / rows_per_block);
    SA2_FOR_ANY_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL(sa2::dkv1_parts_combine_kernel<DH>, dim3(cgrid, 2), dim3(256), 0, s, k));
    return after_launch("dk1/dv1 parts combine");
}

int sa2_bwd_dkv1(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                 const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *dout, const float *lse,
                 const float *delta, const sa2_tensor *dk1, const sa2_tensor *dv1, void *hip_stream) {
    return launch_dkv1(prob, q, k1, k2, v1, v2, dout, lse, delta, dk1, dv1, Kv8Plan{0, 1}, nullptr, hip_stream);
}

static int bwd_all(bool split, int channels, const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
            const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *out, const sa2_tensor *out_residual,
            const sa2_tensor *dout, const float *lse, const sa2_saved *saved, float *delta_ws, const sa2_tensor *dq,
            const sa2_tensor *dk1, const sa2_tensor *dk2, const sa2_tensor *dv1, const sa2_tensor *dv2, void *workspace,
            int64_t workspace_bytes, void *hip_stream) {
    SA2_TRY(check_problem(prob));
    // every size and pointer is checked before the first launch: a call that fails has written nothing
    const Kv8Plan plan = split ? kv8_plan(prob) : two_part_plan(prob);
    const int64_t need = plan.parts > 1 ? plan.parts * kv_part_bytes(prob) : 0;
    if (workspace_bytes < need)
        return fail(SA2_ERR_BAD_SHAPE, "workspace of %lld bytes is smaller than the %lld bytes this problem's dk1/dv1 pass needs (sa2_bwd_%s())",
                    (long long)workspace_bytes, (long long)need, split ? "split_workspace_bytes" : "workspace_bytes");
    if (!delta_ws) return fail(SA2_ERR_NULL_POINTER, "delta is NULL");
    SA2_TRY(check_tensor(out, "out"));
    if (out_residual) SA2_TRY(check_tensor(out_residual, "out_residual"));
    SA2_TRY(check_tensor(dk1, "dk1"));
    SA2_TRY(check_tensor(dv1, "dv1"));
    QLaunch L;
    SA2_TRY(prepare_dq_dkv2(prob, q, k1, k2, v1, v2, dout, lse, delta_ws, saved, dq, dk2, dv2, workspace, workspace_bytes, split, &L));
    L.channels = channels;
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    if (L.k.q_splits <= 1) {
        SA2_TRY(sa2_bwd_delta(prob, out, out_residual, dout, delta_ws, hip_stream));
    } else {
        // a split dQ/dK2 kernel forms delta itself and leaves it in delta_ws
        L.k.o = dev(out);
        if (out_residual) L.k.o_lo = dev(out_residual);
    }
    SA2_TRY(launch_q_mfma(prob, L, 0, s));
    SA2_TRY(launch_q_merge(prob, L, s));
    // the partial rows of dK2/dV2 are spent by now: the partial results of split key slabs reuse the workspace
    return launch_dkv1(prob, q, k1, k2, v1, v2, dout, lse, delta_ws, dk1, dv1, plan, static_cast<float *>(workspace), hip_stream);
}

int sa2_bwd(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
            const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *out, const sa2_tensor *out_residual,
            const sa2_tensor *dout, const float *lse, const sa2_saved *saved, float *delta_ws, const sa2_tensor *dq,
            const sa2_tensor *dk1, const sa2_tensor *dk2, const sa2_tensor *dv1, const sa2_tensor *dv2, void *workspace,
            int64_t workspace_bytes, void *hip_stream) {
    return bwd_all(false, 256, prob, q, k1, k2, v1, v2, out, out_residual, dout, lse, saved, delta_ws, dq, dk1, dk2, dv1, dv2, workspace,
                   workspace_bytes, hip_stream);
}

int sa2_bwd_split(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                  const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *out, const sa2_tensor *out_residual,
                  const sa2_tensor *dout, const float *lse, const sa2_saved *saved, float *delta_ws, const sa2_tensor *dq,
                  const sa2_tensor *dk1, const sa2_tensor *dk2, const sa2_tensor *dv1, const sa2_tensor *dv2, void *workspace,
                  int64_t workspace_bytes, void *hip_stream) {
    return bwd_all(true, 256, prob, q, k1, k2, v1, v2, out, out_residual, dout, lse, saved, delta_ws, dq, dk1, dk2, dv1, dv2, workspace,
                   workspace_bytes, hip_stream);
}

int sa2_bwd_split_padded(const sa2_problem *prob, int32_t channels, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                         const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *out, const sa2_tensor *out_residual,
                         const sa2_tensor *dout, const float *lse, const sa2_saved *saved, float *delta_ws, const sa2_tensor *dq,
                         const sa2_tensor *dk1, const sa2_tensor *dk2, const sa2_tensor *dv1, const sa2_tensor *dv2, void *workspace,
                         int64_t workspace_bytes, void *hip_stream) {
    SA2_TRY(check_problem(prob));
    if (channels < 1 || channels > prob->dim_head)
        return fail(SA2_ERR_BAD_SHAPE, "channels=%d: 1 to dim_head=%d of them are not padding", (int)channels, prob->dim_head);
    return bwd_all(true, channels, prob, q, k1, k2, v1, v2, out, out_residual, dout, lse, saved, delta_ws, dq, dk1, dk2, dv1, dv2, workspace,
                   workspace_bytes, hip_stream);
}

static int64_t align256(int64_t x) { return (x + 255) & ~int64_t(255); }

int64_t sa2_bwd_noalloc_scratch_bytes(const sa2_problem *prob) {
    const int64_t ws = sa2_bwd_workspace_bytes(prob);
    if (ws < 0) return -1;
    return align256((int64_t)prob->batch * prob->heads * prob->seq_len * 4) + ws;
}

int sa2_bwd_noalloc(const sa2_problem *prob, const sa2_tensor *q, const sa2_tensor *k1, const sa2_tensor *k2,
                    const sa2_tensor *v1, const sa2_tensor *v2, const sa2_tensor *out, const sa2_tensor *out_residual,
                    const sa2_tensor *dout, const float *lse, const sa2_saved *saved, const sa2_tensor *dq,
                    const sa2_tensor *dk1, const sa2_tensor *dk2, const sa2_tensor *dv1, const sa2_tensor *dv2,
                    void *hip_stream) {
    SA2_TRY(check_problem(prob));
    const int64_t need = sa2_bwd_noalloc_scratch_bytes(prob);
    if (need > kNoallocScratchBytes)
        return fail(SA2_ERR_UNSUPPORTED, "this problem needs %lld bytes of scratch, the built-in buffer of sa2_bwd_noalloc holds %lld; "
                    "use sa2_bwd with a caller-owned workspace", (long long)need, (long long)kNoallocScratchBytes);
    unsigned char *scratch = nullptr;
    SA2_TRY(noalloc_scratch(&scratch));
    float *delta = reinterpret_cast<float *>(scratch);
    unsigned char *ws = scratch + align256((int64_t)prob->batch * prob->heads * prob->seq_len * 4);
    // every element of the scratch that a kernel reads was written by an earlier kernel of this same
    // call (delta rows, partial rows), so nothing needs clearing between calls
    return sa2_bwd(prob, q, k1, k2, v1, v2, out, out_residual, dout, lse, saved, delta, dq, dk1, dk2, dv1, dv2, ws,
                   sa2_bwd_workspace_bytes(prob), hip_stream);
}

// ---- type and head dimension conversion
int sa2_convert(const sa2_conversion *items, int32_t count, void *hip_stream) {
    static_assert(SA2_CONVERT_MOST == sa2::kConvertMost, "tensors per launch");
    if (!items) return fail(SA2_ERR_NULL_POINTER, "items is NULL");
    if (count < 1 || count > SA2_CONVERT_MOST) return fail(SA2_ERR_BAD_SHAPE, "%d conversions: 1 to %d fit one call", count, SA2_CONVERT_MOST);
    sa2::ConvertParams p{};
    int64_t most = 0;
    for (int x = 0; x < count; ++x) {
        const sa2_conversion &c = items[x];
        if (!c.src.ptr || !c.dst.ptr) return fail(SA2_ERR_NULL_POINTER, "conversion %d: src or dst is NULL", x);
        if (c.batch < 1 || c.seq_len < 1 || c.heads < 1 || c.src_dim < 1 || c.dst_dim < 1)
            return fail(SA2_ERR_BAD_SHAPE, "conversion %d: sizes must be >= 1", x);
        if (c.src_type < 0 || c.src_type > SA2_ELEMENT_F32 || c.dst_type < 0 || c.dst_type > SA2_ELEMENT_F32)
            return fail(SA2_ERR_UNSUPPORTED, "conversion %d: unknown element type", x);
        sa2::ConvertTensor &t = p.t[x];
        auto vec = [](const sa2_tensor &a, int type) {
            const int per16 = type == SA2_ELEMENT_F32 ? 4 : 8;
            return (reinterpret_cast<uintptr_t>(a.ptr) & 15) == 0 && a.stride_b % per16 == 0 && a.stride_n % per16 == 0 && a.stride_h % per16 == 0;
        };
        t.src = static_cast<const char *>(c.src.ptr);
        t.dst = static_cast<char *>(c.dst.ptr);
        t.ssb = c.src.stride_b;
        t.ssn = c.src.stride_n;
        t.ssh = c.src.stride_h;
        t.dsb = c.dst.stride_b;
        t.dsn = c.dst.stride_n;
        t.dsh = c.dst.stride_h;
        t.src_type = c.src_type;
        t.dst_type = c.dst_type;
        t.src_dim = c.src_dim;
        t.dst_dim = c.dst_dim;
        t.N = c.seq_len;
        t.H = c.heads;
        t.pieces = (int64_t)c.batch * c.seq_len * c.heads * ((c.dst_dim + 7) / 8);
        t.src_vec = vec(c.src, c.src_type);
        t.dst_vec = vec(c.dst, c.dst_type);
        most = t.pieces > most ? t.pieces : most;
    }
    const int64_t blocks = (most + 255) / 256;
    const int grid = (int)(blocks < 16 * kComputeUnits ? blocks : 16 * kComputeUnits);
    hipLaunchKernelGGL(sa2::convert_kernel, dim3(grid, count), dim3(256), 0, static_cast<hipStream_t>(hip_stream), p);
    return after_launch("convert");
}

// ---- fused split + per-head RMSNorm of the qkv projection -------------------------------
static constexpr int kNormMaxBlocks = 2048;

static int norm_groups(const sa2_problem *prob) {
    const int64_t rows = (int64_t)prob->batch * prob->seq_len * (prob->heads + 4 * prob->kv_heads);
    const int rpb = 256 / (prob->dim_head / 8);
    return (int)((rows + rpb - 1) / rpb);
}

static int norm_common(const sa2_problem *prob, const void *qkv, int64_t row_stride, const sa2_tensor *const t[5],
                       const void *const w[5], const float *rstd, sa2::NormParams *np) {
    SA2_TRY(check_problem(prob));
    if (!qkv) return fail(SA2_ERR_NULL_POINTER, "qkv is NULL");
    if (!rstd) return fail(SA2_ERR_NULL_POINTER, "rstd is NULL");
    const int64_t channels = (int64_t)(prob->heads + 4 * prob->kv_heads) * prob->dim_head;
    if (row_stride < channels) return fail(SA2_ERR_BAD_SHAPE, "row_stride %lld is smaller than the %lld channels of a token",
                                           (long long)row_stride, (long long)channels);
    if ((reinterpret_cast<uintptr_t>(qkv) & 15) != 0 || row_stride % 8 != 0)
        return fail(SA2_ERR_ALIGNMENT, "qkv rows must be 16-byte aligned");
    static const char *names[5] = {"q", "k1", "k2", "v1", "v2"};
    *np = sa2::NormParams{};
    for (int x = 0; x < 5; ++x) {
        SA2_TRY(check_tensor(t[x], names[x]));
        np->t[x] = dev(t[x]);
        if (w[x] && (reinterpret_cast<uintptr_t>(w[x]) & 15) != 0) return fail(SA2_ERR_ALIGNMENT, "norm weights must be 16-byte aligned");
        np->w[x] = static_cast<const char *>(w[x]);
    }
    np->qkv = static_cast<const char *>(qkv);
    np->row_stride = row_stride * 2;
    np->rstd = const_cast<float *>(rstd);
    np->B = prob->batch;
    np->N = prob->seq_len;
    np->H = prob->heads;
    np->HK = prob->kv_heads;
    return SA2_OK;
}

int sa2_qkv_norm_fwd(const sa2_problem *prob, const void *qkv, int64_t row_stride, const void *w_q, const void *w_k1,
                     const void *w_k2, const void *w_v1, const void *w_v2, float eps, const sa2_tensor *q,
                     const sa2_tensor *k1, const sa2_tensor *k2, const sa2_tensor *v1, const sa2_tensor *v2, float *rstd,
                     void *hip_stream) {
    const sa2_tensor *const t[5] = {q, k1, k2, v1, v2};
    const void *const w[5] = {w_q, w_k1, w_k2, w_v1, w_v2};
    sa2::NormParams np;
    SA2_TRY(norm_common(prob, qkv, row_stride, t, w, rstd, &np));
    np.eps = eps;
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    const int grid = norm_groups(prob);
    SA2_FOR_ANY_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL(sa2::qkv_norm_fwd_kernel<DH>, dim3(grid), dim3(256), 0, s, np));
    return after_launch("qkv norm forward");
}

int64_t sa2_qkv_norm_bwd_workspace_bytes(const sa2_problem *prob) {
    if (check_problem(prob) != SA2_OK) return -1;
    const int groups = norm_groups(prob);
    const int blocks = groups < kNormMaxBlocks ? groups : kNormMaxBlocks;
    return (int64_t)blocks * 5 * prob->dim_head * 4;
}

int sa2_qkv_norm_bwd(const sa2_problem *prob, const void *qkv, int64_t row_stride, const void *w_q, const void *w_k1,
                     const void *w_k2, const void *w_v1, const void *w_v2, const sa2_tensor *dq, const sa2_tensor *dk1,
                     const sa2_tensor *dk2, const sa2_tensor *dv1, const sa2_tensor *dv2, const float *rstd, void *dqkv,
                     float *dw, void *workspace, int64_t workspace_bytes, void *hip_stream) {
    const sa2_tensor *const t[5] = {dq, dk1, dk2, dv1, dv2};
    const void *const w[5] = {w_q, w_k1, w_k2, w_v1, w_v2};
    sa2::NormParams np;
    SA2_TRY(norm_common(prob, qkv, row_stride, t, w, rstd, &np));
    if (!dqkv || !dw || !workspace) return fail(SA2_ERR_NULL_POINTER, "dqkv, dw or workspace is NULL");
    if ((reinterpret_cast<uintptr_t>(dqkv) & 15) != 0) return fail(SA2_ERR_ALIGNMENT, "dqkv must be 16-byte aligned");
    const int64_t need = sa2_qkv_norm_bwd_workspace_bytes(prob);
    if (workspace_bytes < need)
        return fail(SA2_ERR_BAD_SHAPE, "workspace of %lld bytes is smaller than the %lld bytes sa2_qkv_norm_bwd_workspace_bytes() asks for",
                    (long long)workspace_bytes, (long long)need);
    np.dqkv = static_cast<char *>(dqkv);
    np.dw_part = static_cast<float *>(workspace);
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    const int groups = norm_groups(prob);
    const int blocks = groups < kNormMaxBlocks ? groups : kNormMaxBlocks;
    SA2_FOR_ANY_DIM_HEAD(prob->dim_head, hipLaunchKernelGGL(sa2::qkv_norm_bwd_kernel<DH>, dim3(blocks), dim3(256), 0, s, np, groups));
    SA2_TRY(after_launch("qkv norm backward"));
    const int n = 5 * prob->dim_head;
    hipLaunchKernelGGL(sa2::qkv_norm_dw_kernel, dim3((n + 15) / 16), dim3(1024), 0, s, np.dw_part, dw, blocks, n);
    return after_launch("qkv norm weight gradients");
}

// ---- weight gradient of a linear layer
// Shares of the rows: two workgroups per CU, at least sixteen 32-row tiles each.  16384 rows, 1536 x 512 (us): one workgroup per
// CU 48, two 45, three 56 (the partial blocks are written and read once); 16384 rows, 256 x 512: sixteen tiles 21, eight 27.
static int wgrad_shares(int64_t rows, int out_features, int in_features, int *share_tiles) {
    const int64_t tiles = (rows + 31) / 32, blocks = (int64_t)(out_features / 128) * (in_features / 128);
    int64_t shares = 2 * kComputeUnits / blocks;
    shares = shares < tiles / 16 ? shares : tiles / 16;
    shares = shares < 1 ? 1 : shares;
    const int64_t per = (tiles + shares - 1) / shares;
    *share_tiles = (int)per;
    return (int)((tiles + per - 1) / per);
}

static bool wgrad_fits(int64_t rows, int out_features, int in_features) {
    return rows >= 1 && rows < (1ll << 30) && out_features >= 128 && out_features % 128 == 0 && in_features >= 128 && in_features % 128 == 0;
}

int64_t sa2_wgrad_workspace_bytes(int64_t rows, int32_t out_features, int32_t in_features) {
    if (!wgrad_fits(rows, out_features, in_features)) return -1;
    int per;
    return (int64_t)wgrad_shares(rows, out_features, in_features, &per) * out_features * in_features * 4;
}

int sa2_wgrad(const void *dy, int64_t dy_stride, const void *x, int64_t x_stride, int64_t rows, int32_t out_features, int32_t in_features, void *dw,
              void *workspace, int64_t workspace_bytes, void *hip_stream) {
    if (!dy || !x || !dw || !workspace) return fail(SA2_ERR_NULL_POINTER, "dy, x, dw or workspace is NULL");
    if (!wgrad_fits(rows, out_features, in_features))
        return fail(SA2_ERR_BAD_SHAPE, "rows=%lld must be positive, out_features=%d and in_features=%d multiples of 128", (long long)rows, out_features, in_features);
    if (dy_stride < out_features || x_stride < in_features || dy_stride > (1 << 24) || x_stride > (1 << 24))
        return fail(SA2_ERR_BAD_SHAPE, "row strides %lld and %lld do not hold rows of %d and %d", (long long)dy_stride, (long long)x_stride, out_features, in_features);
    if (((reinterpret_cast<uintptr_t>(dy) | reinterpret_cast<uintptr_t>(x) | reinterpret_cast<uintptr_t>(dw) | reinterpret_cast<uintptr_t>(workspace)) & 15) != 0 ||
        dy_stride % 8 != 0 || x_stride % 8 != 0)
        return fail(SA2_ERR_ALIGNMENT, "dy, x, dw, workspace and the rows must be 16-byte aligned");
    if (workspace_bytes < sa2_wgrad_workspace_bytes(rows, out_features, in_features)) return fail(SA2_ERR_BAD_SHAPE, "the workspace is too small (sa2_wgrad_workspace_bytes())");
    sa2::WgradParams p{};
    p.dy = static_cast<const char *>(dy);
    p.x = static_cast<const char *>(x);
    p.dy_row = dy_stride * 2;
    p.x_row = x_stride * 2;
    p.parts = static_cast<float *>(workspace);
    p.dw = static_cast<char *>(dw);
    p.K = (int)rows;
    p.M = out_features;
    p.N = in_features;
    p.shares = wgrad_shares(rows, out_features, in_features, &p.share_tiles);
    const int64_t blocks = (int64_t)(out_features / 128) * (in_features / 128) * p.shares;
    if (blocks > 0x7fffffffll) return fail(SA2_ERR_BAD_SHAPE, "problem too large for a 1-D grid");
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    hipLaunchKernelGGL(sa2::wgrad_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p);
    SA2_TRY(after_launch("weight gradient"));
    const int64_t cgrid = ((int64_t)out_features * in_features / 8 + 255) / 256;
    hipLaunchKernelGGL(sa2::wgrad_combine_kernel, dim3((unsigned)cgrid), dim3(256), 0, s, p);
    return after_launch("weight gradient combine");
}

#ifdef SA2_PROFILING
// Profiling build only: the instruction-mix loop of sa2_prof_mix.hpp.  `operands`: 64 KiB of bf16 values on the device,
// `out`: workgroups * 512 floats, `clocks`: two 64-bit counters (shader clock, 100 MHz clock) of workgroup 0.  Each SIMD
// executes workgroups / 256 * iters * 32 MFMAs (two waves of 16).  mix: 0 = MFMAs only; 1 = + 4 VALU, 1 exponential and
// 1 LDS fragment read per MFMA; 2 = + 7 VALU, 1 exponential and 2 LDS fragment reads per MFMA.
int sa2_prof_mfma_mix(const void *operands, float *out, unsigned long long *clocks, int mix, int workgroups, int iters, void *hip_stream) {
    if (!operands || !out || !clocks) return fail(SA2_ERR_NULL_POINTER, "operands, out or clocks is NULL");
    if (workgroups < 1 || iters < 1) return fail(SA2_ERR_BAD_SHAPE, "workgroups and iters must be positive");
    hipStream_t s = static_cast<hipStream_t>(hip_stream);
    const char *src = static_cast<const char *>(operands);
    if (mix == 0) hipLaunchKernelGGL((sa2::prof_mix_kernel<0, 0, 0>), dim3(workgroups), dim3(512), 0, s, src, out, iters, clocks);
    else if (mix == 1) hipLaunchKernelGGL((sa2::prof_mix_kernel<4, 1, 1>), dim3(workgroups), dim3(512), 0, s, src, out, iters, clocks);
    else if (mix == 2) hipLaunchKernelGGL((sa2::prof_mix_kernel<7, 1, 2>), dim3(workgroups), dim3(512), 0, s, src, out, iters, clocks);
    else return fail(SA2_ERR_UNSUPPORTED, "mix %d is not one of 0, 1, 2", mix);
    return after_launch("instruction-mix loop");
}
#endif

}  // extern "C"
