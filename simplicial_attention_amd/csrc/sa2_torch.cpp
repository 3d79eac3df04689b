// Host path of the package's autograd Functions: argument checks, allocation, the launches of libsa2 and the autograd
// nodes, in one native call per direction.  (From Python through ctypes the same work took 25 us for a forward and 150 us
// for a forward and backward, which is what small calls then cost whatever the kernels do.)
//
// Bound to Python as the module _sa2_torch; two_simplicial_attention.py and qkv_norm.py are its callers.
#include <torch/extension.h>

#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>

#include <array>
#include <atomic>

#include "sa2.h"

namespace py = pybind11;
using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

constexpr int kMostDevices = 64;
// bytes of saved partials that have died, per device (the budget in Python subtracts them from what it admitted)
std::array<std::atomic<int64_t>, kMostDevices> g_released{};

void check(int status) {
    if (status == SA2_OK) return;
    // the exception class of the package (Sa2Error) is raised by its own check function
    py::gil_scoped_acquire gil;
    py::module_::import("simplicial_attention_amd._native").attr("check_failed")(status, std::string(sa2_last_error()));
}

[[noreturn]] void raise(PyObject *type, const std::string &text) {
    py::gil_scoped_acquire gil;
    PyErr_SetString(type, text.c_str());
    throw py::error_already_set();
}

void *stream_of(const Tensor &t) { return c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream(); }

sa2_tensor arg(const Tensor &t) { return {t.data_ptr(), t.stride(0), t.stride(1), t.stride(2)}; }

// the kernels need a unit innermost stride, 16-byte aligned rows and base, rows within reach of each other
Tensor aligned(const Tensor &t) {
    const bool ok = t.stride(3) == 1 && (t.size(1) == 1 || t.stride(1) <= SA2_MOST_STRIDE_N) && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0 && t.stride(0) % 8 == 0 && t.stride(1) % 8 == 0 &&
                    t.stride(2) % 8 == 0;
    return ok ? t : t.clone(at::MemoryFormat::Contiguous);
}

int element_of(const Tensor &t) {
    switch (t.scalar_type()) {
        case at::kBFloat16: return SA2_ELEMENT_BF16;
        case at::kHalf: return SA2_ELEMENT_F16;
        case at::kFloat: return SA2_ELEMENT_F32;
        default: return -1;
    }
}

// Several conversions in one launch.
struct Conversions {
    sa2_conversion items[SA2_CONVERT_MOST];
    int count = 0;
    void add(const Tensor &src, const Tensor &dst) {
        sa2_conversion &c = items[count++];
        c.src = arg(src);
        c.dst = arg(dst);
        c.src_type = element_of(src);
        c.dst_type = element_of(dst);
        c.src_dim = (int)src.size(3);
        c.dst_dim = (int)dst.size(3);
        c.batch = (int)src.size(0);
        c.seq_len = (int)src.size(1);
        c.heads = (int)src.size(2);
    }
    void run(void *stream) {
        if (count) check(sa2_convert(items, count, stream));
    }
};

Tensor rows_of(const Tensor &t) { return t.stride(3) == 1 ? t : t.contiguous(); }

// a (b, n, h, d) tensor as bf16 rows of `dim` channels, converted if it is not that already (the conversion is queued)
Tensor as_rows(const Tensor &t, int64_t dim, Conversions &todo, std::vector<Tensor> &alive) {
    if (t.scalar_type() == at::kBFloat16 && t.size(3) == dim) return aligned(t);
    Tensor src = rows_of(t), dst = at::empty({t.size(0), t.size(1), t.size(2), dim}, t.options().dtype(at::kBFloat16));
    todo.add(src, dst);
    alive.push_back(src);
    return dst;
}

struct Geometry {
    int64_t batch, seq, heads, kv_heads, dim_qk, dim_v, dim;      // dim: the kernels' head dimension
    int64_t w1, w2;
    double scale;
    sa2_problem problem() const {
        return {(int32_t)batch, (int32_t)seq, (int32_t)heads, (int32_t)kv_heads, (int32_t)dim, (int32_t)w1, (int32_t)w2, 1, (float)scale, SA2_BF16};
    }
};

struct Forward {
    Tensor q, k1, k2, v1, v2;          // the kernels' operands
    Tensor out, lse, residual, t_save, m_save, note;
    Tensor result;                     // out in the caller's type and head dimension
};

// An empty tensor that reports `counted` bytes as released when it dies.  It is saved beside the partials and shares their fate;
// these are ordinary tensors, whose memory the allocator keeps for other streams where record_stream asks for it.
Tensor release_note(const Tensor &partials, int64_t counted) {
    const int device = partials.device().index();
    return at::for_blob(partials.data_ptr(), {0})
        .deleter([device, counted](void *) { g_released[device].fetch_add(counted); })
        .options(partials.options())
        .target_device(partials.device())
        .make_tensor();
}

// `admit` (given where a backward may follow): called with the bytes of the per-offset value partials, says whether they may be
// kept for the backward, in which dV2 then needs no recomputation of the attention weights
Forward run_forward(const Tensor &q, const Tensor &k1, const Tensor &k2, const Tensor &v1, const Tensor &v2, const Geometry &g, const py::object *admit) {
    Forward f;
    const c10::DeviceGuard guard(q.device());
    void *stream = stream_of(q);
    Conversions todo;
    std::vector<Tensor> alive;
    f.q = as_rows(q, g.dim, todo, alive);
    f.k1 = as_rows(k1, g.dim, todo, alive);
    f.k2 = as_rows(k2, g.dim, todo, alive);
    f.v1 = as_rows(v1, g.dim, todo, alive);
    f.v2 = as_rows(v2, g.dim, todo, alive);
    todo.run(stream);
    const auto bf16 = q.options().dtype(at::kBFloat16);
    f.out = at::empty({g.batch, g.seq, g.heads, g.dim}, bf16);
    f.lse = at::empty({g.batch, g.heads, g.seq}, q.options().dtype(at::kFloat));
    // bf16 residual of the fp32 accumulator, kept only when a backward may follow
    if (admit) f.residual = at::empty({g.batch, g.seq, g.heads, g.dim}, bf16);
    const sa2_problem prob = g.problem();
    sa2_saved saved{};
    // (a size of 0: the kernels of this head dimension keep none; asked last, so that nothing that fails stands between the
    // admission and the buffers that it is for)
    const int64_t t_bytes = sa2_saved_t_bytes(&prob), m_bytes = sa2_saved_m_bytes(&prob);
    const bool save = admit && t_bytes + m_bytes > 0 && (*admit)(t_bytes + m_bytes, (int)q.device().index()).cast<bool>();
    if (save) {
        try {
            f.t_save = at::empty({t_bytes}, q.options().dtype(at::kByte));
            f.m_save = at::empty({g.batch, g.heads, g.w2, g.seq}, f.lse.options());
            f.note = release_note(f.t_save, t_bytes + m_bytes);
        } catch (...) {
            g_released[q.device().index()].fetch_add(t_bytes + m_bytes);      // (nothing to hang the report on)
            throw;
        }
        saved = {f.t_save.data_ptr(), static_cast<float *>(f.m_save.data_ptr())};
    }
    const int64_t ws_bytes = sa2_fwd_workspace_bytes(&prob);
    Tensor ws;
    if (ws_bytes > 0) ws = at::empty({ws_bytes}, q.options().dtype(at::kByte));
    const sa2_tensor aq = arg(f.q), ak1 = arg(f.k1), ak2 = arg(f.k2), av1 = arg(f.v1), av2 = arg(f.v2), ao = arg(f.out);
    sa2_tensor ar{};
    if (admit) ar = arg(f.residual);
    check(sa2_fwd_ws(&prob, &aq, &ak1, &ak2, &av1, &av2, &ao, admit ? &ar : nullptr, static_cast<float *>(f.lse.data_ptr()),
                     save ? &saved : nullptr, ws_bytes > 0 ? ws.data_ptr() : nullptr, ws_bytes, stream));
    if (q.scalar_type() == at::kBFloat16 && g.dim_v == g.dim) {
        f.result = f.out;
    } else {
        f.result = at::empty({g.batch, g.seq, g.heads, g.dim_v}, q.options());
        Conversions back;
        back.add(f.out, f.result);
        back.run(stream);
    }
    return f;
}

struct Attend : public torch::autograd::Function<Attend> {
    static Tensor forward(AutogradContext *ctx, const Tensor &q, const Tensor &k1, const Tensor &k2, const Tensor &v1, const Tensor &v2,
                          const Geometry &g, const py::object &admit) {
        Forward f = run_forward(q, k1, k2, v1, v2, g, &admit);
        ctx->save_for_backward(saved_of(f));
        ctx->saved_data["geometry"] = c10::List<int64_t>(sizes_of(g, {&q, &k1, &k2, &v1, &v2}));
        ctx->saved_data["scale"] = g.scale;
        return f.result;
    }

    static variable_list backward(AutogradContext *ctx, variable_list douts) {
        variable_list grads = run_backward(ctx->get_saved_variables(), ctx->saved_data["geometry"].toIntVector(), ctx->saved_data["scale"].toDouble(), douts[0]);
        grads.resize(7);
        return grads;
    }

    // what the backward needs of a forward: tensors, and as numbers the geometry and the types of the inputs
    static variable_list saved_of(const Forward &f) { return {f.q, f.k1, f.k2, f.v1, f.v2, f.out, f.lse, f.residual, f.t_save, f.m_save, f.note}; }
    static std::vector<int64_t> sizes_of(const Geometry &g, const std::array<const Tensor *, 5> &inputs) {
        std::vector<int64_t> n{g.batch, g.seq, g.heads, g.kv_heads, g.dim_qk, g.dim_v, g.dim, g.w1, g.w2};
        for (const Tensor *t : inputs) n.push_back((int64_t)t->scalar_type());
        return n;
    }

    static variable_list run_backward(const variable_list &s, const std::vector<int64_t> &n, double scale, const Tensor &given) {
        const Tensor &q = s[0], &k1 = s[1], &k2 = s[2], &v1 = s[3], &v2 = s[4], &out = s[5], &lse = s[6], &residual = s[7], &t_save = s[8], &m_save = s[9];
        Geometry g;
        g.batch = n[0]; g.seq = n[1]; g.heads = n[2]; g.kv_heads = n[3]; g.dim_qk = n[4]; g.dim_v = n[5]; g.dim = n[6]; g.w1 = n[7]; g.w2 = n[8];
        g.scale = scale;
        const c10::DeviceGuard guard(q.device());
        void *stream = stream_of(q);
        Conversions todo;
        std::vector<Tensor> alive;
        const Tensor dout = as_rows(given, g.dim, todo, alive);
        todo.run(stream);
        const auto bf16 = q.options();
        const std::array<int64_t, 4> q_shape{g.batch, g.seq, g.heads, g.dim}, kv_shape{g.batch, g.seq, g.kv_heads, g.dim};
        variable_list grads(5);
        for (int x = 0; x < 5; ++x) grads[x] = at::empty(x == 0 ? q_shape : kv_shape, bf16);
        const sa2_problem prob = g.problem();
        sa2_saved saved{};
        const bool have_saved = t_save.defined();
        if (have_saved) saved = {t_save.data_ptr(), static_cast<float *>(m_save.data_ptr())};
        // delta rows and the kernels' workspace in one buffer
        const int64_t delta_bytes = (g.batch * g.heads * g.seq * 4 + 255) / 256 * 256, ws_bytes = sa2_bwd_split_workspace_bytes(&prob, have_saved);
        const Tensor ws = at::empty({delta_bytes + ws_bytes}, q.options().dtype(at::kByte));
        char *base = static_cast<char *>(ws.data_ptr());
        const sa2_tensor aq = arg(q), ak1 = arg(k1), ak2 = arg(k2), av1 = arg(v1), av2 = arg(v2), ao = arg(out), ar = arg(residual), ad = arg(dout);
        sa2_tensor ag[5];
        for (int x = 0; x < 5; ++x) ag[x] = arg(grads[x]);
        check(sa2_bwd_split_padded(&prob, (int32_t)std::max(g.dim_qk, g.dim_v), &aq, &ak1, &ak2, &av1, &av2, &ao, &ar, &ad,
                                   static_cast<float *>(lse.data_ptr()), have_saved ? &saved : nullptr, reinterpret_cast<float *>(base), &ag[0], &ag[1], &ag[2], &ag[3], &ag[4], base + delta_bytes, ws_bytes, stream));
        // back to the types and head dimensions of the inputs
        Conversions back;
        variable_list result(5);
        for (int x = 0; x < 5; ++x) {
            const auto type = (at::ScalarType)n[9 + x];
            const int64_t dim = x < 3 ? g.dim_qk : g.dim_v;
            if (type == at::kBFloat16 && dim == g.dim) {
                result[x] = grads[x];
            } else {
                result[x] = at::empty({g.batch, g.seq, x == 0 ? g.heads : g.kv_heads, dim}, q.options().dtype(type));
                back.add(grads[x], result[x]);
            }
        }
        back.run(stream);
        return result;
    }
};

int64_t kernel_dim(int64_t dim) {
    for (const int64_t d : {32, 64, 128, 256})
        if (dim <= d) return d;
    return 0;
}

Geometry geometry_of(const Tensor &q, const Tensor &k1, const Tensor &v1, int64_t w1, int64_t w2, double scale) {
    Geometry g;
    g.batch = q.size(0);
    g.seq = q.size(1);
    g.heads = q.size(2);
    g.kv_heads = k1.size(2);
    g.dim_qk = q.size(3);
    g.dim_v = v1.size(3);
    g.dim = kernel_dim(std::max(g.dim_qk, g.dim_v));
    g.w1 = w1;
    g.w2 = w2;
    g.scale = scale;
    return g;
}

// a call that autograd has to see: a backward may follow, or an input carries a forward-mode tangent (which the node refuses,
// also without a graph: the derivative would be lost without a word)
bool in_autograd(std::initializer_list<const Tensor *> inputs) {
    for (const Tensor *t : inputs)
        if ((at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(0).defined()) return true;
    return false;
}

Tensor attend(const Tensor &q, const Tensor &k1, const Tensor &k2, const Tensor &v1, const Tensor &v2, const Geometry &g, const py::object &admit) {
    if (!in_autograd({&q, &k1, &k2, &v1, &v2})) return run_forward(q, k1, k2, v1, v2, g, nullptr).result;
    return Attend::apply(q, k1, k2, v1, v2, g, admit);
}

// shapes, types and windows of the Function and the wrapper; `pads`: other head dimensions and types than the kernels' are welcome
Geometry checked(const Tensor &q, const Tensor &k1, const Tensor &k2, const Tensor &v1, const Tensor &v2, int64_t w1, int64_t w2,
                 std::optional<double> scale, bool pads) {
    const Tensor *all[5] = {&q, &k1, &k2, &v1, &v2};
    for (const Tensor *t : all)
        if (!t->is_cuda()) raise(PyExc_AssertionError, "sliding-window 2-simplicial attention runs on the GPU only");
    for (const Tensor *t : all)
        if (element_of(*t) < 0 || (!pads && t->scalar_type() != q.scalar_type()))
            raise(PyExc_TypeError, "q, k1, k2, v1, v2 must share one dtype out of bfloat16, float16, float32");
    if (q.dim() != 4) raise(PyExc_ValueError, "expected (batch, seq, heads, dim_head) tensors");
    for (const Tensor *t : all)
        if (t->dim() != 4 || t->size(0) != q.size(0) || t->size(1) != q.size(1) || (t != &q && t->size(2) != k1.size(2)) ||
            t->size(3) != (t == &v1 || t == &v2 ? (pads ? v1 : q) : q).size(3) || t->device() != q.device())
            raise(PyExc_ValueError, "key/value shape " + std::string(py::str(py::cast(t->sizes().vec()))) + " does not match the queries' " +
                                        std::string(py::str(py::cast(q.sizes().vec()))));
    if (k1.size(2) < 1 || q.size(2) % k1.size(2) != 0)
        raise(PyExc_ValueError, "query heads " + std::to_string(q.size(2)) + " not divisible by key/value heads " + std::to_string(k1.size(2)));
    if (w1 < 1 || w2 < 1) raise(PyExc_ValueError, "window sizes must be at least 1");
    const int64_t dim = std::max(q.size(3), v1.size(3));
    if (pads ? dim > 256 || dim < 1 : !sa2_supported((int32_t)dim, 1, 1, SA2_BF16))
        raise(PyExc_NotImplementedError, "dim_head=" + std::to_string(dim) + " is not covered by the kernels (dim_head 32, 64, 128 or 256)");
    return geometry_of(q, k1, v1, std::min<int64_t>(w1, INT32_MAX), std::min<int64_t>(w2, INT32_MAX),
                       scale ? *scale : 1.0 / std::sqrt((double)q.size(3)));
}

Tensor checked_attend(const Tensor &q, const Tensor &k1, const Tensor &k2, const Tensor &v1, const Tensor &v2, int64_t w1, int64_t w2,
                      std::optional<double> scale, bool pads, const py::object &admit) {
    return attend(q, k1, k2, v1, v2, checked(q, k1, k2, v1, v2, w1, w2, scale, pads), admit);
}

// The two directions on their own, for the Python form of the node (a tracer records calls of Python Functions only).
using MaybeTensors = std::vector<std::optional<Tensor>>;
MaybeTensors maybe(const variable_list &all) {
    MaybeTensors out;
    for (const Tensor &t : all) out.push_back(t.defined() ? std::optional<Tensor>(t) : std::nullopt);
    return out;
}
variable_list defined(const MaybeTensors &all) {
    variable_list out;
    for (const auto &t : all) out.push_back(t.value_or(Tensor()));
    return out;
}

std::tuple<Tensor, MaybeTensors, std::vector<int64_t>, double> attend_forward(const Tensor &q, const Tensor &k1, const Tensor &k2, const Tensor &v1,
                                                                              const Tensor &v2, int64_t w1, int64_t w2, std::optional<double> scale,
                                                                              bool needs_grad, const py::object &admit) {
    const Geometry g = checked(q, k1, k2, v1, v2, w1, w2, scale, false);
    const Forward f = run_forward(q, k1, k2, v1, v2, g, needs_grad ? &admit : nullptr);
    return {f.result, maybe(Attend::saved_of(f)), Attend::sizes_of(g, {&q, &k1, &k2, &v1, &v2}), g.scale};
}

variable_list attend_backward(const MaybeTensors &saved, const std::vector<int64_t> &sizes, double scale, const Tensor &dout) {
    return Attend::run_backward(defined(saved), sizes, scale, dout);
}

// ---- fused split + per-head RMSNorm of the qkv projection
struct QKVNorm : public torch::autograd::Function<QKVNorm> {
    using Weight = std::optional<Tensor>;
    static variable_list forward(AutogradContext *ctx, const Tensor &qkv, const Weight &wq, const Weight &wk1, const Weight &wk2, const Weight &wv1,
                                 const Weight &wv2, int64_t heads, int64_t kv_heads, int64_t dim, double eps) {
        Saved saved;
        variable_list outs = run(&saved, qkv, {&wq, &wk1, &wk2, &wv1, &wv2}, heads, kv_heads, dim, eps);
        ctx->save_for_backward(saved.tensors);
        ctx->saved_data["geometry"] = c10::List<int64_t>(saved.sizes);
        return outs;
    }

    static variable_list backward(AutogradContext *ctx, variable_list douts) {
        variable_list grads = run_backward(ctx->get_saved_variables(), ctx->saved_data["geometry"].toIntVector(), douts);
        grads.resize(10);
        return grads;
    }

    struct Saved {
        variable_list tensors;
        std::vector<int64_t> sizes;
    };

    // (saved == nullptr: no backward follows)
    static variable_list run(Saved *saved, const Tensor &qkv_in, const std::array<const Weight *, 5> &w, int64_t heads, int64_t kv_heads,
                             int64_t dim, double eps) {
        const int64_t batch = qkv_in.size(0), seq = qkv_in.size(1);
        const Tensor qkv = qkv_in.stride(2) == 1 && qkv_in.stride(0) == seq * qkv_in.stride(1) ? qkv_in : qkv_in.contiguous();
        const c10::DeviceGuard guard(qkv.device());
        variable_list weights(5), outs(5);
        for (int x = 0; x < 5; ++x)
            if (w[x]->has_value()) weights[x] = (*w[x])->detach().to(at::kBFloat16).contiguous();
        for (int x = 0; x < 5; ++x) outs[x] = at::empty({batch, seq, x == 0 ? heads : kv_heads, dim}, qkv.options());
        const Tensor rstd = at::empty({batch * seq, heads + 4 * kv_heads}, qkv.options().dtype(at::kFloat));
        const sa2_problem prob = problem(batch, seq, heads, kv_heads, dim);
        sa2_tensor a[5];
        const void *p[5];
        for (int x = 0; x < 5; ++x) {
            a[x] = arg(outs[x]);
            p[x] = weights[x].defined() ? weights[x].data_ptr() : nullptr;
        }
        check(sa2_qkv_norm_fwd(&prob, qkv.data_ptr(), qkv.stride(1), p[0], p[1], p[2], p[3], p[4], (float)eps, &a[0], &a[1], &a[2], &a[3], &a[4],
                               static_cast<float *>(rstd.data_ptr()), stream_of(qkv)));
        if (saved) {
            saved->tensors = {qkv, rstd, weights[0], weights[1], weights[2], weights[3], weights[4]};
            saved->sizes = {batch, seq, heads, kv_heads, dim};
            for (int x = 0; x < 5; ++x) saved->sizes.push_back(w[x]->has_value() ? (int64_t)(*w[x])->scalar_type() : -1);
        }
        return outs;
    }

    static sa2_problem problem(int64_t batch, int64_t seq, int64_t heads, int64_t kv_heads, int64_t dim) {
        return {(int32_t)batch, (int32_t)seq, (int32_t)heads, (int32_t)kv_heads, (int32_t)dim, 1, 1, 1, 1.f, SA2_BF16};
    }

    static variable_list run_backward(const variable_list &s, const std::vector<int64_t> &n, variable_list douts) {
        const Tensor &qkv = s[0], &rstd = s[1];
        const int64_t batch = n[0], seq = n[1], heads = n[2], kv_heads = n[3], dim = n[4];
        const c10::DeviceGuard guard(qkv.device());
        const sa2_problem prob = problem(batch, seq, heads, kv_heads, dim);
        sa2_tensor a[5];
        const void *p[5];
        for (int x = 0; x < 5; ++x) {
            douts[x] = douts[x].defined() ? aligned(douts[x]) : at::zeros({batch, seq, x == 0 ? heads : kv_heads, dim}, qkv.options());
            a[x] = arg(douts[x]);
            p[x] = s[2 + x].defined() ? s[2 + x].data_ptr() : nullptr;
        }
        const Tensor dqkv = at::empty({batch, seq, qkv.size(2)}, qkv.options());
        const Tensor dw = at::empty({5, dim}, qkv.options().dtype(at::kFloat));
        const int64_t ws_bytes = sa2_qkv_norm_bwd_workspace_bytes(&prob);
        const Tensor ws = at::empty({ws_bytes}, qkv.options().dtype(at::kByte));
        check(sa2_qkv_norm_bwd(&prob, qkv.data_ptr(), qkv.stride(1), p[0], p[1], p[2], p[3], p[4], &a[0], &a[1], &a[2], &a[3], &a[4],
                               static_cast<float *>(rstd.data_ptr()), dqkv.data_ptr(), static_cast<float *>(dw.data_ptr()), ws.data_ptr(), ws_bytes,
                               stream_of(qkv)));
        variable_list result(6);
        result[0] = dqkv;
        // (one cast for weights of one type)
        Tensor cast = dw;
        for (int x = 0; x < 5; ++x) {
            if (n[5 + x] < 0) continue;
            const auto type = (at::ScalarType)n[5 + x];
            if (cast.scalar_type() != type) cast = dw.to(type);
            result[1 + x] = cast.select(0, x);
        }
        return result;
    }
};

variable_list qkv_norm(const Tensor &qkv, const QKVNorm::Weight &wq, const QKVNorm::Weight &wk1, const QKVNorm::Weight &wk2,
                       const QKVNorm::Weight &wv1, const QKVNorm::Weight &wv2, int64_t heads, int64_t kv_heads, int64_t dim, double eps) {
    bool seen = in_autograd({&qkv});
    const std::array<const QKVNorm::Weight *, 5> w{&wq, &wk1, &wk2, &wv1, &wv2};
    for (const auto *x : w) seen = seen || (x->has_value() && in_autograd({&**x}));
    if (!seen) return QKVNorm::run(nullptr, qkv, w, heads, kv_heads, dim, eps);
    return QKVNorm::apply(qkv, wq, wk1, wk2, wv1, wv2, heads, kv_heads, dim, eps);
}

// (for the Python form of the node, as attend_forward and attend_backward)
std::tuple<variable_list, MaybeTensors, std::vector<int64_t>> qkv_norm_forward(const Tensor &qkv, const QKVNorm::Weight &wq, const QKVNorm::Weight &wk1,
                                                                               const QKVNorm::Weight &wk2, const QKVNorm::Weight &wv1,
                                                                               const QKVNorm::Weight &wv2, int64_t heads, int64_t kv_heads, int64_t dim,
                                                                               double eps) {
    QKVNorm::Saved saved;
    variable_list outs = QKVNorm::run(&saved, qkv, {&wq, &wk1, &wk2, &wv1, &wv2}, heads, kv_heads, dim, eps);
    return {outs, maybe(saved.tensors), saved.sizes};
}

MaybeTensors qkv_norm_backward(const MaybeTensors &saved, const std::vector<int64_t> &sizes, const variable_list &douts) {
    return maybe(QKVNorm::run_backward(defined(saved), sizes, douts));
}

// batched tensors (vmap's and is_grads_batched's), functorch's wrappers, subclasses with a dispatch of their own and
// forward-mode tangents: a kernel launched on their data pointers would miss what they carry
bool foreign(const Tensor &t) {
    static const c10::DispatchKeySet keys({c10::DispatchKey::Batched, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                           c10::DispatchKey::Python, c10::DispatchKey::Functionalize});
    return t.key_set().has_any(keys) || t._fw_grad(0).defined();
}

// ---- linear layer whose weight gradient is this library's kernel (the products with the weight stay torch's)
struct Linear : public torch::autograd::Function<Linear> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x, const Tensor &w, const std::optional<Tensor> &bias) {
        // (the weight is for the gradient of x alone: without one it may be changed in place before the backward)
        ctx->save_for_backward({x, x.requires_grad() ? w : Tensor()});
        ctx->saved_data["bias"] = bias.has_value();
        return at::linear(x, w, bias);
    }

    static variable_list backward(AutogradContext *ctx, variable_list douts) {
        const variable_list s = ctx->get_saved_variables();
        const Tensor &x = s[0], &w = s[1], &dy = douts[0];
        const Tensor dy2 = dy.reshape({-1, dy.size(-1)}), x2 = x.reshape({-1, x.size(-1)});
        variable_list grads(3);
        if (ctx->needs_input_grad(0)) grads[0] = dy2.mm(w).view_as(x);
        // (a graph of the backward and batched gradients need torch's product)
        if (ctx->needs_input_grad(1)) grads[1] = at::GradMode::is_enabled() || foreign(dy) || foreign(x) ? dy2.t().mm(x2) : weight_gradient(dy2, x2);
        if (ctx->saved_data["bias"].toBool() && ctx->needs_input_grad(2)) grads[2] = dy2.sum(0);
        return grads;
    }

    static Tensor weight_gradient(const Tensor &dy, const Tensor &x) {
        const c10::DeviceGuard guard(x.device());
        auto rows = [](const Tensor &t) {
            const bool ok = t.stride(1) == 1 && t.stride(0) >= t.size(1) && t.stride(0) % 8 == 0 && reinterpret_cast<uintptr_t>(t.data_ptr()) % 16 == 0;
            return ok ? t : t.clone(at::MemoryFormat::Contiguous);
        };
        const Tensor a = rows(dy), b = rows(x), dw = at::empty({dy.size(1), x.size(1)}, x.options());
        const int64_t ws_bytes = sa2_wgrad_workspace_bytes(x.size(0), (int32_t)dy.size(1), (int32_t)x.size(1));
        const Tensor ws = at::empty({ws_bytes}, x.options().dtype(at::kByte));
        check(sa2_wgrad(a.data_ptr(), a.stride(0), b.data_ptr(), b.stride(0), x.size(0), (int32_t)dy.size(1), (int32_t)x.size(1), dw.data_ptr(), ws.data_ptr(),
                        ws_bytes, stream_of(x)));
        return dw;
    }
};

Tensor linear(const Tensor &x, const Tensor &w, const std::optional<Tensor> &bias) {
    bool plain = !at::GradMode::is_enabled() || !w.requires_grad();
    for (const Tensor *t : {&x, &w, bias ? &*bias : &w}) plain = plain || foreign(*t);
    return plain ? at::linear(x, w, bias) : Linear::apply(x, w, bias);
}

}  // namespace

PYBIND11_MODULE(_sa2_torch, m) {
    m.def("attend", &checked_attend);
    m.def("attend_forward", &attend_forward);
    m.def("attend_backward", &attend_backward);
    m.def("qkv_norm", &qkv_norm);
    m.def("qkv_norm_forward", &qkv_norm_forward);
    m.def("qkv_norm_backward", &qkv_norm_backward);
    m.def("linear", &linear);
    m.def("released_bytes", [](int device) { return device >= 0 && device < kMostDevices ? g_released[device].load() : int64_t(0); });
}
