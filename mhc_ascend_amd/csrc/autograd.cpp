// Autograd nodes of the fused mHC layers in C++ over the C ABI of
// libmhc_hip (the role of the reference's Python autograd functions,
// src/python/mhc/ops.py:387-564, and of its pybind11 layer entries,
// src/python/bindings.cpp:600-952).  Forward and backward prepare their
// arguments exactly as mhc_ascend_amd/native.py does (same checks, dtypes,
// workspaces and error text) and call the same entry points, so results are
// identical bit for bit; doing it in C++ keeps the interpreter out of the
// forward and the autograd engine's hand-off to a Python backward out of
// every step.
//
// The fused MHCResidualWrapper (layer.py:269-322) has nodes of the same kind.
// These nodes are the package's only orchestration of the fused entries;
// tests/pyref_autograd.py restates them in Python for a bit-for-bit check.
//
// The entry points are not linked: bind() receives their addresses from the
// ctypes handle of the already loaded library, so both paths share one copy
// of it (one error state, one set of per-device caches) whichever build of
// it was loaded.
#include <torch/extension.h>

#include <ATen/hip/HIPContext.h>

#include <algorithm>
#include <map>
#include <string>
#include <vector>

#include "mhc_hip.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::tensor_list;

#define MHC_AUTOGRAD_ENTRIES(X)               \
    X(mhc_last_error)                         \
    X(mhc_layer_static_saved_size)            \
    X(mhc_layer_static_fwd)                   \
    X(mhc_layer_static_bwd_workspace_size)    \
    X(mhc_layer_static_bwd)                   \
    X(mhc_layer_dynamic_saved_size)           \
    X(mhc_layer_dynamic_fwd_workspace_size)   \
    X(mhc_layer_dynamic_fwd)                  \
    X(mhc_layer_dynamic_bwd_workspace_size)   \
    X(mhc_layer_dynamic_bwd)                  \
    X(mhc_layer_dynamic_packed_size)          \
    X(mhc_layer_dynamic_infer_workspace_size) \
    X(mhc_layer_dynamic_infer)                \
    X(mhc_sinkhorn_knopp_fwd)                 \
    X(mhc_sinkhorn_knopp_bwd)                 \
    X(mhc_rmsnorm_fwd)                        \
    X(mhc_rmsnorm_bwd_workspace_size)         \
    X(mhc_rmsnorm_bwd)                        \
    X(mhc_stream_aggregate_fwd)               \
    X(mhc_stream_aggregate_bwd)               \
    X(mhc_stream_distribute_mix_add_fwd)      \
    X(mhc_stream_distribute_mix_add_bwd)      \
    X(mhc_wrapper_dynamic_saved_size)         \
    X(mhc_wrapper_dynamic_fwd_workspace_need) \
    X(mhc_wrapper_dynamic_fwd)                \
    X(mhc_wrapper_dynamic_bwd_workspace_need) \
    X(mhc_wrapper_dynamic_bwd)                \
    X(mhc_wrapper_static_fwd)                 \
    X(mhc_wrapper_static_bwd_workspace_size)  \
    X(mhc_wrapper_static_bwd)

struct Entries {
#define MHC_DECLARE(name) decltype(&::name) name = nullptr;
    MHC_AUTOGRAD_ENTRIES(MHC_DECLARE)
#undef MHC_DECLARE
};

Entries lib;
bool bound = false;

void bind(const std::map<std::string, int64_t>& addrs) {
    Entries e;
#define MHC_BIND(name)                                                                            \
    {                                                                                             \
        auto it = addrs.find(#name);                                                              \
        TORCH_CHECK(it != addrs.end() && it->second != 0, "mhc autograd: no address for " #name); \
        e.name = reinterpret_cast<decltype(e.name)>(static_cast<intptr_t>(it->second));           \
    }
    MHC_AUTOGRAD_ENTRIES(MHC_BIND)
#undef MHC_BIND
    lib = e;
    bound = true;
}

std::vector<std::string> entry_names() {
    return {
#define MHC_NAME(name) #name,
        MHC_AUTOGRAD_ENTRIES(MHC_NAME)
#undef MHC_NAME
    };
}

void require_bound() { TORCH_CHECK(bound, "mhc autograd: bind() the HIP library's entry points first"); }

int dtype_code(at::ScalarType t) {
    if (t == at::kFloat) return MHC_DTYPE_F32;
    if (t == at::kBFloat16) return MHC_DTYPE_BF16;
    TORCH_CHECK(false, "mhc_ascend_amd: unsupported storage dtype ", t, " (float32 or bfloat16)");
    return -1;
}

void check(int rc, const char* name) {
    TORCH_CHECK(rc == 0, name, " failed (status ", rc, "): ", lib.mhc_last_error());
}

void check_device(const char* fn, std::initializer_list<const Tensor*> ts) {
    c10::optional<c10::Device> dev;
    for (const Tensor* t : ts) {
        TORCH_CHECK(t->is_cuda(), fn, ": tensors must be on a HIP device (got ", t->device(),
                    "); mhc_ascend_amd has no CPU path");
        if (!dev) {
            dev = t->device();
        } else {
            TORCH_CHECK(t->device() == *dev, fn, ": all tensors must be on the same device (", *dev, " vs ",
                        t->device(), ")");
        }
    }
}

bool storage_dtype(at::ScalarType t) { return t == at::kFloat || t == at::kBFloat16; }

Tensor layer_x(const char* fn, const Tensor& x) {
    TORCH_CHECK(x.dim() == 3, fn, ": x must be 3D [B, n, C]");
    return (storage_dtype(x.scalar_type()) ? x : x.to(at::kFloat)).contiguous();
}

Tensor weight(const Tensor& w) { return (storage_dtype(w.scalar_type()) ? w : w.to(at::kFloat)).contiguous(); }

Tensor f32c(const Tensor& t) {
    if (t.scalar_type() == at::kFloat && t.is_contiguous()) return t;
    return t.to(at::kFloat).contiguous();
}

// alpha as a one-element fp32 device tensor of its own shape (a device
// pointer: no host sync)
Tensor scalar_param(const Tensor& a, c10::Device dev) {
    TORCH_CHECK(a.numel() == 1, "alpha must have one element, got shape ", a.sizes());
    if (a.device() == dev) return f32c(a);
    return a.detach().to(dev, at::kFloat).contiguous();
}

// A contiguous tensor of `sizes` over part of a contiguous buffer, from
// element `offset` on.
Tensor part_of(const Tensor& buf, at::IntArrayRef sizes, int64_t offset) {
    c10::SmallVector<int64_t, 4> strides(sizes.size());
    int64_t st = 1;
    for (size_t i = sizes.size(); i-- > 0;) {
        strides[i] = st;
        st *= sizes[i] > 0 ? sizes[i] : 1;
    }
    return buf.as_strided(sizes, strides, offset);
}

// Appends the gradients of (phi_pre, phi_post, phi_res, alpha_pre, alpha_post,
// alpha_res, b_pre, b_post, b_res), in the parameters' shapes, over the
// entry's three gradient buffers.
void push_param_grads(tensor_list& out, const at::IntArrayRef (&shapes)[9], int64_t n, const Tensor& gphi,
                      const Tensor& galpha, const Tensor& gb) {
    const Tensor* bufs[3] = {&gphi, &galpha, &gb};
    const int64_t nC = gphi.size(1);
    const int64_t want[3][3] = {{n * nC, n * nC, n * n * nC}, {1, 1, 1}, {n, n, n * n}};
    for (int k = 0; k < 3; ++k) {
        int64_t off = 0;
        for (int i = 0; i < 3; ++i) {
            const at::IntArrayRef shape = shapes[3 * k + i];
            TORCH_CHECK(c10::multiply_integers(shape) == want[k][i], "dynamic layer: parameter of shape ", shape,
                        " does not match n = ", n);
            out.push_back(part_of(*bufs[k], shape, off));
            off += want[k][i];
        }
    }
}

Tensor workspace(size_t nbytes, const Tensor& like) {
    return at::empty({(int64_t)std::max<size_t>(nbytes, 1)}, like.options().dtype(at::kByte));
}

void* stream() { return at::hip::getCurrentHIPStream().stream(); }

float* fp(const Tensor& t) { return t.data_ptr<float>(); }

// ---- static H: mhc_ascend_amd.ops.MHCLayerStaticFunction (layer.py:142-170) --
struct StaticLayer : public torch::autograd::Function<StaticLayer> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w_in, const Tensor& hp_in,
                          const Tensor& hq_in, const Tensor& hr_in, int64_t iters, double sk_eps, double rms_eps) {
        const char* fn = "mhc_layer_static_fwd";
        check_device(fn, {&x_in, &w_in, &hp_in, &hq_in, &hr_in});
        const at::DeviceGuard guard(x_in.device());
        const Tensor x = layer_x(fn, x_in);
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
        TORCH_CHECK(w_in.numel() == C && hp_in.numel() == n && hq_in.numel() == n && hr_in.numel() == n * n,
                    "mhc_layer_static_fwd: parameter shapes do not match x [B, n, C]");
        const Tensor w = weight(w_in), hp = f32c(hp_in), hq = f32c(hq_in), hr = f32c(hr_in);
        const auto f32 = x.options().dtype(at::kFloat);
        Tensor out = at::empty({B, n, C}, f32);
        Tensor rms = at::empty({B}, f32);
        Tensor saved = at::empty({(int64_t)(lib.mhc_layer_static_saved_size((int32_t)n, (int32_t)C) / 4)}, f32);
        check(lib.mhc_layer_static_fwd(x.data_ptr(), dtype_code(x.scalar_type()), w.data_ptr(),
                                       dtype_code(w.scalar_type()), fp(hp), fp(hq), fp(hr), fp(out), fp(rms),
                                       fp(saved), B, (int32_t)n, (int32_t)C, (int32_t)iters, (float)sk_eps,
                                       (float)rms_eps, stream()),
              fn);
        ctx->save_for_backward({x, w, hp, hq, hr, saved});
        ctx->saved_data["x_dtype"] = (int64_t)x_in.scalar_type();
        ctx->saved_data["cfg"] = std::vector<double>{(double)iters, sk_eps, rms_eps};
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const char* fn = "mhc_layer_static_bwd";
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &w = sv[1], &hp = sv[2], &hq = sv[3], &hr = sv[4], &saved = sv[5];
        check_device(fn, {&grads[0], &x});
        const at::DeviceGuard guard(x.device());
        const auto cfg = ctx->saved_data["cfg"].toDoubleVector();
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
        TORCH_CHECK(grads[0].sizes() == x.sizes(), "mhc_layer_static_bwd: grad_out must match x [B, n, C]");
        const Tensor g = f32c(grads[0]);
        const auto f32 = x.options().dtype(at::kFloat);
        Tensor grad_x = at::empty_like(x);
        Tensor gw = at::empty({C}, w.options());
        Tensor ghp = at::empty(hp.sizes(), f32), ghq = at::empty(hq.sizes(), f32), ghr = at::empty(hr.sizes(), f32);
        const int xd = dtype_code(x.scalar_type());
        const size_t wsb = lib.mhc_layer_static_bwd_workspace_size(B, (int32_t)n, (int32_t)C, xd);
        Tensor ws = workspace(wsb, x);
        check(lib.mhc_layer_static_bwd(fp(g), x.data_ptr(), xd, dtype_code(w.scalar_type()), fp(hp), fp(hq), fp(hr),
                                       fp(saved), grad_x.data_ptr(), gw.data_ptr(), fp(ghp), fp(ghq), fp(ghr),
                                       ws.data_ptr(), wsb, B, (int32_t)n, (int32_t)C, (int32_t)cfg[0],
                                       (float)cfg[1], (float)cfg[2], stream()),
              fn);
        const auto x_dtype = (at::ScalarType)ctx->saved_data["x_dtype"].toInt();
        return {grad_x.to(x_dtype), gw, ghp, ghq, ghr, Tensor(), Tensor(), Tensor()};
    }
};

// ---- dynamic H: mhc_ascend_amd.ops.MHCLayerDynamicFunction (ops.py:387-564) --
std::vector<Tensor> phi_parts(const Tensor& pre, const Tensor& post, const Tensor& res, int64_t n, int64_t nC) {
    std::vector<Tensor> parts = {f32c(pre), f32c(post), f32c(res)};
    const int64_t rows[3] = {n, n, n * n};
    for (int i = 0; i < 3; ++i) {
        TORCH_CHECK(parts[i].numel() == rows[i] * nC, "dynamic layer: projection of ", parts[i].sizes(),
                    " does not match [", rows[i], ", ", nC, "]");
    }
    return parts;
}

struct DynamicLayer : public torch::autograd::Function<DynamicLayer> {
    static Tensor forward(AutogradContext* ctx, const Tensor& x_in, const Tensor& w_in, const Tensor& pp_in,
                          const Tensor& pq_in, const Tensor& pr_in, const Tensor& ap_in, const Tensor& aq_in,
                          const Tensor& ar_in, const Tensor& bp_in, const Tensor& bq_in, const Tensor& br_in,
                          int64_t iters, double sk_eps, double rms_eps) {
        const char* fn = "mhc_layer_dynamic_fwd";
        check_device(fn, {&x_in, &w_in, &pp_in, &pq_in, &pr_in, &bp_in, &bq_in, &br_in});
        const at::DeviceGuard guard(x_in.device());
        const Tensor x = layer_x(fn, x_in);
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
        const Tensor w = weight(w_in);
        TORCH_CHECK(w.numel() == C, "mhc_layer_dynamic_fwd: rmsnorm_weight must have C elements");
        const auto ph = phi_parts(pp_in, pq_in, pr_in, n, n * C);
        const Tensor ap = scalar_param(ap_in, x.device()), aq = scalar_param(aq_in, x.device()),
                     ar = scalar_param(ar_in, x.device());
        const Tensor bp = f32c(bp_in), bq = f32c(bq_in), br = f32c(br_in);
        const auto f32 = x.options().dtype(at::kFloat);
        Tensor out = at::empty({B, n, C}, f32);
        Tensor saved = at::empty({(int64_t)(lib.mhc_layer_dynamic_saved_size(B, (int32_t)n, (int32_t)C) / 4)}, f32);
        const size_t wsb = lib.mhc_layer_dynamic_fwd_workspace_size(B, (int32_t)n, (int32_t)C);
        Tensor ws = workspace(wsb, x);
        check(lib.mhc_layer_dynamic_fwd(x.data_ptr(), dtype_code(x.scalar_type()), w.data_ptr(),
                                        dtype_code(w.scalar_type()), fp(ph[0]), fp(ph[1]), fp(ph[2]), fp(ap), fp(aq),
                                        fp(ar), fp(bp), fp(bq), fp(br), fp(out), fp(saved), ws.data_ptr(), wsb, B,
                                        (int32_t)n, (int32_t)C, (int32_t)iters, (float)sk_eps, (float)rms_eps,
                                        stream()),
              fn);
        ctx->save_for_backward({x, w, saved, ph[0], ph[1], ph[2], ap, aq, ar, bp, bq, br});
        ctx->saved_data["x_dtype"] = (int64_t)x_in.scalar_type();
        ctx->saved_data["cfg"] = std::vector<double>{(double)iters, sk_eps, rms_eps};
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const char* fn = "mhc_layer_dynamic_bwd";
        const auto sv = ctx->get_saved_variables();
        const Tensor &x = sv[0], &w = sv[1], &saved = sv[2];
        check_device(fn, {&grads[0], &x});
        const at::DeviceGuard guard(x.device());
        const auto cfg = ctx->saved_data["cfg"].toDoubleVector();
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2), np = 2 * n + n * n;
        TORCH_CHECK(grads[0].sizes() == x.sizes(), "mhc_layer_dynamic_bwd: grad_output must match x [B, n, C]");
        const Tensor g = f32c(grads[0]);
        const auto f32 = x.options().dtype(at::kFloat);
        Tensor grad_x = at::empty_like(x);
        Tensor gw = at::empty({C}, w.options());
        Tensor gphi = at::empty({np, n * C}, f32);
        Tensor galpha = at::empty({3}, f32);
        Tensor gb = at::empty({np}, f32);
        const int xd = dtype_code(x.scalar_type());
        const size_t wsb = lib.mhc_layer_dynamic_bwd_workspace_size(B, (int32_t)n, (int32_t)C, xd);
        Tensor ws = workspace(wsb, x);
        check(lib.mhc_layer_dynamic_bwd(fp(g), x.data_ptr(), xd, dtype_code(w.scalar_type()), fp(sv[3]), fp(sv[4]),
                                        fp(sv[5]), fp(sv[6]), fp(sv[7]), fp(sv[8]), fp(sv[9]), fp(sv[10]),
                                        fp(sv[11]), fp(saved), grad_x.data_ptr(), gw.data_ptr(), fp(gphi),
                                        fp(galpha), fp(gb), ws.data_ptr(), wsb, B, (int32_t)n, (int32_t)C,
                                        (int32_t)cfg[0], (float)cfg[1], (float)cfg[2], stream()),
              fn);
        const auto x_dtype = (at::ScalarType)ctx->saved_data["x_dtype"].toInt();
        tensor_list out;
        out.reserve(14);
        out.push_back(grad_x.to(x_dtype));
        out.push_back(gw);
        push_param_grads(out,
                         {sv[3].sizes(), sv[4].sizes(), sv[5].sizes(), sv[6].sizes(), sv[7].sizes(), sv[8].sizes(),
                          sv[9].sizes(), sv[10].sizes(), sv[11].sizes()},
                         n, gphi, galpha, gb);
        out.resize(14);
        return out;
    }
};

// ---- fused MHCResidualWrapper (layer.py:269-322) ----------------------------
// residual / branch [tokens, hidden] as the kernels read them: residual in
// fp32 or bf16 (others become fp32), branch in the residual's dtype.
std::pair<Tensor, Tensor> wrapper_inputs(const char* fn, const Tensor& residual, const Tensor& branch) {
    check_device(fn, {&residual, &branch});
    TORCH_CHECK(residual.sizes() == branch.sizes() && residual.dim() == 2, fn,
                ": residual and branch must both be [tokens, hidden] of one shape");
    Tensor r = (storage_dtype(residual.scalar_type()) ? residual : residual.to(at::kFloat)).contiguous();
    return {r, branch.to(r.scalar_type()).contiguous()};
}

int32_t wrapper_mode(const std::string& mode, int64_t n, const char* fn) {
    TORCH_CHECK_VALUE(mode == "decay" || mode == "zero", "Unknown residual_mode: ", mode);
    // the reference writes stream 1 (layer.py:301), which needs n >= 2
    TORCH_CHECK(n >= 2, fn, ": expansion_rate must be >= 2 (stream 1 holds the branch)");
    return mode == "decay" ? MHC_WRAPPER_DECAY : MHC_WRAPPER_ZERO;
}

struct StaticWrapper : public torch::autograd::Function<StaticWrapper> {
    static Tensor forward(AutogradContext* ctx, const Tensor& res_in, const Tensor& br_in, const Tensor& w_in,
                          const Tensor& hp_in, const Tensor& hq_in, const Tensor& hr_in, int64_t mode, int64_t n,
                          int64_t iters, double sk_eps, double rms_eps) {
        const char* fn = "wrapper_static_fwd";
        auto [r, b] = wrapper_inputs(fn, res_in, br_in);
        check_device(fn, {&r, &w_in, &hp_in, &hq_in, &hr_in});
        const at::DeviceGuard guard(r.device());
        const int64_t T = r.size(0), C = r.size(1);
        const Tensor w = weight(w_in);
        TORCH_CHECK(w.numel() == C && hp_in.numel() == n && hq_in.numel() == n && hr_in.numel() == n * n,
                    "wrapper_static_fwd: parameter shapes do not match n and C");
        const Tensor hp = f32c(hp_in), hq = f32c(hq_in), hr = f32c(hr_in);
        const auto f32 = r.options().dtype(at::kFloat);
        Tensor out = at::empty({T, C}, f32);
        Tensor saved = at::empty({(int64_t)(lib.mhc_layer_static_saved_size((int32_t)n, (int32_t)C) / 4)}, f32);
        check(lib.mhc_wrapper_static_fwd(r.data_ptr(), b.data_ptr(), dtype_code(r.scalar_type()), (int32_t)mode,
                                         w.data_ptr(), dtype_code(w.scalar_type()), fp(hp), fp(hq), fp(hr), fp(out),
                                         fp(saved), T, (int32_t)n, (int32_t)C, (int32_t)iters, (float)sk_eps,
                                         (float)rms_eps, stream()),
              "mhc_wrapper_static_fwd");
        ctx->save_for_backward({r, b, w, hp, hq, hr, saved});
        ctx->saved_data["dtypes"] = std::vector<int64_t>{(int64_t)res_in.scalar_type(), (int64_t)br_in.scalar_type()};
        ctx->saved_data["cfg"] = std::vector<double>{(double)mode, (double)n, (double)iters, sk_eps, rms_eps};
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const char* fn = "wrapper_static_bwd";
        const auto sv = ctx->get_saved_variables();
        const Tensor &r = sv[0], &b = sv[1], &w = sv[2], &saved = sv[6];
        check_device(fn, {&grads[0], &r});
        const at::DeviceGuard guard(r.device());
        const auto cfg = ctx->saved_data["cfg"].toDoubleVector();
        const int64_t T = r.size(0), C = r.size(1), n = (int64_t)cfg[1];
        const int32_t mode = (int32_t)cfg[0];
        TORCH_CHECK(grads[0].sizes() == r.sizes(), "wrapper_static_bwd: grad_out must be [tokens, hidden]");
        const Tensor g = f32c(grads[0]);
        const auto f32 = r.options().dtype(at::kFloat);
        Tensor gr = at::empty_like(r), gb = at::empty_like(b);
        Tensor gw = at::empty({C}, w.options());
        Tensor ghp = at::empty(sv[3].sizes(), f32), ghq = at::empty(sv[4].sizes(), f32),
               ghr = at::empty(sv[5].sizes(), f32);
        const int dt = dtype_code(r.scalar_type());
        const size_t wsb = lib.mhc_wrapper_static_bwd_workspace_size(T, (int32_t)n, (int32_t)C, dt, mode);
        Tensor ws = workspace(wsb, r);
        check(lib.mhc_wrapper_static_bwd(fp(g), r.data_ptr(), b.data_ptr(), dt, mode, dtype_code(w.scalar_type()),
                                         fp(sv[3]), fp(sv[4]), fp(sv[5]), fp(saved), gr.data_ptr(), gb.data_ptr(),
                                         gw.data_ptr(), fp(ghp), fp(ghq), fp(ghr), ws.data_ptr(), wsb, T, (int32_t)n,
                                         (int32_t)C, (int32_t)cfg[2], (float)cfg[3], (float)cfg[4], stream()),
              "mhc_wrapper_static_bwd");
        const auto dts = ctx->saved_data["dtypes"].toIntVector();
        return {gr.to((at::ScalarType)dts[0]), gb.to((at::ScalarType)dts[1]), gw, ghp, ghq, ghr, Tensor(), Tensor(),
                Tensor(), Tensor(), Tensor()};
    }
};

struct DynamicWrapper : public torch::autograd::Function<DynamicWrapper> {
    static Tensor forward(AutogradContext* ctx, const Tensor& res_in, const Tensor& br_in, const Tensor& w_in,
                          const Tensor& pp_in, const Tensor& pq_in, const Tensor& pr_in, const Tensor& ap_in,
                          const Tensor& aq_in, const Tensor& ar_in, const Tensor& bp_in, const Tensor& bq_in,
                          const Tensor& bres_in, int64_t mode, int64_t n, int64_t iters, double sk_eps,
                          double rms_eps) {
        const char* fn = "wrapper_dynamic_fwd";
        auto [r, b] = wrapper_inputs(fn, res_in, br_in);
        check_device(fn, {&r, &w_in, &pp_in, &pq_in, &pr_in, &bp_in, &bq_in, &bres_in});
        const at::DeviceGuard guard(r.device());
        const int64_t T = r.size(0), C = r.size(1);
        const Tensor w = weight(w_in);
        TORCH_CHECK(w.numel() == C, "wrapper_dynamic_fwd: rmsnorm_weight must have C elements");
        const auto ph = phi_parts(pp_in, pq_in, pr_in, n, n * C);
        const Tensor ap = scalar_param(ap_in, r.device()), aq = scalar_param(aq_in, r.device()),
                     ar = scalar_param(ar_in, r.device());
        const Tensor bp = f32c(bp_in), bq = f32c(bq_in), bres = f32c(bres_in);
        const auto f32 = r.options().dtype(at::kFloat);
        Tensor out = at::empty({T, C}, f32);
        Tensor saved =
            at::empty({(int64_t)(lib.mhc_wrapper_dynamic_saved_size(T, (int32_t)n, (int32_t)C) / 4)}, f32);
        const size_t wsb = lib.mhc_wrapper_dynamic_fwd_workspace_need(
            r.data_ptr(), b.data_ptr(), dtype_code(r.scalar_type()), T, (int32_t)n, (int32_t)C);
        Tensor ws = workspace(wsb, r);
        check(lib.mhc_wrapper_dynamic_fwd(r.data_ptr(), b.data_ptr(), dtype_code(r.scalar_type()), (int32_t)mode,
                                          w.data_ptr(), dtype_code(w.scalar_type()), fp(ph[0]), fp(ph[1]), fp(ph[2]),
                                          fp(ap), fp(aq), fp(ar), fp(bp), fp(bq), fp(bres), fp(out), fp(saved),
                                          ws.data_ptr(), wsb, T, (int32_t)n, (int32_t)C, (int32_t)iters,
                                          (float)sk_eps, (float)rms_eps, stream()),
              "mhc_wrapper_dynamic_fwd");
        ctx->save_for_backward({r, b, w, saved, ph[0], ph[1], ph[2], ap, aq, ar, bres});
        // b_pre and b_post are not read by the backward: their shapes only
        ctx->saved_data["b_pre"] = bp.sizes().vec();
        ctx->saved_data["b_post"] = bq.sizes().vec();
        ctx->saved_data["dtypes"] = std::vector<int64_t>{(int64_t)res_in.scalar_type(), (int64_t)br_in.scalar_type()};
        ctx->saved_data["cfg"] = std::vector<double>{(double)mode, (double)n, (double)iters, sk_eps, rms_eps};
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const char* fn = "wrapper_dynamic_bwd";
        const auto sv = ctx->get_saved_variables();
        const Tensor &r = sv[0], &b = sv[1], &w = sv[2], &saved = sv[3];
        check_device(fn, {&grads[0], &r});
        const at::DeviceGuard guard(r.device());
        const auto cfg = ctx->saved_data["cfg"].toDoubleVector();
        const int64_t T = r.size(0), C = r.size(1), n = (int64_t)cfg[1], np = 2 * n + n * n;
        const int32_t mode = (int32_t)cfg[0];
        TORCH_CHECK(grads[0].sizes() == r.sizes(), "wrapper_dynamic_bwd: grad_out must be [tokens, hidden]");
        const Tensor g = f32c(grads[0]);
        const auto f32 = r.options().dtype(at::kFloat);
        Tensor gr = at::empty_like(r), gb = at::empty_like(b);
        Tensor gw = at::empty({C}, w.options());
        Tensor gphi = at::empty({np, n * C}, f32);
        Tensor galpha = at::empty({3}, f32);
        Tensor gbias = at::empty({np}, f32);
        const int dt = dtype_code(r.scalar_type());
        const size_t wsb = lib.mhc_wrapper_dynamic_bwd_workspace_need(
            fp(g), r.data_ptr(), b.data_ptr(), gr.data_ptr(), gb.data_ptr(), dt, mode, T, (int32_t)n, (int32_t)C,
            (int32_t)cfg[2], (float)cfg[3]);
        Tensor ws = workspace(wsb, r);
        check(lib.mhc_wrapper_dynamic_bwd(fp(g), r.data_ptr(), b.data_ptr(), dt, mode, dtype_code(w.scalar_type()),
                                          fp(sv[4]), fp(sv[5]), fp(sv[6]), fp(sv[7]), fp(sv[8]), fp(sv[9]),
                                          fp(sv[10]), fp(saved), gr.data_ptr(), gb.data_ptr(), gw.data_ptr(),
                                          fp(gphi), fp(galpha), fp(gbias), ws.data_ptr(), wsb, T, (int32_t)n,
                                          (int32_t)C, (int32_t)cfg[2], (float)cfg[3], (float)cfg[4], stream()),
              "mhc_wrapper_dynamic_bwd");
        const auto dts = ctx->saved_data["dtypes"].toIntVector();
        tensor_list out;
        out.reserve(17);
        out.push_back(gr.to((at::ScalarType)dts[0]));
        out.push_back(gb.to((at::ScalarType)dts[1]));
        out.push_back(gw);
        const auto bp = ctx->saved_data["b_pre"].toIntVector(), bq = ctx->saved_data["b_post"].toIntVector();
        push_param_grads(out,
                         {sv[4].sizes(), sv[5].sizes(), sv[6].sizes(), sv[7].sizes(), sv[8].sizes(), sv[9].sizes(), bp,
                          bq, sv[10].sizes()},
                         n, gphi, galpha, gbias);
        out.resize(17);
        return out;
    }
};

// ---- forward-only dynamic layer (ops.py:337-380) ------------------------------
Tensor dynamic_infer(const Tensor& x_in, const Tensor& packed, const Tensor& ap_in, const Tensor& aq_in,
                     const Tensor& ar_in, const Tensor& bp_in, const Tensor& bq_in, const Tensor& br_in, int64_t iters,
                     double sk_eps, double rms_eps, bool out_bf16) {
    require_bound();
    const char* fn = "mhc_layer_dynamic_infer";
    const at::NoGradGuard no_grad;
    check_device(fn, {&x_in, &packed, &bp_in, &bq_in, &br_in});
    const at::DeviceGuard guard(x_in.device());
    const Tensor x = layer_x(fn, x_in);
    const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
    TORCH_CHECK(packed.scalar_type() == at::kByte &&
                    (size_t)packed.numel() >= lib.mhc_layer_dynamic_packed_size((int32_t)n, (int32_t)C),
                fn, ": packed parameters do not match x [B, n, C]");
    const Tensor ap = scalar_param(ap_in, x.device()), aq = scalar_param(aq_in, x.device()),
                 ar = scalar_param(ar_in, x.device());
    const Tensor bp = f32c(bp_in), bq = f32c(bq_in), br = f32c(br_in);
    TORCH_CHECK(bp.numel() == n && bq.numel() == n && br.numel() == n * n, fn,
                ": b_pre/b_post must have n and b_res n*n elements");
    Tensor out = at::empty({B, n, C}, x.options().dtype(out_bf16 ? at::kBFloat16 : at::kFloat));
    const size_t wsb = lib.mhc_layer_dynamic_infer_workspace_size(B, (int32_t)n, (int32_t)C);
    Tensor ws = workspace(wsb, x);
    check(lib.mhc_layer_dynamic_infer(x.data_ptr(), dtype_code(x.scalar_type()), packed.data_ptr(), fp(ap), fp(aq),
                                      fp(ar), fp(bp), fp(bq), fp(br), out.data_ptr(),
                                      out_bf16 ? MHC_DTYPE_BF16 : MHC_DTYPE_F32, ws.data_ptr(), wsb, B, (int32_t)n,
                                      (int32_t)C, (int32_t)iters, (float)sk_eps, (float)rms_eps, stream()),
          fn);
    return out;
}

// ---- standalone operators (ops.py:32-265) -------------------------------------
// The same checks, dtypes and error text as the functions of
// mhc_ascend_amd/native.py; the tensors saved are the caller's own.
Tensor storage(const Tensor& t) { return (storage_dtype(t.scalar_type()) ? t : t.to(at::kFloat)).contiguous(); }

// A per-token coefficient tensor as (fp32 tensor, batch stride): one that is
// broadcast over the batch (stride 0) is passed once.
std::pair<Tensor, int64_t> coef_view(const char* fn, const Tensor& t_in, int64_t B, int64_t per) {
    const Tensor t = t_in.to(at::kFloat);
    if (t.dim() >= 2 && t.size(0) == B && t.stride(0) == 0) {
        const Tensor one = t.select(0, 0).contiguous();
        TORCH_CHECK(one.numel() == per, fn, ": coefficient shape ", t.sizes(), " does not match n");
        return {one, 0};
    }
    const Tensor c = t.contiguous();
    TORCH_CHECK(c.numel() == B * per, fn, ": coefficient shape ", t.sizes(), " does not match [B=", B, ", ", per, "]");
    return {c, per};
}

struct Sinkhorn : public torch::autograd::Function<Sinkhorn> {
    static Tensor forward(AutogradContext* ctx, const Tensor& inp, int64_t iters, double eps) {
        check_device("sinkhorn_knopp_fwd", {&inp});
        const at::DeviceGuard guard(inp.device());
        TORCH_CHECK(inp.dim() == 3, "Input must be 3D tensor [B, M, N]");
        TORCH_CHECK(inp.size(1) == inp.size(2), "Sinkhorn-Knopp requires square matrices (M == N), got M=",
                    inp.size(1), ", N=", inp.size(2));
        TORCH_CHECK(inp.scalar_type() == at::kFloat, "inp must be float32");
        const Tensor a = inp.contiguous();
        Tensor out = at::empty_like(a);
        check(lib.mhc_sinkhorn_knopp_fwd(fp(a), fp(out), a.size(0), (int32_t)a.size(1), (int32_t)iters, (float)eps,
                                         stream()),
              "mhc_sinkhorn_knopp_fwd");
        ctx->save_for_backward({inp, out});
        ctx->saved_data["iters"] = iters;
        ctx->saved_data["eps"] = eps;
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const auto sv = ctx->get_saved_variables();
        const Tensor g = f32c(grads[0]);
        check_device("sinkhorn_knopp_bwd", {&g, &sv[0]});
        const at::DeviceGuard guard(g.device());
        TORCH_CHECK(g.sizes() == sv[0].sizes(), "grad_out shape must match inp");
        const Tensor a = sv[0].contiguous();
        Tensor gi = at::empty_like(a);
        check(lib.mhc_sinkhorn_knopp_bwd(fp(g), fp(a), nullptr, fp(gi), a.size(0), (int32_t)a.size(1),
                                         (int32_t)ctx->saved_data["iters"].toInt(),
                                         (float)ctx->saved_data["eps"].toDouble(), stream()),
              "mhc_sinkhorn_knopp_bwd");
        return {gi, Tensor(), Tensor()};
    }
};

struct RmsNorm : public torch::autograd::Function<RmsNorm> {
    static Tensor forward(AutogradContext* ctx, const Tensor& inp, const Tensor& w_in, double eps) {
        check_device("rmsnorm_fwd", {&inp, &w_in});
        const at::DeviceGuard guard(inp.device());
        TORCH_CHECK(inp.dim() == 2, "Input must be 2D tensor [B, C]");
        const Tensor x = storage(inp);
        const int64_t B = x.size(0), C = x.size(1);
        TORCH_CHECK(w_in.numel() == C, "weight must have C elements");
        const Tensor w = f32c(w_in);
        Tensor out = at::empty_like(x);
        Tensor rms = at::empty({B}, x.options().dtype(at::kFloat));
        check(lib.mhc_rmsnorm_fwd(x.data_ptr(), dtype_code(x.scalar_type()), fp(w), out.data_ptr(), fp(rms), B,
                                  (int32_t)C, (float)eps, stream()),
              "mhc_rmsnorm_fwd");
        ctx->save_for_backward({inp, w_in, rms});
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const auto sv = ctx->get_saved_variables();
        const Tensor &inp = sv[0], &w_in = sv[1], &rms = sv[2];
        check_device("rmsnorm_bwd", {&grads[0], &inp, &w_in, &rms});
        const at::DeviceGuard guard(inp.device());
        const Tensor x = storage(inp);
        const int64_t B = x.size(0), C = x.size(1);
        const Tensor g = grads[0].to(x.scalar_type()).contiguous();
        TORCH_CHECK(g.sizes() == x.sizes(), "grad_out shape must match inp");
        const Tensor w = f32c(w_in);
        Tensor gx = at::empty_like(x);
        Tensor gw = at::empty({C}, x.options().dtype(at::kFloat));
        const int dt = dtype_code(x.scalar_type());
        const size_t wsb = lib.mhc_rmsnorm_bwd_workspace_size(B, (int32_t)C, dt);
        Tensor ws = workspace(wsb, x);
        check(lib.mhc_rmsnorm_bwd(g.data_ptr(), x.data_ptr(), dt, fp(w), fp(rms), gx.data_ptr(), fp(gw), ws.data_ptr(),
                                  wsb, B, (int32_t)C, stream()),
              "mhc_rmsnorm_bwd");
        return {gx.to(inp.scalar_type()), gw, Tensor()};
    }
};

struct Aggregate : public torch::autograd::Function<Aggregate> {
    static Tensor forward(AutogradContext* ctx, const Tensor& inp, const Tensor& h_in) {
        const char* fn = "stream_aggregate_fwd";
        check_device(fn, {&inp, &h_in});
        const at::DeviceGuard guard(inp.device());
        TORCH_CHECK(inp.dim() == 3, "Input must be 3D tensor [B, n, C]");
        const Tensor x = storage(inp);
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
        const auto [h, hs] = coef_view(fn, h_in, B, n);
        Tensor out = at::empty({B, C}, x.options());
        Tensor act = at::empty({B, n}, x.options().dtype(at::kFloat));
        check(lib.mhc_stream_aggregate_fwd(x.data_ptr(), dtype_code(x.scalar_type()), fp(h), hs, out.data_ptr(),
                                           fp(act), B, (int32_t)n, (int32_t)C, stream()),
              "mhc_stream_aggregate_fwd");
        ctx->save_for_backward({inp, act});
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const auto sv = ctx->get_saved_variables();
        const Tensor &inp = sv[0], &act = sv[1];
        check_device("stream_aggregate_bwd", {&grads[0], &inp, &act});
        const at::DeviceGuard guard(inp.device());
        const Tensor x = storage(inp);
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
        const Tensor g = grads[0].to(x.scalar_type()).contiguous();
        TORCH_CHECK(g.dim() == 2 && g.size(0) == B && g.size(1) == C, "grad_out must be [B, C]");
        Tensor gx = at::empty_like(x);
        Tensor graw = at::empty({B, n}, act.options());
        check(lib.mhc_stream_aggregate_bwd(g.data_ptr(), x.data_ptr(), dtype_code(x.scalar_type()), fp(act), n,
                                           gx.data_ptr(), nullptr, fp(graw), B, (int32_t)n, (int32_t)C, stream()),
              "mhc_stream_aggregate_bwd");
        return {gx.to(inp.scalar_type()), graw};
    }
};

struct Distribute : public torch::autograd::Function<Distribute> {
    static Tensor forward(AutogradContext* ctx, const Tensor& y_in, const Tensor& h_in, const Tensor& m_in,
                          const Tensor& x_in) {
        const char* fn = "stream_distribute_mix_add_fwd";
        check_device(fn, {&y_in, &h_in, &m_in, &x_in});
        const at::DeviceGuard guard(x_in.device());
        TORCH_CHECK(x_in.dim() == 3, "x_inp must be 3D tensor [B, n, C]");
        const Tensor x = storage(x_in);
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
        const Tensor y = y_in.to(x.scalar_type()).contiguous();
        TORCH_CHECK(y.dim() == 2 && y.size(0) == B && y.size(1) == C, "y_norm must be [B, C]");
        const auto [h, hs] = coef_view(fn, h_in, B, n);
        const auto [m, ms] = coef_view(fn, m_in, B, n * n);
        const auto f32 = x.options().dtype(at::kFloat);
        Tensor out = at::empty({B, n, C}, f32);
        Tensor act = at::empty({B, n}, f32);
        check(lib.mhc_stream_distribute_mix_add_fwd(y.data_ptr(), fp(h), hs, fp(m), ms, x.data_ptr(),
                                                    dtype_code(x.scalar_type()), fp(out), fp(act), B, (int32_t)n,
                                                    (int32_t)C, stream()),
              "mhc_stream_distribute_mix_add_fwd");
        ctx->save_for_backward({x_in, y_in, m_in, act});
        return out;
    }

    static tensor_list backward(AutogradContext* ctx, tensor_list grads) {
        const char* fn = "stream_distribute_mix_add_bwd";
        const auto sv = ctx->get_saved_variables();
        const Tensor &x_in = sv[0], &y_in = sv[1], &m_in = sv[2], &act = sv[3];
        check_device(fn, {&grads[0], &x_in, &y_in, &m_in, &act});
        const at::DeviceGuard guard(x_in.device());
        const Tensor x = storage(x_in);
        const int64_t B = x.size(0), n = x.size(1), C = x.size(2);
        const Tensor y = y_in.to(x.scalar_type()).contiguous();
        const Tensor g = f32c(grads[0]);
        TORCH_CHECK(g.sizes() == x.sizes(), "grad_out shape must match x_inp");
        const auto [m, ms] = coef_view(fn, m_in, B, n * n);
        const auto f32 = x.options().dtype(at::kFloat);
        Tensor gx = at::empty_like(x), gy = at::empty({B, C}, x.options());
        Tensor gm = at::empty({B, n, n}, f32), graw = at::empty({B, n}, f32);
        check(lib.mhc_stream_distribute_mix_add_bwd(fp(g), x.data_ptr(), y.data_ptr(), dtype_code(x.scalar_type()),
                                                    fp(m), ms, fp(act), n, gx.data_ptr(), gy.data_ptr(), fp(gm),
                                                    nullptr, fp(graw), B, (int32_t)n, (int32_t)C, stream()),
              "mhc_stream_distribute_mix_add_bwd");
        return {gy.to(y_in.scalar_type()), graw, gm, gx.to(x_in.scalar_type())};
    }
};

Tensor sinkhorn_knopp(const Tensor& inp, int64_t iters, double eps) {
    require_bound();
    return Sinkhorn::apply(inp, iters, eps);
}

Tensor rmsnorm(const Tensor& inp, const Tensor& w, double eps) {
    require_bound();
    return RmsNorm::apply(inp, w, eps);
}

Tensor stream_aggregate(const Tensor& inp, const Tensor& h) {
    require_bound();
    return Aggregate::apply(inp, h);
}

Tensor stream_distribute_mix_add(const Tensor& y, const Tensor& h, const Tensor& m, const Tensor& x) {
    require_bound();
    return Distribute::apply(y, h, m, x);
}

Tensor static_layer(const Tensor& x, const Tensor& w, const Tensor& hp, const Tensor& hq, const Tensor& hr,
                    int64_t iters, double sk_eps, double rms_eps) {
    require_bound();
    return StaticLayer::apply(x, w, hp, hq, hr, iters, sk_eps, rms_eps);
}

Tensor dynamic_layer(const Tensor& x, const Tensor& w, const Tensor& pp, const Tensor& pq, const Tensor& pr,
                     const Tensor& ap, const Tensor& aq, const Tensor& ar, const Tensor& bp, const Tensor& bq,
                     const Tensor& br, int64_t iters, double sk_eps, double rms_eps) {
    require_bound();
    return DynamicLayer::apply(x, w, pp, pq, pr, ap, aq, ar, bp, bq, br, iters, sk_eps, rms_eps);
}

Tensor static_wrapper(const Tensor& residual, const Tensor& branch, const Tensor& w, const Tensor& hp,
                      const Tensor& hq, const Tensor& hr, const std::string& mode, int64_t n, int64_t iters,
                      double sk_eps, double rms_eps) {
    require_bound();
    const int32_t m = wrapper_mode(mode, n, "wrapper_static_fwd");
    return StaticWrapper::apply(residual, branch, w, hp, hq, hr, (int64_t)m, n, iters, sk_eps, rms_eps);
}

Tensor dynamic_wrapper(const Tensor& residual, const Tensor& branch, const Tensor& w, const Tensor& pp,
                       const Tensor& pq, const Tensor& pr, const Tensor& ap, const Tensor& aq, const Tensor& ar,
                       const Tensor& bp, const Tensor& bq, const Tensor& bres, const std::string& mode, int64_t n,
                       int64_t iters, double sk_eps, double rms_eps) {
    require_bound();
    const int32_t m = wrapper_mode(mode, n, "wrapper_dynamic_fwd");
    return DynamicWrapper::apply(residual, branch, w, pp, pq, pr, ap, aq, ar, bp, bq, bres, (int64_t)m, n, iters,
                                 sk_eps, rms_eps);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "C++ autograd nodes of the fused mHC layers and the standalone operators over libmhc_hip's C ABI";
    m.def("entry_names", &entry_names, "C-ABI entry points bind() needs");
    m.def("bind", &bind, "set the C-ABI entry points from {name: address}");
    m.def("static_layer", &static_layer,
          "static-H layer with autograd: (x, weight, H_pre, H_post, H_res, num_iters, sinkhorn_eps, "
          "rmsnorm_eps) -> fp32 [B, n, C]");
    m.def("dynamic_layer", &dynamic_layer,
          "dynamic-H layer with autograd: (x, weight, phi_pre, phi_post, phi_res, alpha_pre, alpha_post, "
          "alpha_res, b_pre, b_post, b_res, num_iters, sinkhorn_eps, rmsnorm_eps) -> fp32 [B, n, C]");
    m.def("static_wrapper", &static_wrapper,
          "fused static-H MHCResidualWrapper with autograd: (residual, branch, weight, H_pre, H_post, H_res, "
          "residual_mode, n, num_iters, sinkhorn_eps, rmsnorm_eps) -> fp32 [tokens, C]");
    m.def("dynamic_wrapper", &dynamic_wrapper,
          "fused dynamic-H MHCResidualWrapper with autograd: (residual, branch, weight, phi_pre, phi_post, phi_res, "
          "alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res, residual_mode, n, num_iters, sinkhorn_eps, "
          "rmsnorm_eps) -> fp32 [tokens, C]");
    m.def("dynamic_infer", &dynamic_infer,
          "forward-only dynamic-H layer: (x, packed, alpha_pre, alpha_post, alpha_res, b_pre, b_post, b_res, "
          "num_iters, sinkhorn_eps, rmsnorm_eps, out_bf16) -> [B, n, C]");
    m.def("sinkhorn_knopp", &sinkhorn_knopp, "(inp [B, n, n] fp32, num_iters, eps) with autograd");
    m.def("rmsnorm", &rmsnorm, "(inp [B, C], weight, eps) with autograd");
    m.def("stream_aggregate", &stream_aggregate, "(inp [B, n, C], H_pre_raw [B, n]) with autograd");
    m.def("stream_distribute_mix_add", &stream_distribute_mix_add,
          "(y_norm [B, C], H_post_raw [B, n], M [B, n, n], x_inp [B, n, C]) -> fp32 [B, n, C] with autograd");
}
