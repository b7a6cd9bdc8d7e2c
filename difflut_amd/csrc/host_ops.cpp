// The layer operators' host path: torch autograd functions over the C ABI of libdifflut_hip.so.
//
// One call of a layer is a handful of allocations and one library call each way.  Written as Python autograd functions over
// ctypes, forward and backward of a small layer took 115-130 us of host time against 60-75 us on the device (1024 rows, 4096 ->
// 4096 probabilistic nodes; 1000 rows, 3137 -> 2999 DWN nodes); a backward in Python also hands the interpreter lock from the
// calling thread to autograd's and back.  The same calls here take neither.
//
// The conventions are those of the operators' Python side (difflut_amd/ops.py): inputs made contiguous fp32, outputs new
// tensors, everything on torch's current stream, errors as RuntimeError, no synchronisation.
#include <c10/hip/HIPStream.h>
#include <climits>
#include <dlfcn.h>
#include <torch/extension.h>

#include "../../include/difflut_hip.h"

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

// ------------------------------------------------------------------ the library
#define DL_FUNCTIONS(X)                                                                                                  \
    X(dl_error_string) X(dl_dwn_saved_bytes) X(dl_dwn_fwd_workspace_bytes) X(dl_dwn_bwd_workspace_bytes)                 \
    X(dl_dwn_bwd_reads_x) X(dl_dwn_layer_fwd) X(dl_dwn_layer_bwd) X(dl_dwn_layer_bwd_nodes) X(dl_dwn_stable_layer_bwd)   \
    X(dl_dwn_stable_raw_bwd)                                                                                             \
    X(dl_table_sigmoid_fwd) X(dl_table_sigmoid_bwd) X(dl_hybrid_saved_bytes) X(dl_hybrid_fwd_workspace_bytes)            \
    X(dl_hybrid_bwd_workspace_bytes) X(dl_hybrid_bwd_saved_workspace_bytes) X(dl_hybrid_layer_fwd)                       \
    X(dl_hybrid_layer_bwd) X(dl_hybrid_layer_bwd_saved) X(dl_hybrid_raw_fwd) X(dl_hybrid_raw_bwd) X(dl_prob_saved_bytes) X(dl_prob_bwd_saved_workspace_bytes)      \
    X(dl_prob_layer_fwd) X(dl_prob_layer_fwd_nodes) X(dl_prob_layer_bwd) X(dl_prob_layer_bwd_nodes)                      \
    X(dl_prob_ordered_saved_bytes) X(dl_prob_ordered_bwd_workspace_bytes) X(dl_prob_ordered_fwd) X(dl_prob_ordered_bwd)  \
    X(dl_soft_map_saved_bytes) X(dl_soft_map_workspace_bytes) X(dl_soft_map_fwd) X(dl_soft_map_bwd) X(dl_unfold_rows)    \
    X(dl_unfold_flip) X(dl_fold) X(dl_dwn_planes_bytes) X(dl_dwn_tiled_bytes) X(dl_dwn_pack_planes)                      \
    X(dl_thermometer_planes) X(dl_dwn_groups_workspace_bytes) X(dl_dwn_eval_groups_workspace_bytes) X(dl_dwn_layer_fwd_planes)                                 \
    X(dl_dwn_layer_fwd_planes_groups) X(dl_dwn_layer_eval_planes) X(dl_dwn_layer_eval_planes_groups) X(dl_dwn_layer_rows) X(dl_dwn_rows_pay) \
    X(dl_dwn_layer_bwd_groups) X(dl_dwn_layer_bwd_tiled) X(dl_dwn_chain_fusable) X(dl_dwn_bwd_fused_workspace_bytes)     \
    X(dl_dwn_layer_bwd_chain_fused) X(dl_dwn_chain_first_fusable) X(dl_dwn_bwd_first_workspace_bytes)                    \
    X(dl_dwn_layer_bwd_chain_first) X(dl_cross_entropy_workspace_bytes) X(dl_cross_entropy) X(dl_adam_step)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
    DL_FUNCTIONS(X)
#undef X
} L;

void load(const std::string &path) {
    void *handle = dlopen(path.c_str(), RTLD_NOW | RTLD_LOCAL);
    TORCH_CHECK(handle, "cannot load ", path, ": ", dlerror());
#define X(name)                                                          \
    L.name = reinterpret_cast<decltype(&::name)>(dlsym(handle, #name));  \
    TORCH_CHECK(L.name, path, " has no ", #name);
    DL_FUNCTIONS(X)
#undef X
}

void check(int code) {
    TORCH_CHECK(code == 0, "libdifflut_hip: ", L.dl_error_string(code), " (code ", code, ")");
}
void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

void require_device(const Tensor &t) {
    TORCH_CHECK(!t.defined() || t.is_cuda(), "difflut_amd kernels run on ROCm devices only; got a tensor on '", t.device(),
                "'. All tensors of one call must be on the same ROCm device (or all on the CPU).");
}
Tensor f32(const Tensor &t) {
    return t.scalar_type() == at::kFloat && t.is_contiguous() ? t : t.contiguous().to(at::kFloat);
}
Tensor floats(at::IntArrayRef sizes, const Tensor &like) {
    return at::empty(sizes, at::TensorOptions().dtype(at::kFloat).device(like.device()));
}
Tensor bytes(size_t n, const Tensor &like) {
    return at::empty({(int64_t)std::max<size_t>(n, 256)}, at::TensorOptions().dtype(at::kByte).device(like.device()));
}
const float *in(const Tensor &t) { return t.defined() ? t.const_data_ptr<float>() : nullptr; }
float *out(const Tensor &t) { return t.defined() ? t.mutable_data_ptr<float>() : nullptr; }
void *raw(const Tensor &t) { return t.defined() ? t.mutable_data_ptr() : nullptr; }
const int32_t *ints(const Tensor &t) { return t.const_data_ptr<int32_t>(); }

// per-node values as the float32 device array [N] the kernels read; a layer's bank hands over just that
Tensor per_node(const Tensor &v, int64_t N, const Tensor &like) {
    if (v.scalar_type() == at::kFloat && v.dim() == 1 && v.size(0) == N && v.device() == like.device() && !v.requires_grad() &&
        v.is_contiguous())
        return v;
    return v.detach().to(like.device(), at::kFloat).reshape({-1}).expand({N}).contiguous();
}

// ------------------------------------------------------------------ what a call keeps for its backward
struct Plan {
    Tensor idx, inv_ptr, inv_pos;
    int N, k, I;
};
struct Dims {
    int B, I, N, k, O;
};
#define DIMS(d) (d).B, (d).I, (d).N, (d).k, (d).O
struct Kept : torch::CustomClassHolder {
    Plan plan;
    Dims dims{};
    Tensor alpha_n, beta_n;         // every node's own values, or
    float alpha = 0.0f, beta = 0.0f;  // one for the layer (with beta_n: beta = max |beta_n|)
    bool ordered = false;             // the plan is that of nodes that take their inputs in order
};
template <typename T>
void keep(AutogradContext *ctx, c10::intrusive_ptr<T> kept) {
    ctx->saved_data["kept"] = c10::IValue::make_capsule(std::move(kept));
}
template <typename T>
c10::intrusive_ptr<T> kept_of(AutogradContext *ctx) {
    return c10::static_intrusive_pointer_cast<T>(ctx->saved_data["kept"].toCapsule());
}
Dims lookup_dims(const Tensor &x, const Tensor &luts, const Plan &p) {
    TORCH_CHECK(x.dim() == 2 && luts.dim() == 3, "expected x [B, I] and tables [N, O, 2^k], got ", x.sizes(), " and ", luts.sizes());
    TORCH_CHECK(luts.size(0) == p.N && luts.size(2) == (int64_t)1 << p.k && x.size(1) == p.I, "shape mismatch: x ", x.sizes(),
                ", luts ", luts.sizes(), ", mapping [", p.N, ",", p.k, "] over ", p.I, " inputs");
    return {(int)x.size(0), (int)x.size(1), (int)luts.size(0), p.k, (int)luts.size(1)};
}
// whether the DWN backward needs x: not where the forward leaves the address of every node and row
bool backward_reads_x(const Dims &d) { return L.dl_dwn_bwd_reads_x(d.N, d.k, d.O) != 0; }
std::pair<Tensor, Tensor> dwn_lookup(const Tensor &x, const Tensor &luts, const Plan &p, const Dims &d) {
    Tensor y = floats({d.B, (int64_t)d.N * d.O}, x), saved = bytes(L.dl_dwn_saved_bytes(DIMS(d)), x),
           ws = bytes(L.dl_dwn_fwd_workspace_bytes(DIMS(d)), x);
    check(L.dl_dwn_layer_fwd(in(x), ints(p.idx), in(luts), out(y), raw(saved), raw(ws), ws.numel(), DIMS(d), stream()));
    return {y, saved};
}

// ------------------------------------------------------------------ DWN
struct DwnLayer : torch::autograd::Function<DwnLayer> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const Tensor &luts_, const Kept *given) {
        require_device(x_);
        require_device(luts_);
        const Tensor x = f32(x_), luts = f32(luts_);
        auto k = c10::make_intrusive<Kept>(*given);
        k->dims = lookup_dims(x, luts, k->plan);
        auto [y, saved] = dwn_lookup(x, luts, k->plan, k->dims);
        if (k->alpha_n.defined()) {
            k->alpha_n = per_node(k->alpha_n, k->dims.N, x);
            k->beta_n = per_node(k->beta_n, k->dims.N, x);
        }
        ctx->save_for_backward({luts, saved, backward_reads_x(k->dims) ? x : Tensor()});
        keep(ctx, std::move(k));
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor &luts = s[0], &saved = s[1], &x = s[2];
        const auto k = kept_of<Kept>(ctx);
        const Dims &d = k->dims;
        const Plan &p = k->plan;
        const Tensor gy = f32(grads[0]);
        const Tensor gx = ctx->needs_input_grad(0) ? floats({d.B, d.I}, gy) : Tensor();
        const Tensor gl = at::empty_like(luts), ws = bytes(L.dl_dwn_bwd_workspace_bytes(DIMS(d)), gy);
        if (k->alpha_n.defined())
            check(L.dl_dwn_layer_bwd_nodes(in(x), raw(saved), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(luts), in(gy),
                                           in(k->alpha_n), in(k->beta_n), k->beta, out(gx), out(gl), raw(ws), ws.numel(), DIMS(d),
                                           stream()));
        else
            check(L.dl_dwn_layer_bwd(in(x), raw(saved), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(luts), in(gy), k->alpha,
                                     k->beta, out(gx), out(gl), raw(ws), ws.numel(), DIMS(d), stream()));
        return {gx, gl, Tensor()};
    }
};

struct TableSigmoid : torch::autograd::Function<TableSigmoid> {
    static Tensor forward(AutogradContext *ctx, const Tensor &raw_) {
        require_device(raw_);
        const Tensor r = f32(raw_), luts = at::empty_like(r);
        check(L.dl_table_sigmoid_fwd(in(r), out(luts), r.numel(), stream()));
        ctx->save_for_backward({luts});
        return luts;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor gl = f32(grads[0]), graw = at::empty_like(s[0]);
        check(L.dl_table_sigmoid_bwd(in(gl), in(s[0]), out(graw), s[0].numel(), stream()));
        return {graw};
    }
};

struct DwnStableLayer : torch::autograd::Function<DwnStableLayer> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const Tensor &luts_, const Tensor &scale_, const Kept *given) {
        require_device(x_);
        require_device(luts_);
        require_device(scale_);
        const Tensor x = f32(x_), luts = f32(luts_), scale = f32(scale_.detach()).reshape({-1});
        TORCH_CHECK(scale.numel() == luts.size(0), "gradient_scale has ", scale.numel(), " entries for ", luts.size(0), " nodes");
        auto k = c10::make_intrusive<Kept>(*given);
        k->dims = lookup_dims(x, luts, k->plan);
        auto [y, saved] = dwn_lookup(x, luts, k->plan, k->dims);
        ctx->save_for_backward({luts, saved, scale, backward_reads_x(k->dims) ? x : Tensor()});
        keep(ctx, std::move(k));
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const auto k = kept_of<Kept>(ctx);
        const Dims &d = k->dims;
        const Plan &p = k->plan;
        const Tensor gy = f32(grads[0]);
        const Tensor gx = ctx->needs_input_grad(0) ? floats({d.B, d.I}, gy) : Tensor();
        const Tensor gl = at::empty_like(s[0]), ws = bytes(L.dl_dwn_bwd_workspace_bytes(DIMS(d)), gy);
        check(L.dl_dwn_stable_layer_bwd(in(s[3]), raw(s[1]), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(s[0]), in(gy), in(s[2]),
                                        out(gx), out(gl), raw(ws), ws.numel(), DIMS(d), stream()));
        return {gx, gl, Tensor(), Tensor()};
    }
};

// The same on the tables' raw values: one node, and the sigmoid's adjoint where the table gradient is written.
struct DwnStableRaw : torch::autograd::Function<DwnStableRaw> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const Tensor &raw_, const Tensor &scale_, const Kept *given) {
        require_device(scale_);
        const Tensor x = f32(x_), w = f32(raw_), scale = f32(scale_.detach()).reshape({-1}), luts = at::empty_like(w);
        TORCH_CHECK(scale.numel() == w.size(0), "gradient_scale has ", scale.numel(), " entries for ", w.size(0), " nodes");
        auto k = c10::make_intrusive<Kept>(*given);
        k->dims = lookup_dims(x, w, k->plan);
        check(L.dl_table_sigmoid_fwd(in(w), out(luts), w.numel(), stream()));
        auto [y, saved] = dwn_lookup(x, luts, k->plan, k->dims);
        ctx->save_for_backward({luts, saved, scale});
        keep(ctx, std::move(k));
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const auto k = kept_of<Kept>(ctx);
        const Dims &d = k->dims;
        const Plan &p = k->plan;
        const Tensor gy = f32(grads[0]);
        const Tensor gx = ctx->needs_input_grad(0) ? floats({d.B, d.I}, gy) : Tensor();
        const Tensor graw = at::empty_like(s[0]), ws = bytes(L.dl_dwn_bwd_workspace_bytes(DIMS(d)), gy);
        check(L.dl_dwn_stable_raw_bwd(raw(s[1]), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(s[0]), in(gy), in(s[2]), out(gx), out(graw),
                                      raw(ws), ws.numel(), DIMS(d), stream()));
        return {gx, graw, Tensor(), Tensor()};
    }
};

struct HybridLayer : torch::autograd::Function<HybridLayer> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const Tensor &luts_, const Kept *given, bool keep_tiles) {
        require_device(x_);
        require_device(luts_);
        const Tensor x = f32(x_), luts = f32(luts_);
        auto k = c10::make_intrusive<Kept>(*given);
        const Dims d = k->dims = lookup_dims(x, luts, k->plan);
        Tensor y, tiles;
        if (keep_tiles && d.k <= DL_MAX_FAST_K) {
            y = floats({d.B, (int64_t)d.N * d.O}, x);
            tiles = bytes(L.dl_hybrid_saved_bytes(DIMS(d)), x);
            const Tensor ws = bytes(L.dl_hybrid_fwd_workspace_bytes(DIMS(d)), x);
            check(L.dl_hybrid_layer_fwd(in(x), ints(k->plan.idx), in(luts), out(y), raw(tiles), tiles.numel(), raw(ws), ws.numel(),
                                        DIMS(d), stream()));
        } else {
            y = dwn_lookup(x, luts, k->plan, d).first;
        }
        // the backward reads x itself only where it was not re-tiled
        ctx->save_for_backward({tiles.defined() && tiles.numel() > 256 ? Tensor() : x, luts, tiles});
        keep(ctx, std::move(k));
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &luts = s[1], &tiles = s[2];
        const auto k = kept_of<Kept>(ctx);
        const Dims &d = k->dims;
        const Plan &p = k->plan;
        const Tensor gy = f32(grads[0]);
        const Tensor gx = ctx->needs_input_grad(0) ? floats({d.B, d.I}, gy) : Tensor();
        const Tensor gl = at::empty_like(luts);
        if (!tiles.defined()) {
            const Tensor ws = bytes(L.dl_hybrid_bwd_workspace_bytes(DIMS(d)), gy);
            check(L.dl_hybrid_layer_bwd(in(x), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(luts), in(gy), out(gx), out(gl),
                                        raw(ws), ws.numel(), DIMS(d), stream()));
        } else {
            const Tensor ws = bytes(L.dl_hybrid_bwd_saved_workspace_bytes(DIMS(d)), gy);
            check(L.dl_hybrid_layer_bwd_saved(in(x), raw(tiles), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(luts), in(gy),
                                              out(gx), out(gl), raw(ws), ws.numel(), DIMS(d), stream()));
        }
        return {gx, gl, Tensor(), Tensor()};
    }
};

// The same on the tables' raw values, whose sigmoid and its gradient are part of the launches: for a layer small enough that what it
// costs is launches and autograd nodes, two of six and one of two.
struct HybridRaw : torch::autograd::Function<HybridRaw> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const Tensor &raw_, const Kept *given) {
        const Tensor x = f32(x_), w = f32(raw_), luts = at::empty_like(w);
        auto k = c10::make_intrusive<Kept>(*given);
        const Dims d = k->dims = lookup_dims(x, w, k->plan);
        const Tensor y = floats({d.B, (int64_t)d.N * d.O}, x), tiles = bytes(L.dl_hybrid_saved_bytes(DIMS(d)), x),
                     ws = bytes(L.dl_hybrid_fwd_workspace_bytes(DIMS(d)), x);
        check(L.dl_hybrid_raw_fwd(in(x), ints(k->plan.idx), in(w), out(luts), out(y), raw(tiles), tiles.numel(), raw(ws), ws.numel(), DIMS(d),
                                  stream()));
        ctx->save_for_backward({luts, tiles});
        keep(ctx, std::move(k));
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const auto k = kept_of<Kept>(ctx);
        const Dims &d = k->dims;
        const Plan &p = k->plan;
        const Tensor gy = f32(grads[0]);
        const Tensor gx = ctx->needs_input_grad(0) ? floats({d.B, d.I}, gy) : Tensor();
        const Tensor graw = at::empty_like(s[0]), ws = bytes(L.dl_hybrid_bwd_saved_workspace_bytes(DIMS(d)), gy);
        check(L.dl_hybrid_raw_bwd(raw(s[1]), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(s[0]), in(gy), out(gx), out(graw), raw(ws),
                                  ws.numel(), DIMS(d), stream()));
        return {gx, graw, Tensor()};
    }
};

// ------------------------------------------------------------------ probabilistic
struct ProbLayer : torch::autograd::Function<ProbLayer> {
    // given->alpha_n: every node's temperature, or given->alpha for the layer
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const Tensor &raw_, const Kept *given) {
        require_device(x_);
        require_device(raw_);
        const Tensor x = f32(x_), w = f32(raw_);
        auto k = c10::make_intrusive<Kept>(*given);
        const Plan &p = k->plan;
        TORCH_CHECK(x.dim() == 2 && w.dim() == 3, "expected x [B, I] and raw_weights [N, 2^k, O], got ", x.sizes(), " and ", w.sizes());
        TORCH_CHECK(w.size(0) == p.N && w.size(1) == (int64_t)1 << p.k && x.size(1) == p.I, "shape mismatch: x ", x.sizes(),
                    ", raw_weights ", w.sizes(), ", mapping [", p.N, ",", p.k, "] over ", p.I, " inputs");
        const Dims d = k->dims = {(int)x.size(0), (int)x.size(1), (int)w.size(0), p.k, (int)w.size(2)};
        // kernels of their own for nodes of one output that take their inputs in order: they save the re-tiling of x and of its
        // gradient (512 rows, 8000 nodes of six inputs: 156 -> 92 us); a block is sixteen nodes, so few nodes stay on blocks of four
        k->ordered = k->ordered && d.O == 1 && d.k <= DL_MAX_FAST_K && d.N > 12 && d.I < (1 << 23);
        const Tensor y = floats({d.B, (int64_t)d.N * d.O}, x),
                     saved = bytes(k->ordered ? L.dl_prob_ordered_saved_bytes(d.N, d.k) : L.dl_prob_saved_bytes(DIMS(d)), x);
        Tensor T;
        if (k->alpha_n.defined()) {
            T = per_node(k->alpha_n, d.N, x);
            k->alpha_n = Tensor();
        }
        if (k->ordered) {
            check(L.dl_prob_ordered_fwd(in(x), in(w), k->alpha, in(T), out(y), raw(saved), saved.numel(), d.B, d.N, d.k, stream()));
        } else if (T.defined()) {
            check(L.dl_prob_layer_fwd_nodes(in(x), ints(p.idx), in(w), in(T), out(y), raw(saved), saved.numel(), DIMS(d), stream()));
        } else {
            check(L.dl_prob_layer_fwd(in(x), ints(p.idx), in(w), k->alpha, out(y), raw(saved), saved.numel(), DIMS(d), stream()));
        }
        ctx->save_for_backward({x, w, saved, T});
        keep(ctx, std::move(k));
        return y;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &w = s[1], &saved = s[2], &T = s[3];
        const auto k = kept_of<Kept>(ctx);
        const Dims &d = k->dims;
        const Plan &p = k->plan;
        const Tensor gy = f32(grads[0]);
        const Tensor gx = ctx->needs_input_grad(0) ? floats({d.B, d.I}, gy) : Tensor();
        const Tensor gw = at::empty_like(w),
                     ws = bytes(k->ordered ? L.dl_prob_ordered_bwd_workspace_bytes(d.B, d.N, d.k) : L.dl_prob_bwd_saved_workspace_bytes(DIMS(d)), gy);
        if (k->ordered)
            check(L.dl_prob_ordered_bwd(in(x), raw(saved), k->alpha, in(T), in(gy), out(gx), out(gw), raw(ws), ws.numel(), d.B, d.N, d.k,
                                        stream()));
        else if (T.defined())
            check(L.dl_prob_layer_bwd_nodes(in(x), raw(saved), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(w), in(T), in(gy),
                                            out(gx), out(gw), raw(ws), ws.numel(), DIMS(d), stream()));
        else
            check(L.dl_prob_layer_bwd(in(x), raw(saved), ints(p.idx), ints(p.inv_ptr), ints(p.inv_pos), in(w), k->alpha, in(gy), out(gx),
                                      out(gw), raw(ws), ws.numel(), DIMS(d), stream()));
        return {gx, gw, Tensor()};
    }
};

// ------------------------------------------------------------------ soft connectivity
struct SoftMap : torch::autograd::Function<SoftMap> {
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, const Tensor &W_, double tau, int64_t precision) {
        require_device(x_);
        require_device(W_);
        const Tensor x = f32(x_), W = f32(W_);
        TORCH_CHECK_VALUE(x.dim() == 2, "expected x [B, I], got ", x.sizes());
        const int B = (int)x.size(0), I = (int)x.size(1), M = (int)W.size(0), prec = (int)precision;
        TORCH_CHECK(W.size(1) == I, "shape mismatch: x ", x.sizes(), " vs W ", W.sizes());
        const Tensor m = floats({B, M}, x), stats = bytes(L.dl_soft_map_saved_bytes(B, I, M, prec), x),
                     ws = bytes(L.dl_soft_map_workspace_bytes(B, I, M, prec), x);
        check(L.dl_soft_map_fwd(in(x), in(W), (float)tau, out(m), (float *)raw(stats), raw(ws), ws.numel(), B, I, M, prec, stream()));
        ctx->save_for_backward({x, W, m, stats});
        ctx->saved_data["tau"] = tau;
        ctx->saved_data["precision"] = precision;
        return m;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const auto s = ctx->get_saved_variables();
        const Tensor &x = s[0], &W = s[1], &m = s[2], &stats = s[3];
        const int B = (int)x.size(0), I = (int)x.size(1), M = (int)W.size(0), prec = (int)ctx->saved_data["precision"].toInt();
        const Tensor gm = f32(grads[0]), gx = at::empty_like(x), gW = at::empty_like(W),
                     ws = bytes(L.dl_soft_map_workspace_bytes(B, I, M, prec), x);
        check(L.dl_soft_map_bwd(in(x), in(W), (float)ctx->saved_data["tau"].toDouble(), in(m), (const float *)raw(stats), in(gm), out(gx), out(gW),
                                raw(ws), ws.numel(), B, I, M, prec, stream()));
        return {gx, gW, Tensor(), Tensor()};
    }
};

// ------------------------------------------------------------------ a chain of DWN layers
struct Stack : torch::CustomClassHolder {
    std::vector<Plan> plans;
    std::vector<std::array<Tensor, 2>> per_node;    // alpha [N], beta [N] of a layer (undefined: one value for it)
    std::vector<std::array<double, 2>> scalars;     // alpha, beta - or, with per-node values, {unused, max |beta|}
    int64_t groups = 0;                             // of a GroupSum behind the last layer; 0 = none
    double tau = 1.0;
    bool encoded = false, patches = false;          // the first layer reads a thermometer code / the patches of an image
    std::array<int, 6> geom{};
    std::vector<int64_t> image;
    std::vector<Dims> dims;
};
Tensor code_thresholds(const Tensor &thresholds, int features) {
    require_device(thresholds);
    const Tensor thr = f32(thresholds);
    TORCH_CHECK(thr.dim() == 2 && thr.size(0) == features, "thresholds ", thr.sizes(), " do not match ", features, " features");
    return thr;
}
// bit-planes of the first layer's input: x itself, its thermometer code or its patch matrix; sets rows and width
Tensor first_planes(const Tensor &x, const Tensor &thresholds, const Tensor &flip_, Stack &st, int &B, int &width) {
    if (st.patches) {
        st.image = x.sizes().vec();
        TORCH_CHECK(x.dim() == 4, "expected an image batch [B, C, H, W], got ", x.sizes());
        const auto &g = st.geom;
        const int C = (int)x.size(1), H = (int)x.size(2), W = (int)x.size(3);
        const long long rows = L.dl_unfold_rows((int)x.size(0), H, W, g[0], g[1], g[2], g[3], g[4], g[5]);
        TORCH_CHECK(rows > 0, "receptive field (", g[0], ", ", g[1], ") with stride (", g[2], ", ", g[3], "), padding (", g[4], ", ",
                    g[5], ") does not fit a ", H, "x", W, " image");
        B = (int)rows, width = C * g[0] * g[1];
        const Tensor planes = bytes(L.dl_dwn_planes_bytes(B, width), x);
        Tensor flip;
        if (flip_.defined()) {
            require_device(flip_);
            TORCH_CHECK(flip_.dim() == 2 && flip_.size(0) == B && flip_.size(1) == width, "flip mask ", flip_.sizes(),
                        " does not match the patch matrix [", B, ", ", width, "]");
            flip = flip_.contiguous();
            if (flip.scalar_type() != at::kBool) flip = flip.to(at::kByte);
        }
        check(L.dl_unfold_flip(in(x), (const uint8_t *)raw(flip), nullptr, raw(planes), (int)x.size(0), C, H, W, g[0], g[1], g[2], g[3],
                               g[4], g[5], stream()));
        return planes;
    }
    TORCH_CHECK(x.dim() == 2, "expected x [B, I], got ", x.sizes());
    B = (int)x.size(0), width = (int)x.size(1);
    if (!thresholds.defined()) {
        const Tensor planes = bytes(L.dl_dwn_planes_bytes(B, width), x);
        check(L.dl_dwn_pack_planes(in(x), raw(planes), B, width, stream()));
        return planes;
    }
    const Tensor thr = code_thresholds(thresholds, width);
    const int nbits = (int)thr.size(1);
    const Tensor planes = bytes(L.dl_dwn_planes_bytes(B, width * nbits), x);
    check(L.dl_thermometer_planes(in(x), in(thr), raw(planes), B, width, nbits, stream()));
    width *= nbits;
    return planes;
}
// Whether a chain's first layer reads x itself, in one launch without planes (dl_dwn_layer_rows)
bool first_by_rows(const Tensor &x, const Tensor &thresholds, at::ArrayRef<Tensor> luts, const Plan &p, int64_t groups, bool training) {
    const Tensor &t = luts[0];
    if (x.dim() != 2 || t.dim() != 3 || (thresholds.defined() && thresholds.dim() != 2) || (luts.size() == 1 && !groups)) return false;
    const int64_t bits = thresholds.defined() ? thresholds.size(1) : 1;
    if (x.size(0) > INT_MAX || x.size(1) > INT_MAX || bits > INT_MAX || x.size(1) == 0) return false;
    return L.dl_dwn_rows_pay((int)x.size(0), (int)x.size(1), (int)bits, p.N, p.k, (int)t.size(1), luts.size() == 1 ? (int)groups : 0, training) == 1;
}
// where the first layer reads x itself: its rows and width, and the thresholds of its code (undefined: none)
Tensor as_it_comes(const Tensor &x, const Tensor &thresholds, int &B, int &width, int &nbits) {
    B = (int)x.size(0), width = (int)x.size(1);
    if (!thresholds.defined()) return thresholds;
    const Tensor thr = code_thresholds(thresholds, width);
    nbits = (int)thr.size(1);
    width *= nbits;
    return thr;
}
Dims chain_dims(size_t l, const Plan &p, const Tensor &lut, int B, int width) {
    TORCH_CHECK(lut.dim() == 3 && p.k <= DL_MAX_FAST_K && lut.size(0) == p.N && lut.size(2) == (int64_t)1 << p.k && width == p.I,
                "layer ", l, ": cannot chain (k=", p.k, ", tables ", lut.sizes(), ", mapping [", p.N, ",", p.k, "] over ", p.I,
                " inputs, incoming width ", width, ")");
    return {B, width, p.N, p.k, (int)lut.size(1)};
}

struct DwnStack : torch::autograd::Function<DwnStack> {
    // thresholds, flip: not inputs that autograd knows
    static Tensor forward(AutogradContext *ctx, const Tensor &x_, at::TensorList luts_, const Tensor *thresholds, const Tensor *flip,
                          c10::intrusive_ptr<Stack> st) {
        require_device(x_);
        const Tensor x = f32(x_);
        std::vector<Tensor> luts;
        for (const Tensor &t : luts_) {
            require_device(t);
            luts.push_back(f32(t));
        }
        int B = 0, width = 0, nbits = 1;
        st->encoded = thresholds->defined();
        Tensor planes, thr, y;
        if (!st->patches && first_by_rows(x, *thresholds, luts, st->plans[0], st->groups, true)) thr = as_it_comes(x, *thresholds, B, width, nbits);
        else planes = first_planes(x, *thresholds, *flip, *st, B, width);
        variable_list save(luts.begin(), luts.end());
        for (size_t l = 0; l < luts.size(); ++l) {
            const Plan &p = st->plans[l];
            const Dims d = chain_dims(l, p, luts[l], B, width);
            const bool last = l + 1 == luts.size();
            const Tensor kept = bytes(L.dl_dwn_saved_bytes(DIMS(d)), x);
            Tensor next;
            const bool first = !planes.defined();  // reads x itself
            if (first || ((!last || st->groups) && L.dl_dwn_rows_pay(B, 0, 1, d.N, d.k, d.O, last ? (int)st->groups : 0, 1) == 1)) {
                if (last) y = floats({B, st->groups}, x);
                else next = bytes(L.dl_dwn_planes_bytes(B, d.N * d.O), x);
                check(L.dl_dwn_layer_rows(first ? in(x) : nullptr, first ? in(thr) : nullptr, nbits, raw(planes), ints(p.idx),
                                          in(luts[l]), raw(next), last ? out(y) : nullptr, raw(kept), DIMS(d), (int)st->groups,
                                          (float)st->tau, stream()));
            } else if (last && st->groups) {
                y = floats({B, st->groups}, x);
                const Tensor ws = bytes(L.dl_dwn_groups_workspace_bytes(B, d.N, d.O, (int)st->groups), x);
                check(L.dl_dwn_layer_fwd_planes_groups(raw(planes), ints(p.idx), in(luts[l]), out(y), raw(kept), raw(ws), ws.numel(),
                                                       DIMS(d), (int)st->groups, (float)st->tau, stream()));
            } else {
                if (last) y = floats({B, (int64_t)d.N * d.O}, x);
                else next = bytes(L.dl_dwn_planes_bytes(B, d.N * d.O), x);
                check(L.dl_dwn_layer_fwd_planes(raw(planes), ints(p.idx), in(luts[l]), out(y), raw(next), raw(kept), DIMS(d), stream()));
            }
            save.push_back(kept);
            st->dims.push_back(d);
            planes = next;
            width = d.N * d.O;
        }
        ctx->save_for_backward(std::move(save));
        keep(ctx, std::move(st));
        return y;
    }

    static variable_list backward(AutogradContext *ctx, variable_list gys) {
        const auto saved_all = ctx->get_saved_variables();
        const auto st = kept_of<Stack>(ctx);
        const int n = (int)st->dims.size();
        const Tensor *luts = saved_all.data(), *saved = luts + n;
        const bool wants_input_grad = ctx->needs_input_grad(0) && !st->encoded;
        Tensor g = f32(gys[0]);
        const Tensor like = g;
        int tiled = 0;
        std::vector<Tensor> grads(n);
        std::vector<bool> have_tables(n, false);  // table gradient already produced by the call for the layer behind
        auto tiled_array = [&](int B, int C) { return floats({(int64_t)(L.dl_dwn_tiled_bytes(B, C) / 4)}, like); };
        for (int l = n - 1; l >= 0; --l) {
            const Dims &d = st->dims[l];
            const Plan &p = st->plans[l];
            const bool nodes = st->per_node[l][0].defined();
            const float beta_max = (float)st->scalars[l][1];
            // the second layer's call can give the first layer's input gradient too: its own is then not stored
            const bool first = l == 1 && st->patches && wants_input_grad && st->dims[0].O == 1 && nodes && st->per_node[0][0].defined() &&
                               L.dl_dwn_chain_first_fusable(DIMS(d), st->dims[0].k, st->dims[0].I, beta_max) == 1;
            // the gather of this layer can fill the table gradient of the layer in front as it goes: that layer's own
            // pass over its [B, N] output gradient is then left out
            const int k_prev = l > 0 ? st->dims[l - 1].k : 0;
            const bool fuse = first || (nodes && l > 0 && st->dims[l - 1].O == 1 && L.dl_dwn_chain_fusable(DIMS(d), k_prev, beta_max) == 1);
            // the first layer's table gradient is then all that is left: nobody reads this input gradient
            const bool unread = fuse && l == 1 && !wants_input_grad;
            Tensor gx;
            int gx_tiled = 1;
            if (l > 0) {
                if (!first && !unread) gx = tiled_array(d.B, d.I);
            } else {
                gx_tiled = st->patches;
                if (wants_input_grad) gx = gx_tiled ? tiled_array(d.B, d.I) : floats({d.B, d.I}, like);
            }
            if (have_tables[l] && !gx.defined() && !first && !unread) {  // nothing left to compute for this layer
                g = Tensor();
                continue;
            }
            if (!have_tables[l]) grads[l] = at::empty_like(luts[l]);
            const Tensor own_grad = have_tables[l] ? Tensor() : grads[l];
            const bool headed = l == n - 1 && st->groups;
            const int groups = headed ? (int)st->groups : 1;
            const float tau = headed ? (float)st->tau : 1.0f;
            if (nodes) {  // every node's own alpha and beta
                const Tensor alpha_n = per_node(st->per_node[l][0], d.N, like), beta_n = per_node(st->per_node[l][1], d.N, like);
                if (fuse) {
                    grads[l - 1] = at::empty_like(luts[l - 1]);
                    have_tables[l - 1] = true;
                }
                if (first) {
                    const Dims &f = st->dims[0];
                    const Plan &fp = st->plans[0];
                    const Tensor first_alpha = per_node(st->per_node[0][0], f.N, like), first_beta = per_node(st->per_node[0][1], f.N, like);
                    const Tensor gfirst = tiled_array(d.B, f.I), ws = bytes(L.dl_dwn_bwd_first_workspace_bytes(DIMS(d), f.I), like);
                    check(L.dl_dwn_layer_bwd_chain_first(
                        raw(saved[l]), ints(p.inv_ptr), ints(p.inv_pos), in(luts[l]), in(g), headed ? 2 : tiled, groups, tau, in(alpha_n),
                        in(beta_n), beta_max, out(own_grad), raw(saved[0]), out(grads[0]), ints(fp.idx), ints(fp.inv_ptr),
                        ints(fp.inv_pos), in(luts[0]), in(first_alpha), in(first_beta), (float)st->scalars[0][1], f.I, out(gfirst),
                        raw(ws), ws.numel(), DIMS(d), stream()));
                    g = gfirst;
                    break;
                }
                const Tensor ws = bytes(fuse ? L.dl_dwn_bwd_fused_workspace_bytes(DIMS(d), k_prev) : L.dl_dwn_bwd_workspace_bytes(DIMS(d)), like);
                check(L.dl_dwn_layer_bwd_chain_fused(
                    raw(saved[l]), ints(p.inv_ptr), ints(p.inv_pos), in(luts[l]), in(g), headed ? 2 : tiled, groups, tau, in(alpha_n),
                    in(beta_n), beta_max, out(gx), gx_tiled, out(own_grad), fuse ? raw(saved[l - 1]) : nullptr, k_prev,
                    fuse ? out(grads[l - 1]) : nullptr, raw(ws), ws.numel(), DIMS(d), stream()));
            } else {
                const float alpha = (float)st->scalars[l][0];
                const Tensor ws = bytes(L.dl_dwn_bwd_workspace_bytes(DIMS(d)), like);
                if (headed)
                    check(L.dl_dwn_layer_bwd_groups(raw(saved[l]), ints(p.inv_ptr), ints(p.inv_pos), in(luts[l]), in(g), groups, tau, alpha,
                                                    beta_max, out(gx), gx_tiled, out(grads[l]), raw(ws), ws.numel(), DIMS(d), stream()));
                else
                    check(L.dl_dwn_layer_bwd_tiled(raw(saved[l]), ints(p.inv_ptr), ints(p.inv_pos), in(luts[l]), in(g), tiled, alpha,
                                                   beta_max, out(gx), gx_tiled, out(grads[l]), raw(ws), ws.numel(), DIMS(d), stream()));
            }
            g = gx;
            tiled = gx_tiled;
        }
        if (st->patches && g.defined()) {
            const auto &s = st->image;
            const auto &q = st->geom;
            const Tensor gimg = floats(s, like);
            check(L.dl_fold(in(g), 1, out(gimg), (int)s[0], (int)s[1], (int)s[2], (int)s[3], q[0], q[1], q[2], q[3], q[4], q[5], stream()));
            g = gimg;
        }
        variable_list result{g};
        result.insert(result.end(), grads.begin(), grads.end());
        result.insert(result.end(), 3, Tensor());
        return result;
    }
};

// ------------------------------------------------------------------ loss
struct CrossEntropy : torch::autograd::Function<CrossEntropy> {
    static Tensor forward(AutogradContext *ctx, const Tensor &logits_, const Tensor &labels_) {
        require_device(logits_);
        require_device(labels_);
        const Tensor logits = f32(logits_);
        TORCH_CHECK(logits.dim() == 2 && labels_.dim() == 1 && labels_.size(0) == logits.size(0),
                    "expected logits [B, C] and labels [B], got ", logits_.sizes(), " and ", labels_.sizes());
        const Tensor labels = labels_.to(at::kLong).contiguous();
        const int B = (int)logits.size(0), C = (int)logits.size(1);
        const Tensor loss = floats({}, logits), glogits = at::empty_like(logits), ws = bytes(L.dl_cross_entropy_workspace_bytes(B), logits);
        check(L.dl_cross_entropy(in(logits), (const long long *)labels.const_data_ptr<int64_t>(), out(loss), out(glogits), raw(ws), ws.numel(), B, C, stream()));
        ctx->save_for_backward({glogits});
        return loss;
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) { return {ctx->get_saved_variables()[0] * grads[0], Tensor()}; }
};

// ------------------------------------------------------------------ optimizer
// One step of dl_adam_step over tensors of one device; the caller has made sure they are contiguous fp32.
void adam_step(const std::vector<std::array<Tensor, 4>> &items, double lr, double beta1, double beta2, double eps, double weight_decay,
               int64_t step, bool maximize) {
    if (items.empty()) return;
    std::vector<void *> p, m, v;
    std::vector<const void *> g;
    std::vector<long long> numel;
    for (const auto &[param, grad, first, second] : items) {
        p.push_back(out(param)), g.push_back(in(grad)), m.push_back(out(first)), v.push_back(out(second));
        numel.push_back(param.numel());
    }
    const c10::DeviceGuard guard(items[0][0].device());
    check(L.dl_adam_step(p.data(), g.data(), m.data(), v.data(), numel.data(), (int)items.size(), (float)lr, (float)beta1, (float)beta2,
                         (float)eps, (float)weight_decay, (int)step, maximize, stream()));
}

// ------------------------------------------------------------------ Python side
// A mapping plan as (idx32, inv_ptr, inv_pos, I)
typedef std::tuple<Tensor, Tensor, Tensor, int64_t> PlanArgs;
Plan plan_of(const PlanArgs &a) {
    const auto &[idx, inv_ptr, inv_pos, I] = a;
    return {idx, inv_ptr, inv_pos, (int)idx.size(0), (int)idx.size(1), (int)I};
}
typedef std::optional<Tensor> Maybe;
Tensor tensor_of(const Maybe &t) { return t ? *t : Tensor(); }

Tensor dwn_layer(const Tensor &x, const Tensor &luts, const PlanArgs &plan, const Maybe &alpha_n, const Maybe &beta_n, double alpha, double beta) {
    Kept k;
    k.plan = plan_of(plan);
    k.alpha_n = tensor_of(alpha_n), k.beta_n = tensor_of(beta_n);
    k.alpha = (float)alpha, k.beta = (float)beta;
    return DwnLayer::apply(x, luts, (const Kept *)&k);
}
Tensor dwn_stable_layer(const Tensor &x, const Tensor &luts, const Tensor &scale, const PlanArgs &plan) {
    Kept k;
    k.plan = plan_of(plan);
    return DwnStableLayer::apply(x, luts, scale, (const Kept *)&k);
}
Tensor hybrid_layer(const Tensor &x, const Tensor &luts, const PlanArgs &plan, bool keep_tiles) {
    Kept k;
    k.plan = plan_of(plan);
    return HybridLayer::apply(x, luts, (const Kept *)&k, keep_tiles);
}
Tensor dwn_stable_raw_layer(const Tensor &x, const Tensor &w, const Tensor &scale, const PlanArgs &plan) {
    require_device(x);
    require_device(w);
    Kept k;
    k.plan = plan_of(plan);
    if (w.dim() == 3 && L.dl_dwn_bwd_reads_x(k.plan.N, k.plan.k, (int)w.size(1)) == 0) return DwnStableRaw::apply(x, w, scale, (const Kept *)&k);
    return DwnStableLayer::apply(x, TableSigmoid::apply(w), scale, (const Kept *)&k);
}
Tensor hybrid_raw_layer(const Tensor &x, const Tensor &w, const PlanArgs &plan, bool keep_tiles) {
    require_device(x);
    require_device(w);
    Kept k;
    k.plan = plan_of(plan);
    if (keep_tiles && x.dim() == 2 && w.dim() == 3 && k.plan.k <= DL_MAX_FAST_K &&
        L.dl_hybrid_saved_bytes((int)x.size(0), k.plan.I, k.plan.N, k.plan.k, (int)w.size(1)) > 256)
        return HybridRaw::apply(x, w, (const Kept *)&k);
    return HybridLayer::apply(x, TableSigmoid::apply(w), (const Kept *)&k, keep_tiles);
}
Tensor prob_layer(const Tensor &x, const Tensor &w, const PlanArgs &plan, bool ordered, const Maybe &T_n, double T) {
    Kept k;
    k.plan = plan_of(plan);
    k.ordered = ordered;
    k.alpha_n = tensor_of(T_n), k.alpha = (float)T;
    return ProbLayer::apply(x, w, (const Kept *)&k);
}
c10::intrusive_ptr<Stack> stack_of(const std::vector<PlanArgs> &plans, size_t layers, int64_t groups, double tau) {
    TORCH_CHECK(plans.size() == layers && layers > 0, plans.size(), " mappings for ", layers, " layers");
    auto st = c10::make_intrusive<Stack>();
    for (const auto &p : plans) st->plans.push_back(plan_of(p));
    st->groups = groups, st->tau = tau;
    return st;
}
Tensor dwn_stack(const Tensor &x, const std::vector<Tensor> &luts, const std::vector<PlanArgs> &plans,
                 const std::vector<std::tuple<Maybe, Maybe, double, double>> &scalars, const Maybe &thresholds,
                 const std::vector<int> &geom, const Maybe &flip, int64_t groups, double tau) {
    auto st = stack_of(plans, luts.size(), groups, tau);
    TORCH_CHECK(scalars.size() == luts.size(), scalars.size(), " pairs of scalars for ", luts.size(), " layers");
    for (const auto &[a_n, b_n, a, b] : scalars) {
        st->per_node.push_back({tensor_of(a_n), tensor_of(b_n)});
        st->scalars.push_back({a, b});
    }
    if (!geom.empty()) {
        TORCH_CHECK(geom.size() == 6, "the geometry of a patch matrix has six numbers");
        st->patches = true;
        std::copy(geom.begin(), geom.end(), st->geom.begin());
    }
    const Tensor thr = tensor_of(thresholds), mask = tensor_of(flip);
    return DwnStack::apply(x, at::TensorList(luts), &thr, &mask, st);
}
Tensor dwn_stack_eval(const Tensor &x_, const Maybe &thresholds, const std::vector<Tensor> &luts_, const std::vector<PlanArgs> &plans,
                      int64_t groups, double tau) {
    at::NoGradGuard no_grad;
    require_device(x_);
    const Tensor x = f32(x_);
    auto st = stack_of(plans, luts_.size(), groups, tau);
    const size_t n = luts_.size();
    int B = 0, width = 0, nbits = 1;
    Tensor planes, thr, y;
    if (first_by_rows(x, tensor_of(thresholds), luts_, st->plans[0], groups, false)) thr = as_it_comes(x, tensor_of(thresholds), B, width, nbits);
    else planes = first_planes(x, tensor_of(thresholds), Tensor(), *st, B, width);
    for (size_t l = 0; l < n; ++l) {
        require_device(luts_[l]);
        const Tensor lut = f32(luts_[l]);
        const Plan &p = st->plans[l];
        const Dims d = chain_dims(l, p, lut, B, width);
        const bool last = l + 1 == n, head = last && groups;
        Tensor next;
        if (head) y = floats({B, groups}, x);
        else if (last) y = floats({B, (int64_t)d.N * d.O}, x);
        else next = bytes(L.dl_dwn_planes_bytes(B, d.N * d.O), x);
        const bool first = !planes.defined();  // reads x itself
        if (first || ((head || !last) && L.dl_dwn_rows_pay(B, 0, 1, d.N, d.k, d.O, head ? (int)groups : 0, 0) == 1)) {
            check(L.dl_dwn_layer_rows(first ? in(x) : nullptr, first ? in(thr) : nullptr, nbits, raw(planes), ints(p.idx), in(lut),
                                           raw(next), head ? out(y) : nullptr, nullptr, DIMS(d), (int)groups, (float)tau, stream()));
        } else if (head) {
            const size_t need = L.dl_dwn_eval_groups_workspace_bytes(B, d.N, d.O, (int)groups);
            const Tensor ws = need ? bytes(need, x) : Tensor();
            check(L.dl_dwn_layer_eval_planes_groups(raw(planes), ints(p.idx), in(lut), out(y), raw(ws), need, DIMS(d), (int)groups,
                                                    (float)tau, stream()));
        } else {
            check(L.dl_dwn_layer_eval_planes(raw(planes), ints(p.idx), in(lut), out(y), raw(next), DIMS(d), stream()));
        }
        planes = next;
        width = d.N * d.O;
    }
    return y;
}

// Whether rows 0, n - 1 and `count` rows from `start` on (around the end) of a bank's nodes still hold the views the bank handed out:
// nodes[keys[row]]._buffers[name] is views[row].  In Python, 18 rows took 3.5 us a bank, two banks a call of a layer.
bool views_hold(const py::dict &nodes, const py::tuple &keys, const py::str &name, const py::list &views, Py_ssize_t start, Py_ssize_t count) {
    static PyObject *const buffers_name = PyUnicode_InternFromString("_buffers");
    const Py_ssize_t n = PyList_GET_SIZE(views.ptr());
    if (n == 0 || PyTuple_GET_SIZE(keys.ptr()) != n) return false;
    const auto holds = [&](Py_ssize_t row) {
        PyObject *node = PyDict_GetItemWithError(nodes.ptr(), PyTuple_GET_ITEM(keys.ptr(), row));
        if (!node) {
            if (PyErr_Occurred()) throw py::error_already_set();
            return false;
        }
        const py::object buffers = py::reinterpret_steal<py::object>(PyObject_GetAttr(node, buffers_name));
        if (!buffers) throw py::error_already_set();
        if (!PyDict_Check(buffers.ptr())) return false;
        PyObject *view = PyDict_GetItemWithError(buffers.ptr(), name.ptr());
        if (!view && PyErr_Occurred()) throw py::error_already_set();
        return view == PyList_GET_ITEM(views.ptr(), row);
    };
    if (!holds(0) || !holds(n - 1)) return false;
    for (Py_ssize_t i = 0; i < count; ++i)
        if (!holds((start + i) % n)) return false;
    return true;
}

}  // namespace

PYBIND11_MODULE(difflut_host, m) {
    const auto free_gil = py::call_guard<py::gil_scoped_release>();
    m.def("load", &load);
    m.def("views_hold", &views_hold);
    m.def("dwn_layer", &dwn_layer, free_gil);
    m.def("dwn_stable_layer", &dwn_stable_layer, free_gil);
    m.def("hybrid_layer", &hybrid_layer, free_gil);
    m.def("dwn_stable_raw_layer", &dwn_stable_raw_layer, free_gil);
    m.def("hybrid_raw_layer", &hybrid_raw_layer, free_gil);
    m.def("table_sigmoid", [](const Tensor &t) { return TableSigmoid::apply(t); }, free_gil);
    m.def("prob_layer", &prob_layer, free_gil);
    m.def("soft_map", [](const Tensor &x, const Tensor &W, double tau, int64_t precision) { return SoftMap::apply(x, W, tau, precision); },
          free_gil);
    m.def("dwn_stack", &dwn_stack, free_gil);
    m.def("dwn_stack_eval", &dwn_stack_eval, free_gil);
    m.def("adam_step", &adam_step);
    m.def("cross_entropy", [](const Tensor &logits, const Tensor &labels) { return CrossEntropy::apply(logits, labels); }, free_gil);
}
