// Autograd nodes of the attention modules, compiled against libtorch (host code only).
//
// It does what _BlockAttnFunction in attention_blockcuda.py does -- the reference's function is
// models/attention_blockcuda.py:20-112 (key-mask variant: models/attention_blockcuda_mask.py) -- with the node, the
// saved tensors and the output allocations on the C++ side of PyTorch: for small problems (the reference's L = 1024
// tasks) a training step is bound by the host, and the Python function spends about three times the kernels' run
// time between autograd's engine, ctypes and tensor bookkeeping.  The arithmetic is the library's: the row-major
// and strided entry points declared in include/spion_hip.h.  The Python function stays the statement of the
// behaviour; tests run both and compare.
#include <ATen/FuncTorchTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/extension.h>

#include <stdexcept>
#include <string>

#include "../../include/spion_hip.h"

namespace {

using torch::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

void check_library(const char* where) {
    if (!spion_error_pending()) return;
    std::string text = spion_last_error();
    spion_clear_error();
    throw std::runtime_error(std::string(where) + ": " + text);
}

// Layout of a [B, H, L, d] view for the strided entry points; false when they cannot take it (last dimension not
// unit-stride, strides not multiples of 16 bytes, storage not 16-byte aligned).
bool head_layout(const Tensor& t, spion_head_layout& lay) {
    if (t.dim() != 4) return false;
    const int64_t sb = t.stride(0), sh = t.stride(1), sl = t.stride(2), sf = t.stride(3);
    if (sf != 1 || reinterpret_cast<uintptr_t>(t.data_ptr()) % 16) return false;
    const int64_t unit = 16 / t.element_size();
    if (sb % unit || sh % unit || sl % unit || sl < t.size(3) || sb < 0 || sh < 0) return false;
    if (t.size(2) * sl >= (int64_t(1) << 29)) return false;
    lay.batch_stride = sb;
    lay.head_stride = (int)sh;
    lay.row_stride = (int)sl;
    return true;
}

Tensor empty_heads(c10::IntArrayRef shape, bool interleaved, const torch::TensorOptions& opt) {
    if (!interleaved) return torch::empty(shape, opt);
    return torch::empty({shape[0], shape[2], shape[1], shape[3]}, opt).transpose(1, 2);  // memory [B, L, H, d]
}

bool same_strides(const Tensor& a, const Tensor& b) { return a.strides() == b.strides(); }

// q, k, v are the three slices of one [B, L, 3, H, d] buffer, in this order
bool adjacent_head_views(const Tensor& q, const Tensor& k, const Tensor& v) {
    const int64_t H = q.size(1), L = q.size(2), d = q.size(3);
    const int64_t want[4] = {L * 3 * H * d, d, 3 * H * d, 1};
    for (const Tensor* t : {&q, &k, &v})
        for (int i = 0; i < 4; ++i)
            if (t->stride(i) != want[i]) return false;
    const char *pq = (const char*)q.data_ptr(), *pk = (const char*)k.data_ptr(), *pv = (const char*)v.data_ptr();
    const int64_t step = H * d * 4;
    return pk - pq == step && pv - pk == step;
}

const float* fp(const Tensor& t) { return t.defined() ? static_cast<const float*>(t.data_ptr()) : nullptr; }
float* fpm(Tensor& t) { return static_cast<float*>(t.data_ptr()); }
const int* ip(const Tensor& t) { return static_cast<const int*>(t.data_ptr()); }

// Whether a call needs no node: nothing is recorded for a backward, no input carries a forward-mode tangent (which does
// not depend on grad mode, and which a node refuses instead of dropping it) and no functorch transform is at work.
bool has_tangent(const Tensor& t) { return t.defined() && t._fw_grad(/*level=*/0).defined(); }
bool without_node(std::initializer_list<const Tensor*> inputs) {
    if (torch::GradMode::is_enabled() || at::functorch::functorchTLSAccessor()) return false;
    for (const Tensor* t : inputs)
        if (has_tangent(*t)) return false;
    return true;
}

// The stream a backward is launched on: the calling thread's, which the tensors it makes belong to as well.  The engine puts
// a node's backward on the stream of its forward; compiled autograd, and a caller of the node itself, do not.
int64_t current_stream(int64_t device) {
    return reinterpret_cast<int64_t>(c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(device)).stream());
}

// What a node keeps of the handle its backward works on, which a program may destroy before, for instance with the module
// it is tied to.  (The module itself is not held: Python's collector does not see what a compiled node refers to, and a
// module that keeps its own output would never be freed.)
// It is a tensor without elements whose storage lets go: compiled autograd takes no other object along with a node.
void keep_handle(AutogradContext* ctx, int64_t handle) {
    void* h = reinterpret_cast<void*>(handle);
    ctx->saved_data["handle"] = handle;
    if (spion_hold(h)) check_library("attn_forward");
    c10::Storage hold(c10::Storage::use_byte_size_t(), 0, c10::DataPtr(h, h, &spion_release, c10::Device(c10::kCPU)));
    ctx->saved_data["hold"] = at::detail::make_tensor<c10::TensorImpl>(
        std::move(hold), c10::DispatchKeySet(c10::DispatchKey::CPU), caffe2::TypeMeta::Make<uint8_t>());
}

// The index tensors are kept beside the saved tensors, out of the reach of saved-tensor hooks: the library knows an index by
// its address, and one that a hook brings back somewhere else would be analysed anew (a wait for the stream, and an error
// under capture) and stay on file for whatever index lies there next.
void keep_index(AutogradContext* ctx, const Tensor& offsets, const Tensor& columns, const Tensor& sum_mat) {
    ctx->saved_data["offsets"] = offsets;
    ctx->saved_data["columns"] = columns;
    ctx->saved_data["sum_mat"] = sum_mat;
}

// The layout of heads the strided entry points have to take: contiguous ones may start off 16 bytes, and saved-tensor hooks
// may have put saved ones somewhere else.
void taken_layout(const Tensor& t, spion_head_layout& lay) {
    TORCH_CHECK_TYPE(t.is_cuda() && head_layout(t, lay), "heads on the GPU, 16-byte aligned, expected");
}

// Saved tensors as the backward finds them: hooks may bring any of them back as something else, while the kernels take types
// and sizes as they were saved and one layout for q, k and v.  Other strides are put right; another device or type, or fewer
// values, are refused.
void keep_sizes(AutogradContext* ctx, const Tensor& q) {
    ctx->saved_data["sizes"] =
        std::vector<int64_t>{q.size(0), q.size(1), q.size(2), q.size(3), static_cast<int64_t>(q.device().index())};
}
struct SavedTensors {
    const std::vector<int64_t> sizes;
    const variable_list saved;
    explicit SavedTensors(AutogradContext* ctx)
        : sizes(ctx->saved_data["sizes"].toIntVector()), saved(ctx->get_saved_variables()) {}
    const Tensor& checked(size_t i, at::ScalarType type) const {
        const Tensor& t = saved.at(i);
        TORCH_CHECK_TYPE(t.defined() && t.is_cuda() && t.device().index() == sizes[4] && t.scalar_type() == type,
                         "saved tensors of the device and type they were saved with expected");
        return t;
    }
    Tensor heads(size_t i, at::ScalarType type) const {
        const Tensor& t = checked(i, type);
        TORCH_CHECK_TYPE(t.sizes() == c10::IntArrayRef(sizes.data(), 4), "saved heads of the size they were saved with expected");
        spion_head_layout lay{};
        return head_layout(t, lay) ? t : t.contiguous();
    }
    // the saved tensors 0 to 2, in one layout
    void inputs(at::ScalarType type, Tensor& q, Tensor& k, Tensor& v) const {
        q = heads(0, type);
        k = heads(1, type);
        v = heads(2, type);
        if (same_strides(k, q) && same_strides(v, q)) return;
        q = q.contiguous();
        k = k.contiguous();
        v = v.contiguous();
    }
    // fp32 values, `per_head` for each of the heads
    Tensor values(size_t i, int64_t per_head) const {
        const Tensor& t = checked(i, torch::kFloat32);
        TORCH_CHECK_TYPE(t.numel() >= sizes[0] * sizes[1] * per_head, "saved values as many as were saved expected");
        return t.contiguous();
    }
};

// What a forward of the attention core leaves for its backward.
struct CoreResult {
    Tensor q, k, v, out, p_flat;
    bool strided = false;
};

// Scratch of a call of the core, of its stream as every tensor made here is.  Where there is no memory for it, the `least` floats
// that the element kernels, or the handle's workspaces, do with.
Tensor core_scratch(void* h, const Tensor& offsets, const Tensor& columns, int64_t nnz, bool backward, int64_t least,
                    const torch::TensorOptions& opt) {
    const int64_t floats = spion_attn_scratch(h, ip(offsets), ip(columns), (int)nnz, backward);
    if (floats < 0) check_library(backward ? "attn_backward" : "attn_forward");
    if (floats <= least) return floats > 0 ? torch::empty({floats}, opt) : Tensor();
    try {
        return torch::empty({floats}, opt);
    } catch (const c10::OutOfMemoryError&) {
        return least > 0 ? torch::empty({least}, opt) : Tensor();
    }
}
float* fps(Tensor& t) { return t.defined() ? fpm(t) : nullptr; }
int64_t count(const Tensor& t) { return t.defined() ? t.numel() : 0; }

// pen: penalties [B, H*L] (mask_heads 0), a key mask [B, L] of mask_heads heads a sample, or nothing.
CoreResult core_forward(const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& pen, int64_t mask_heads,
                        const Tensor& offsets, const Tensor& columns, const Tensor& sum_mat, int64_t handle, int64_t nnz,
                        int64_t num_heads, bool reads_views, int64_t stream) {
    void* h = reinterpret_cast<void*>(handle);
    spion_set_stream(h, reinterpret_cast<void*>(stream));
    TORCH_CHECK(query.dim() == 4 && key.sizes() == query.sizes() && value.sizes() == query.sizes(),
                "query, key and value must be [B, H, L, d] tensors of one shape");
    const int64_t B = query.size(0), H = query.size(1);
    // the kernels take every size from the handle: tensors of other sizes would be read and written past their ends
    int hd = 0, hl = 0, hnb = 0;
    if (spion_block_sizes(h, &hd, &hl, &hnb)) check_library("attn_forward");
    TORCH_CHECK_VALUE(B * H == hnb && H == num_heads && query.size(2) == hl && query.size(3) == hd, "query shape ",
                      query.sizes(), " does not match the handle (", hnb, " heads in all, ", num_heads, " a sample, ", hl,
                      " rows of ", hd, ")");
    TORCH_CHECK_VALUE(!pen.defined() || (mask_heads ? mask_heads == H && pen.numel() >= B * query.size(2)
                                                    : pen.numel() >= B * H * query.size(2)),
                      "key mask smaller than [B, L]");
    for (const Tensor* t : {&query, &key, &value, &pen})
        TORCH_CHECK(!t->defined() || (t->scalar_type() == torch::kFloat32 && t->device() == query.device() && t->is_cuda()),
                    "fp32 tensors on one GPU expected");
    const auto opt = query.options();
    CoreResult r;
    r.p_flat = torch::empty({B * H * nnz}, opt);
    Tensor scratch = core_scratch(h, offsets, columns, nnz, false, 0, opt);
    spion_head_layout lin{}, lout{}, lk{}, lv{};
    r.strided = reads_views && !(query.is_contiguous() && key.is_contiguous() && value.is_contiguous()) &&
                head_layout(query, lin) && head_layout(key, lk) && head_layout(value, lv) && same_strides(key, query) &&
                same_strides(value, query);
    r.q = r.strided ? query : query.contiguous();
    r.k = r.strided ? key : key.contiguous();
    r.v = r.strided ? value : value.contiguous();
    if (r.strided) {
        r.out = empty_heads(query.sizes(), query.stride(1) < query.stride(2), opt);
        head_layout(r.out, lout);
    } else {
        r.out = torch::empty(query.sizes(), opt);
    }
    spion_attn_forward_scratch(h, fp(r.q), fp(r.k), fp(r.v), fp(pen), (int)mask_heads, fpm(r.p_flat), fpm(r.out), ip(offsets),
                               ip(columns), (int)nnz, (int)num_heads, r.strided ? &lin : nullptr, r.strided ? &lout : nullptr,
                               fps(scratch), count(scratch));
    check_library("attn_forward");
    return r;
}

struct SparseAttnNode : public torch::autograd::Function<SparseAttnNode> {
    // pen_opt, mask_heads: key penalties or the key mask of the key-mask modules, or nothing (core_forward).  stream: torch's current raw stream at the
    // call.  fixed: takes what carries no gradient, the probabilities of the key-mask modules (compiled autograd refuses
    // nodes with outputs that are marked so).
    static variable_list forward(AutogradContext* ctx, Tensor query, Tensor key, Tensor value,
                                 c10::optional<Tensor> pen_opt, int64_t mask_heads, Tensor offsets, Tensor columns,
                                 Tensor sum_mat, int64_t handle, int64_t nnz, int64_t num_heads, bool reads_views, int64_t stream, Tensor* fixed) {
        const Tensor pen = pen_opt.has_value() ? *pen_opt : Tensor();
        CoreResult r = core_forward(query, key, value, pen, mask_heads, offsets, columns, sum_mat, handle, nnz, num_heads,
                                    reads_views, stream);
        keep_handle(ctx, handle);
        ctx->saved_data["nnz"] = nnz;
        ctx->saved_data["heads"] = num_heads;
        ctx->saved_data["strided"] = r.strided;
        keep_index(ctx, offsets, columns, sum_mat);
        keep_sizes(ctx, r.q);
        ctx->save_for_backward({r.q, r.k, r.v, r.p_flat, r.out});
        ctx->set_materialize_grads(false);  // the gradient of the returned probabilities is ignored anyway
        if (!pen.defined()) return {r.out, r.p_flat};
        *fixed = r.p_flat;
        return {r.out};
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const Tensor &offsets = ctx->saved_data["offsets"].toTensor(), &columns = ctx->saved_data["columns"].toTensor(),
                     &sum_mat = ctx->saved_data["sum_mat"].toTensor();
        void* h = reinterpret_cast<void*>(ctx->saved_data["handle"].toInt());
        const int64_t nnz = ctx->saved_data["nnz"].toInt();
        const SavedTensors saved(ctx);
        Tensor q, k, v, out = saved.heads(4, torch::kFloat32);
        saved.inputs(torch::kFloat32, q, k, v);
        const Tensor p_flat = saved.values(3, nnz);
        const int heads = (int)ctx->saved_data["heads"].toInt();
        spion_set_stream(h, reinterpret_cast<void*>(current_stream(q.device().index())));
        const auto opt = q.options();
        Tensor go = grads[0];
        if (!go.defined()) go = torch::zeros(q.sizes(), opt);  // only the probabilities were used downstream
        Tensor dq, dk, dv;
        const bool strided = ctx->saved_data["strided"].toBool();
        spion_head_layout lin{}, lout{}, lgrad{};
        if (strided) {
            spion_head_layout lgo{};
            if (!same_strides(go, out) || !head_layout(go, lgo)) go = torch::empty_like(out).copy_(go);  // out's strides
            if (adjacent_head_views(q, k, v)) {  // slices of one fused projection: the gradients likewise
                Tensor buf = torch::empty({q.size(0), q.size(2), 3, q.size(1), q.size(3)}, opt);
                dq = buf.select(2, 0).transpose(1, 2);
                dk = buf.select(2, 1).transpose(1, 2);
                dv = buf.select(2, 2).transpose(1, 2);
            } else {
                const bool inter = q.stride(1) < q.stride(2);
                dq = empty_heads(q.sizes(), inter, opt);
                dk = empty_heads(q.sizes(), inter, opt);
                dv = empty_heads(q.sizes(), inter, opt);
            }
            taken_layout(q, lin);
            taken_layout(out, lout);
            head_layout(dq, lgrad);
        } else {
            q = q.contiguous();
            k = k.contiguous();
            v = v.contiguous();
            out = out.contiguous();
            go = go.contiguous();
            dq = torch::empty(q.sizes(), opt);
            dk = torch::empty(q.sizes(), opt);
            dv = torch::empty(q.sizes(), opt);
        }
        // (in place of the ABI's two [NB*nnz] scratch arguments, models/attention_blockcuda.py:83-84)
        Tensor scratch = core_scratch(h, offsets, columns, nnz, true, std::max<int64_t>(q.size(0) * q.size(1) * nnz, 1), opt);
        spion_attn_backward_scratch(h, fp(q), fp(k), fp(v), fp(p_flat), fp(out), fp(go), fpm(dq), fpm(dk), fpm(dv), ip(offsets),
                                    ip(columns), (int)nnz, heads, strided ? &lin : nullptr, strided ? &lout : nullptr,
                                    strided ? &lgrad : nullptr, fps(scratch), count(scratch));
        check_library("attn_backward");
        variable_list r(14);
        r[0] = dq;
        r[1] = dk;
        r[2] = dv;
        return r;
    }
};

// 1e6 * (1 - mask) per head, [B, H*L], from a [B, L] fp32 key mask (models/attention_blockcuda_mask.py:42-43).
Tensor key_penalty(const Tensor& mask, int64_t heads, int64_t stream) {
    Tensor pen = torch::empty({mask.size(0), heads * mask.size(1)}, mask.options());
    spion_key_penalty(fp(mask), fpm(pen), (int)mask.size(0), (int)heads, (int)mask.size(1), reinterpret_cast<void*>(stream));
    check_library("attn_forward");
    return pen;
}
// The modules hand over a key mask, or penalties made from one the kernels do not take (is_mask = false); either has to lie on
// the device of the heads.  Where the forward's kernels alone need it, they read a mask of the heads' sizes themselves.
struct KeyOperand {
    c10::optional<Tensor> t;
    int64_t mask_heads = 0;  // 0: penalties
    Tensor or_none() const { return t.has_value() ? *t : Tensor(); }
};
c10::optional<Tensor> penalty_of(const c10::optional<Tensor>& mask_or_pen, bool is_mask, int64_t heads, c10::Device device,
                                 int64_t stream) {
    TORCH_CHECK(!mask_or_pen.has_value() || mask_or_pen->device() == device, "fp32 tensors on one GPU expected");
    if (!is_mask || !mask_or_pen.has_value()) return mask_or_pen;
    if (has_tangent(*mask_or_pen)) return (1e6 * (1.0 - mask_or_pen->repeat({1, heads}))).contiguous();
    return key_penalty(*mask_or_pen, heads, stream);
}

KeyOperand key_operand(const c10::optional<Tensor>& mask_or_pen, bool is_mask, int64_t batch, int64_t heads, int64_t length,
                       c10::Device device, int64_t stream) {
    if (is_mask && mask_or_pen.has_value() && !has_tangent(*mask_or_pen)) {
        const Tensor& m = *mask_or_pen;
        if (m.device() == device && m.is_cuda() && m.scalar_type() == torch::kFloat32 && m.dim() == 2 && m.size(0) == batch &&
            m.size(1) == length && m.is_contiguous() && !m.requires_grad() && reinterpret_cast<uintptr_t>(m.data_ptr()) % 16 == 0)
            return {mask_or_pen, heads};
    }
    return {penalty_of(mask_or_pen, is_mask, heads, device, stream), 0};
}

// The gradient of a core's output in that output's strides, as the strided entry points take it.
Tensor grad_like(const Tensor& go, const Tensor& out) {
    spion_head_layout lay{};
    if (go.scalar_type() == out.scalar_type() && same_strides(go, out) && head_layout(go, lay)) return go;
    return torch::empty_like(out).copy_(go);
}

// ---- the dense phase: what _DenseAttnFunction in attention_cuda.py does through the strided entry points ----------
struct DenseResult {
    Tensor q, k, v, attn, out, mean;  // attn: memory [key][query]
};
DenseResult dense_forward(const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& pen, int64_t mask_heads,
                          int64_t handle, bool emit_mean, int64_t stream) {
    void* h = reinterpret_cast<void*>(handle);
    spion_set_stream(h, reinterpret_cast<void*>(stream));
    const auto opt = query.options();
    const int64_t B = query.size(0), H = query.size(1), L = query.size(2);
    DenseResult r;
    spion_head_layout lin{}, lk{}, lv{}, lout{};
    const bool views = head_layout(query, lin) && head_layout(key, lk) && head_layout(value, lv) && same_strides(key, query) &&
                       same_strides(value, query);
    r.q = views ? query : query.contiguous();
    r.k = views ? key : key.contiguous();
    r.v = views ? value : value.contiguous();
    taken_layout(r.q, lin);
    r.attn = torch::empty({B, H, L, L}, opt);
    r.out = empty_heads(query.sizes(), r.q.stride(1) < r.q.stride(2), opt);
    head_layout(r.out, lout);
    if (emit_mean) r.mean = torch::empty({L, L}, opt);
    if (mask_heads) {
        spion_dense_forward_strided_keys(h, fp(r.q), fp(r.k), fp(r.v), fp(pen), fpm(r.attn), fpm(r.out),
                                         emit_mean ? fpm(r.mean) : nullptr, (int)H, &lin, &lout);
    } else if (emit_mean) {
        spion_dense_forward_strided_mean(h, fp(r.q), fp(r.k), fp(r.v), fp(pen), fpm(r.attn), fpm(r.out), fpm(r.mean), (int)H,
                                         &lin, &lout);
    } else {
        spion_dense_forward_strided(h, fp(r.q), fp(r.k), fp(r.v), fp(pen), fpm(r.attn), fpm(r.out), (int)H, &lin, &lout);
    }
    check_library("attn_forward");
    return r;
}
struct DenseAttnNode : public torch::autograd::Function<DenseAttnNode> {
    static variable_list forward(AutogradContext* ctx, Tensor query, Tensor key, Tensor value, c10::optional<Tensor> pen,
                                 int64_t mask_heads, int64_t handle, bool emit_mean, int64_t stream, Tensor* mean) {
        DenseResult r = dense_forward(query, key, value, pen.has_value() ? *pen : Tensor(), mask_heads, handle, emit_mean, stream);
        keep_handle(ctx, handle);
        keep_sizes(ctx, r.q);
        ctx->save_for_backward({r.q, r.k, r.v, r.attn, r.out});
        ctx->set_materialize_grads(false);  // the gradient of the returned map is ignored (as in the reference)
        *mean = r.mean;  // (no output of the node: it carries no gradient, see SparseAttnNode)
        return {r.out, r.attn.transpose(2, 3)};
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const SavedTensors saved(ctx);
        Tensor q, k, v;
        saved.inputs(torch::kFloat32, q, k, v);
        const Tensor attn = saved.values(3, q.size(2) * q.size(2)), out = saved.heads(4, torch::kFloat32);
        void* h = reinterpret_cast<void*>(ctx->saved_data["handle"].toInt());
        spion_set_stream(h, reinterpret_cast<void*>(current_stream(q.device().index())));
        const auto opt = q.options();
        const Tensor go = grads[0].defined() ? grad_like(grads[0], out) : torch::zeros_like(out);
        Tensor dq, dk, dv;
        if (adjacent_head_views(q, k, v)) {  // slices of one fused projection: the gradients likewise
            Tensor buf = torch::empty({q.size(0), q.size(2), 3, q.size(1), q.size(3)}, opt);
            dq = buf.select(2, 0).transpose(1, 2);
            dk = buf.select(2, 1).transpose(1, 2);
            dv = buf.select(2, 2).transpose(1, 2);
        } else {
            const bool inter = q.stride(1) < q.stride(2);
            dq = empty_heads(q.sizes(), inter, opt);
            dk = empty_heads(q.sizes(), inter, opt);
            dv = empty_heads(q.sizes(), inter, opt);
        }
        spion_head_layout lin{}, lout{}, lgrad{};
        taken_layout(q, lin);
        taken_layout(out, lout);
        head_layout(dq, lgrad);
        Tensor scratch;
        try {
            if (const int64_t floats = spion_dense_scratch(h); floats > 0) scratch = torch::empty({floats}, opt);
        } catch (const c10::OutOfMemoryError&) {  // the call does without
        }
        spion_dense_backward_scratch(h, fp(q), fp(k), fp(v), fp(attn), fp(out), fp(go), fpm(dq), fpm(dk), fpm(dv), (int)q.size(1),
                                     &lin, &lout, &lgrad, fps(scratch), count(scratch));
        check_library("attn_backward");
        return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ---- bf16: what _BlockBF16Function in attention_blockbf16.py does -----------------------------------------------
struct BF16Result {
    Tensor q, k, v, out, lse;
    bool strided = false;
};
const void* vp(const Tensor& t) { return t.data_ptr(); }
BF16Result bf16_forward(const Tensor& query, const Tensor& key, const Tensor& value, const Tensor& pen, int64_t mask_heads,
                        const Tensor& offsets, const Tensor& columns, const Tensor& sum_mat, int64_t handle, int64_t nnz, int64_t stream) {
    void* h = reinterpret_cast<void*>(handle);
    spion_set_stream(h, reinterpret_cast<void*>(stream));
    const auto opt = query.options().dtype(torch::kBFloat16);
    const int64_t B = query.size(0), H = query.size(1), L = query.size(2);
    BF16Result r;
    r.lse = torch::empty({B * H, L}, query.options().dtype(torch::kFloat32));
    // bf16 heads that are views of projections are read in place and the output is interleaved the same way; anything
    // else is converted and made contiguous first
    spion_head_layout lin{}, lk{}, lv{}, lout{};
    bool all = true;
    for (const Tensor* t : {&query, &key, &value}) all = all && t->scalar_type() == torch::kBFloat16;
    r.strided = all && !(query.is_contiguous() && key.is_contiguous() && value.is_contiguous()) && head_layout(query, lin) &&
                head_layout(key, lk) && head_layout(value, lv) && same_strides(key, query) && same_strides(value, query);
    if (r.strided) {
        r.q = query;
        r.k = key;
        r.v = value;
        r.out = empty_heads(query.sizes(), query.stride(1) < query.stride(2), opt);
        head_layout(r.out, lout);
        (mask_heads ? spion_block_bf16_attn_forward_strided_keys : spion_block_bf16_attn_forward_strided)(
            h, vp(r.q), vp(r.k), vp(r.v), fp(pen), r.out.data_ptr(), fpm(r.lse), ip(offsets), ip(columns), ip(sum_mat), (int)nnz,
            (int)H, &lin, &lout);
    } else {
        r.q = query.to(torch::kBFloat16).contiguous();
        r.k = key.to(torch::kBFloat16).contiguous();
        r.v = value.to(torch::kBFloat16).contiguous();
        r.out = torch::empty(query.sizes(), opt);
        if (mask_heads)
            spion_block_bf16_attn_forward_keys(h, vp(r.q), vp(r.k), vp(r.v), fp(pen), (int)mask_heads, r.out.data_ptr(), fpm(r.lse),
                                               ip(offsets), ip(columns), ip(sum_mat), (int)nnz);
        else
            spion_block_bf16_attn_forward(h, vp(r.q), vp(r.k), vp(r.v), fp(pen), r.out.data_ptr(), fpm(r.lse), ip(offsets),
                                          ip(columns), ip(sum_mat), (int)nnz);
    }
    check_library("spion_block_bf16_attn_forward");
    return r;
}
struct BF16AttnNode : public torch::autograd::Function<BF16AttnNode> {
    static Tensor forward(AutogradContext* ctx, Tensor query, Tensor key, Tensor value, c10::optional<Tensor> pen_opt,
                          Tensor offsets, Tensor columns, Tensor sum_mat, int64_t handle, int64_t nnz, int64_t stream) {
        const Tensor pen = pen_opt.has_value() ? *pen_opt : Tensor();
        const BF16Result r = bf16_forward(query, key, value, pen, 0, offsets, columns, sum_mat, handle, nnz, stream);
        keep_handle(ctx, handle);
        ctx->saved_data["nnz"] = nnz;
        ctx->saved_data["strided"] = r.strided;
        keep_index(ctx, offsets, columns, sum_mat);
        keep_sizes(ctx, r.q);
        ctx->save_for_backward({r.q, r.k, r.v, r.out, r.lse, pen});
        return r.out;
    }
    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        const Tensor &offsets = ctx->saved_data["offsets"].toTensor(), &columns = ctx->saved_data["columns"].toTensor(),
                     &sum_mat = ctx->saved_data["sum_mat"].toTensor();
        const SavedTensors saved(ctx);
        Tensor q, k, v, out = saved.heads(3, torch::kBFloat16);
        saved.inputs(torch::kBFloat16, q, k, v);
        const Tensor lse = saved.values(4, q.size(2)), pen = saved.saved[5].defined() ? saved.values(5, q.size(2)) : Tensor();
        void* h = reinterpret_cast<void*>(ctx->saved_data["handle"].toInt());
        const int nnz = (int)ctx->saved_data["nnz"].toInt();
        spion_set_stream(h, reinterpret_cast<void*>(current_stream(q.device().index())));
        Tensor dq, dk, dv;
        if (ctx->saved_data["strided"].toBool()) {
            const Tensor go = grad_like(grads[0], out);
            const bool inter = q.stride(1) < q.stride(2);
            dq = empty_heads(q.sizes(), inter, q.options());
            dk = empty_heads(q.sizes(), inter, q.options());
            dv = empty_heads(q.sizes(), inter, q.options());
            spion_head_layout lin{}, lout{}, lgrad{};
            taken_layout(q, lin);
            taken_layout(out, lout);
            head_layout(dq, lgrad);
            spion_block_bf16_attn_backward_strided(h, vp(q), vp(k), vp(v), fp(pen), vp(out), fp(lse), vp(go), dq.data_ptr(),
                                                   dk.data_ptr(), dv.data_ptr(), ip(offsets), ip(columns), ip(sum_mat), nnz,
                                                   (int)q.size(1), &lin, &lout, &lgrad);
        } else {
            q = q.contiguous();
            k = k.contiguous();
            v = v.contiguous();
            out = out.contiguous();
            const Tensor go = grads[0].to(torch::kBFloat16).contiguous();
            dq = torch::empty_like(q);
            dk = torch::empty_like(q);
            dv = torch::empty_like(q);
            spion_block_bf16_attn_backward(h, vp(q), vp(k), vp(v), fp(pen), vp(out), fp(lse), vp(go), dq.data_ptr(),
                                           dk.data_ptr(), dv.data_ptr(), ip(offsets), ip(columns), ip(sum_mat), nnz);
        }
        check_library("spion_block_bf16_attn_backward");
        return {dq, dk, dv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
    }
};

// ---- the projections of models/attention.py:84-103 on the library's own kernels ------------------
Tensor aligned(const Tensor& t) {  // contiguous, 16-byte aligned
    Tensor c = t.contiguous();
    return reinterpret_cast<uintptr_t>(c.data_ptr()) % 16 ? c.clone() : c;
}

// y = x.w^T + b: w [outputs, features], b [outputs], fp32 tensors with memory of their own on x's device.  The kernels
// take the sizes of all of them from x and the heads, so anything else would be read past its end.
bool projection_fits(const Tensor& x, const Tensor& w, const Tensor& b, int64_t outputs, int64_t features) {
    for (const Tensor* t : {&x, &w, &b})
        if (!t->defined() || t->scalar_type() != torch::kFloat32 || t->device() != x.device() ||
            t->layout() != torch::kStrided || t->unsafeGetTensorImpl()->is_python_dispatch())
            return false;
    return w.dim() == 2 && w.size(0) == outputs && w.size(1) == features && b.dim() == 1 && b.size(0) == outputs;
}
void check_projection(const Tensor& x, const Tensor& w, const Tensor& b, int64_t outputs, int64_t features) {
    TORCH_CHECK_VALUE(projection_fits(x, w, b, outputs, features), "projection: weight [", outputs, ", ", features,
                      "] and bias [", outputs, "], fp32 on the input's device, expected");
}
// Whether the projection kernels take this layer's four linear layers as they are; the layer uses torch's otherwise.
bool projections_fit(const Tensor& x, const Tensor& wq, const Tensor& wk, const Tensor& wv, const Tensor& bq, const Tensor& bk,
                     const Tensor& bv, const Tensor& wf, const Tensor& bf, int64_t H, int64_t d) {
    if (x.dim() != 3 || !wf.defined() || wf.dim() != 2) return false;
    const int64_t n = H * d, dim = x.size(2), outputs = wf.size(0), rows = x.size(0) * x.size(1);
    for (const int64_t size : {n, dim, outputs, rows})
        if (size <= 0 || size % 32) return false;
    if (rows >= 1 << 30 || std::max(3 * n, outputs) > 1 << 20 || std::max(3 * n * dim, outputs * n) > 1 << 30) return false;
    return projection_fits(x, wq, bq, n, dim) && projection_fits(x, wk, bk, n, dim) && projection_fits(x, wv, bv, n, dim) &&
           projection_fits(x, wf, bf, outputs, n);
}

// What a backward of `segs` projections of x to n outputs each is asked for: the gradients of x, in its memory layout, and of
// weights and biases together.
struct ProjectionGrads {
    Tensor dx, dw, db;
};
ProjectionGrads project_backward(const float* dy, const Tensor* w, const Tensor& x, int64_t rows, int64_t n, int segs, int64_t dim,
                                 int64_t stream, bool input, bool weights) {
    const auto opt = x.options();
    const int64_t outputs = segs * n;
    void* s = reinterpret_cast<void*>(stream);
    ProjectionGrads r;
    const float* wp[3] = {};
    if (input) {
        r.dx = torch::empty_like(x);
        for (int i = 0; i < segs; ++i) wp[i] = fp(w[i]);
    }
    Tensor ws;
    if (weights) {
        r.dw = torch::empty({outputs, dim}, opt);
        ws = torch::empty({spion_project_workspace(rows, (int)outputs, (int)dim)}, opt);
        r.db = torch::empty({outputs}, opt);
    }
    if (input && weights)
        spion_project_backward(dy, wp, fp(x), fpm(r.dx), fpm(r.dw), fpm(r.db), fpm(ws), rows, (int)n, segs, (int)dim, s);
    else if (input)
        spion_project_backward_input(dy, wp, fpm(r.dx), rows, (int)n, segs, (int)dim, s);
    else if (weights)
        spion_project_backward_weight(dy, fp(x), fpm(r.dw), fpm(r.db), fpm(ws), rows, (int)outputs, (int)dim, s);
    check_library("projection");
    return r;
}

// What the nodes below saved, as hooks bring it back: the kernels take sizes from what was saved.
const Tensor& saved_as(const Tensor& t, c10::IntArrayRef sizes, int64_t device) {
    TORCH_CHECK_TYPE(t.defined() && t.is_cuda() && t.device().index() == device && t.scalar_type() == torch::kFloat32 &&
                         t.sizes() == sizes,
                     "saved tensors of the device, type and size they were saved with expected");
    return t;
}

// X [B, L, dim] -> the [B, H, L, d] heads of the three projections, slices of one [B, L, 3, H, d] buffer.
std::vector<Tensor> qkv_forward(const Tensor& x, const Tensor (&w)[3], const Tensor (&b)[3], int64_t H, int64_t d,
                                int64_t stream) {
    TORCH_CHECK_VALUE(x.dim() == 3, "projection: input [B, L, features] expected");
    const int64_t B = x.size(0), L = x.size(1), dim = x.size(2);
    for (int i = 0; i < 3; ++i) check_projection(x, w[i], b[i], H * d, dim);
    TORCH_CHECK(x.is_cuda(), "fp32 tensors on the GPU expected");
    Tensor buf = torch::empty({B, L, 3, H, d}, x.options());
    const float* wp[3] = {fp(w[0]), fp(w[1]), fp(w[2])};
    const float* bp[3] = {fp(b[0]), fp(b[1]), fp(b[2])};
    spion_project_forward(fp(x), wp, bp, fpm(buf), B * L, (int)(H * d), 3, (int)dim, reinterpret_cast<void*>(stream));
    check_library("projection");
    std::vector<Tensor> out;
    for (int i = 0; i < 3; ++i)  // the slice [:, :, i].transpose(1, 2)
        out.push_back(buf.as_strided({B, H, L, d}, {L * 3 * H * d, d, 3 * H * d, 1}, i * H * d));
    return out;
}

// The backward of both projections runs torch's own operations on the saved inputs when it is itself recorded
// (create_graph): the kernels would leave no graph, and second-order terms would be lost without a word.
struct QkvNode : public torch::autograd::Function<QkvNode> {
    static variable_list forward(AutogradContext* ctx, Tensor x, Tensor wq, Tensor wk, Tensor wv, Tensor bq, Tensor bk,
                                 Tensor bv, int64_t H, int64_t d, int64_t stream) {
        const Tensor w[3] = {aligned(wq), aligned(wk), aligned(wv)}, b[3] = {aligned(bq), aligned(bk), aligned(bv)};
        ctx->save_for_backward({x, wq, wk, wv});
        ctx->saved_data["H"] = H;
        ctx->saved_data["d"] = d;
        ctx->saved_data["x_sizes"] = x.sizes().vec();
        ctx->saved_data["device"] = static_cast<int64_t>(x.device().index());
        return qkv_forward(aligned(x), w, b, H, d, stream);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const int64_t H = ctx->saved_data["H"].toInt(), d = ctx->saved_data["d"].toInt(), n = H * d,
                      device = ctx->saved_data["device"].toInt(), stream = current_stream(device);
        const auto sizes = ctx->saved_data["x_sizes"].toIntVector();
        const int64_t B = sizes[0], L = sizes[1], dim = sizes[2], rows = B * L;
        saved_as(saved[0], sizes, device);
        for (int i = 1; i < 4; ++i) saved_as(saved[i], {n, dim}, device);
        for (auto& t : g)
            if (!t.defined()) t = torch::zeros({B, H, L, d}, saved[0].options());
        if (torch::GradMode::is_enabled()) {
            const Tensor dy = torch::stack({g[0].transpose(1, 2), g[1].transpose(1, 2), g[2].transpose(1, 2)}, 2)
                                  .reshape({rows, 3 * n});
            const Tensor dw = dy.t().matmul(saved[0].reshape({rows, dim})), db = dy.sum(0);
            variable_list r(10);
            r[0] = dy.matmul(torch::cat({saved[1], saved[2], saved[3]}, 0)).view({B, L, dim});
            for (int i = 0; i < 3; ++i) {
                r[1 + i] = dw.narrow(0, i * n, n);
                r[4 + i] = db.narrow(0, i * n, n);
            }
            return r;
        }
        const Tensor x = aligned(saved[0]);
        Tensor keep;  // [B, L, 3, H, d]
        const float* dy = fp(g[0]);
        if (!adjacent_head_views(g[0], g[1], g[2]) || reinterpret_cast<uintptr_t>(dy) % 16) {
            keep = torch::stack({g[0].transpose(1, 2), g[1].transpose(1, 2), g[2].transpose(1, 2)}, 2).contiguous();
            dy = fp(keep);
        }
        variable_list r(10);
        bool any = false;
        for (int i = 1; i < 7; ++i) any = any || ctx->needs_input_grad(i);
        const Tensor w[3] = {aligned(saved[1]), aligned(saved[2]), aligned(saved[3])};
        const ProjectionGrads grads = project_backward(dy, w, x, rows, n, 3, dim, stream, ctx->needs_input_grad(0), any);
        r[0] = grads.dx;
        if (any)
            for (int i = 0; i < 3; ++i) {
                r[1 + i] = grads.dw.narrow(0, i * n, n);
                r[4 + i] = grads.db.narrow(0, i * n, n);
            }
        return r;
    }
};

// The output projection on heads [B, H, L, d] that lie interleaved ([B, L, H*d] in memory: what the core's forward makes
// for the slices above), y [B, L, dim].
Tensor merge_forward(const Tensor& merged, const Tensor& w, const Tensor& b, int64_t stream) {
    TORCH_CHECK_VALUE(merged.dim() == 4 && w.dim() == 2, "projection: heads [B, L, H, d] and a weight matrix expected");
    const int64_t B = merged.size(0), L = merged.size(1), n = merged.size(2) * merged.size(3);
    check_projection(merged, w, b, w.size(0), n);
    TORCH_CHECK(merged.is_cuda(), "fp32 tensors on the GPU expected");
    Tensor y = torch::empty({B, L, w.size(0)}, merged.options());
    const float* wp[1] = {fp(w)};
    const float* bp[1] = {fp(b)};
    spion_project_forward(fp(merged), wp, bp, fpm(y), B * L, (int)w.size(0), 1, (int)n, reinterpret_cast<void*>(stream));
    check_library("projection");
    return y;
}
struct MergeNode : public torch::autograd::Function<MergeNode> {
    static Tensor forward(AutogradContext* ctx, Tensor heads, Tensor w, Tensor b, int64_t stream) {
        ctx->save_for_backward({heads, w});
        ctx->saved_data["heads_sizes"] = heads.sizes().vec();
        ctx->saved_data["outputs"] = w.size(0);
        ctx->saved_data["device"] = static_cast<int64_t>(heads.device().index());
        return merge_forward(aligned(heads.transpose(1, 2)), aligned(w), aligned(b), stream);
    }
    static variable_list backward(AutogradContext* ctx, variable_list g) {
        const auto saved = ctx->get_saved_variables();
        const int64_t device = ctx->saved_data["device"].toInt(), stream = current_stream(device);
        const auto sizes = ctx->saved_data["heads_sizes"].toIntVector();
        const int64_t B = sizes[0], H = sizes[1], L = sizes[2], d = sizes[3];
        const int64_t rows = B * L, n = H * d, dim = ctx->saved_data["outputs"].toInt();
        saved_as(saved[0], sizes, device);
        saved_as(saved[1], {dim, n}, device);
        variable_list r(4);
        if (torch::GradMode::is_enabled()) {
            const Tensor dy = g[0].reshape({rows, dim});
            r[0] = dy.matmul(saved[1]).view({B, L, H, d}).transpose(1, 2);
            r[1] = dy.t().matmul(saved[0].transpose(1, 2).reshape({rows, n}));
            r[2] = dy.sum(0);
            return r;
        }
        const Tensor a = aligned(saved[0].transpose(1, 2)), w = aligned(saved[1]), dy = aligned(g[0]);
        const ProjectionGrads grads = project_backward(fp(dy), &w, a, rows, dim, 1, n, stream, ctx->needs_input_grad(0),
                                                       ctx->needs_input_grad(1) || ctx->needs_input_grad(2));
        if (grads.dx.defined()) r[0] = grads.dx.transpose(1, 2);
        r[1] = grads.dw;
        r[2] = grads.db;
        return r;
    }
};

// The attention layer in its sparse phase (models/attention.py:84-103): projections, sparse core, output projection in
// one call from Python.  Returns [y, p_flat].
std::vector<Tensor> sparse_layer(const Tensor& x, const Tensor& wq, const Tensor& wk, const Tensor& wv, const Tensor& bq,
                                 const Tensor& bk, const Tensor& bv, const Tensor& wf, const Tensor& bf,
                                 const c10::optional<Tensor>& mask_or_pen, bool is_mask, const Tensor& offsets,
                                 const Tensor& columns, const Tensor& sum_mat, int64_t handle, int64_t nnz, int64_t num_heads, int64_t head_dim,
                                 int64_t stream) {
    const c10::DeviceGuard on(x.device());  // `stream` is one of x's device, which need not be the current one
    TORCH_CHECK_VALUE(x.dim() == 3, "projection: input [B, L, features] expected");
    const KeyOperand keys = key_operand(mask_or_pen, is_mask, x.size(0), num_heads, x.size(1), x.device(), stream);
    const Tensor pen_or_none = keys.or_none();
    if (without_node({&x, &wq, &wk, &wv, &bq, &bk, &bv, &wf, &bf, &pen_or_none})) {
        const Tensor w[3] = {aligned(wq), aligned(wk), aligned(wv)}, b[3] = {aligned(bq), aligned(bk), aligned(bv)};
        const auto qkv = qkv_forward(aligned(x), w, b, num_heads, head_dim, stream);
        const CoreResult r = core_forward(qkv[0], qkv[1], qkv[2], pen_or_none, keys.mask_heads, offsets, columns, sum_mat, handle,
                                          nnz, num_heads, true, stream);
        return {merge_forward(aligned(r.out.transpose(1, 2)), aligned(wf), aligned(bf), stream), r.p_flat};
    }
    const auto qkv = QkvNode::apply(x, wq, wk, wv, bq, bk, bv, num_heads, head_dim, stream);
    Tensor fixed;
    const auto core = SparseAttnNode::apply(qkv[0], qkv[1], qkv[2], keys.t, keys.mask_heads, offsets, columns, sum_mat, handle, nnz, num_heads,
                                            true, stream, &fixed);
    return {MergeNode::apply(core[0], wf, bf, stream), core.size() > 1 ? core[1] : fixed};
}

// The two projections by themselves, around a core of the caller's (the dense phase).
std::vector<Tensor> project_heads(const Tensor& x, const Tensor& wq, const Tensor& wk, const Tensor& wv, const Tensor& bq,
                                  const Tensor& bk, const Tensor& bv, int64_t num_heads, int64_t head_dim, int64_t stream) {
    const c10::DeviceGuard on(x.device());
    return QkvNode::apply(x, wq, wk, wv, bq, bk, bv, num_heads, head_dim, stream);
}
Tensor merge_heads(const Tensor& heads, const Tensor& w, const Tensor& b, int64_t stream) {
    const c10::DeviceGuard on(heads.device());
    return MergeNode::apply(heads, w, b, stream);
}

std::vector<Tensor> sparse_attention(const Tensor& query, const Tensor& key, const Tensor& value,
                                     const c10::optional<Tensor>& mask_or_pen, bool is_mask, const Tensor& offsets,
                                     const Tensor& columns, const Tensor& sum_mat, int64_t handle, int64_t nnz, int64_t num_heads,
                                     bool reads_views, int64_t stream) {
    const c10::DeviceGuard on(query.device());
    const bool heads = query.dim() == 4;  // (core_forward asks for them)
    const KeyOperand keys = key_operand(mask_or_pen, is_mask, heads ? query.size(0) : -1, num_heads, heads ? query.size(2) : -1,
                                        query.device(), stream);
    const Tensor pen_or_none = keys.or_none();
    if (without_node({&query, &key, &value, &pen_or_none})) {
        const CoreResult r = core_forward(query, key, value, pen_or_none, keys.mask_heads, offsets, columns, sum_mat, handle, nnz,
                                          num_heads, reads_views, stream);
        return {r.out, r.p_flat};
    }
    Tensor fixed;
    auto r = SparseAttnNode::apply(query, key, value, keys.t, keys.mask_heads, offsets, columns, sum_mat, handle, nnz, num_heads, reads_views,
                                   stream, &fixed);
    if (r.size() == 1) r.push_back(fixed);
    return r;
}

// The kernels read a penalty for every key of every head: fewer, or a tensor elsewhere, would be read past its end.
void check_penalties(const Tensor& pen, int64_t mask_heads, const Tensor& query) {
    if (!pen.defined()) return;
    TORCH_CHECK(pen.scalar_type() == torch::kFloat32 && pen.device() == query.device(), "fp32 tensors on one GPU expected");
    TORCH_CHECK_VALUE(pen.numel() >= query.size(0) * (mask_heads ? 1 : query.size(1)) * query.size(2),
                      "key mask smaller than [B, L]");
}

// fp32 heads of the handle's sizes on one GPU (the module's test); mask_or_pen as for sparse_attention.  [out, map, mean or
// nothing]
std::vector<Tensor> dense_attention(const Tensor& query, const Tensor& key, const Tensor& value,
                                    const c10::optional<Tensor>& mask_or_pen, bool is_mask, int64_t handle, bool emit_mean,
                                    int64_t stream) {
    const c10::DeviceGuard on(query.device());
    const KeyOperand keys = key_operand(mask_or_pen, is_mask, query.size(0), query.size(1), query.size(2), query.device(), stream);
    const Tensor pen_or_none = keys.or_none();
    check_penalties(pen_or_none, keys.mask_heads, query);
    if (without_node({&query, &key, &value, &pen_or_none})) {
        DenseResult r = dense_forward(query, key, value, pen_or_none, keys.mask_heads, handle, emit_mean, stream);
        return {r.out, r.attn.transpose(2, 3), r.mean};
    }
    Tensor mean;
    const auto r = DenseAttnNode::apply(query, key, value, keys.t, keys.mask_heads, handle, emit_mean, stream, &mean);
    return {r[0], r[1], mean};
}

// The same for the bf16 module: heads of any floating type.
Tensor bf16_attention(const Tensor& query, const Tensor& key, const Tensor& value, const c10::optional<Tensor>& mask_or_pen,
                      bool is_mask, const Tensor& offsets, const Tensor& columns, const Tensor& sum_mat, int64_t handle,
                      int64_t nnz, int64_t stream) {
    const c10::DeviceGuard on(query.device());
    // a backward needs the penalties too, whatever has become of the mask by then
    const bool plain = without_node({&query, &key, &value});
    const KeyOperand keys = plain ? key_operand(mask_or_pen, is_mask, query.size(0), query.size(1), query.size(2), query.device(), stream)
                                  : KeyOperand{penalty_of(mask_or_pen, is_mask, query.size(1), query.device(), stream), 0};
    const Tensor pen_or_none = keys.or_none();
    check_penalties(pen_or_none, keys.mask_heads, query);
    if (plain && without_node({&pen_or_none}))
        return bf16_forward(query, key, value, pen_or_none, keys.mask_heads, offsets, columns, sum_mat, handle, nnz, stream).out;
    return BF16AttnNode::apply(query, key, value, keys.t, offsets, columns, sum_mat, handle, nnz, stream);
}

}  // namespace

PYBIND11_MODULE(TORCH_EXTENSION_NAME, m) {
    m.doc() = "C++ autograd nodes of the sparse attention modules";
    m.def("sparse_attention", &sparse_attention, "forward of the sparse attention modules; returns [out, p_flat]",
          py::arg("query"), py::arg("key"), py::arg("value"), py::arg("mask_or_pen"), py::arg("is_mask"), py::arg("offsets"),
          py::arg("columns"), py::arg("sum_mat"), py::arg("handle"), py::arg("nnz"), py::arg("num_heads"),
          py::arg("reads_views"), py::arg("stream"));
    m.def("dense_attention", &dense_attention, "forward of the dense-phase modules; returns [out, map, mean map or None]");
    m.def("bf16_attention", &bf16_attention, "forward of the bf16 module");
    m.def("sparse_layer", &sparse_layer, "forward of the attention layer in its sparse phase; returns [y, p_flat]");
    m.def("projections_fit", &projections_fit, "whether the projection kernels take this layer's linear layers");
    m.def("project_heads", &project_heads, "the three input projections; returns the [B, H, L, d] heads");
    m.def("merge_heads", &merge_heads, "the output projection of [B, H, L, d] heads");
}
