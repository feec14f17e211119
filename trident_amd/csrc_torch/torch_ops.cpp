// The operator's host path in C++: argument structures, allocations, launches and the autograd nodes of
// function.scaled_dot_product_attention, softmax, masked_softmax and dropout.
//
// A small training step is bounded by its host work: two Python autograd Functions, the argument structure and ctypes took
// 55 us of a step whose kernels take 22 (fp16, B=32 H=8 S=128 D=64). The functions below do the same without the
// interpreter, in the backward without its lock. They take plain calls only: exact torch tensors on one GPU, no tracing,
// no functorch transform, no torch function or dispatch mode, no forward-mode differentiation. For anything else, errors
// included, they return None and launch nothing, and the Python Functions in operation.py and rowops.py, which state the
// rules, take the call.
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/extension.h>

#include <cmath>
#include <limits>
#include <mutex>
#include <unordered_map>

#include "tri_attn.h"
#include "tri_rowops.h"

namespace {

using at::Tensor;

// The library's entry points, handed over by bind() (the library is loaded by the Python side).
struct Library {
    decltype(&tri_attn_strerror) strerror = nullptr;
    decltype(&tri_attn_fwd) fwd = nullptr;
    decltype(&tri_attn_bwd) bwd = nullptr;
    decltype(&tri_attn_bwd_dmask) bwd_dmask = nullptr;
    decltype(&tri_attn_uses_matrix_cores) uses_matrix_cores = nullptr;
    decltype(&tri_attn_workspace_size) workspace_size = nullptr;
    decltype(&tri_attn_mask_classes_size) mask_classes_size = nullptr;
    decltype(&tri_attn_classify_mask) classify_mask = nullptr;
    decltype(&tri_attn_prepare_mask) prepare_mask = nullptr;
    decltype(&tri_softmax_fwd) softmax_fwd = nullptr;
    decltype(&tri_softmax_bwd) softmax_bwd = nullptr;
    decltype(&tri_softmax_workspace_size) softmax_workspace_size = nullptr;
    decltype(&tri_dropout_fwd) dropout_fwd = nullptr;
    decltype(&tri_dropout_bwd) dropout_bwd = nullptr;
} lib;

// The namespaces of the Python modules config and operation, whose switches are read where a call needs them.
PyObject* config_dict = nullptr;
PyObject* operation_dict = nullptr;
PyObject *name_use_trace, *name_reference_limits, *name_cache, *name_pads_from, *name_next_seed;

void check(int status) {
    TORCH_CHECK(status == 0, "tri_attn: ", lib.strerror(status));
}

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return TRI_ATTN_F32;
        case at::kHalf: return TRI_ATTN_F16;
        case at::kBFloat16: return TRI_ATTN_BF16;
        default: return -1;
    }
}

bool is_true(PyObject* dict, PyObject* name) {  // (GIL held)
    PyObject* v = PyDict_GetItemWithError(dict, name);  // borrowed
    if (v == nullptr) throw python_error();
    const int r = PyObject_IsTrue(v);
    if (r < 0) throw python_error();
    return r != 0;
}

int64_t int_of(PyObject* dict, PyObject* name) {  // (GIL held)
    PyObject* v = PyDict_GetItemWithError(dict, name);
    if (v == nullptr) throw python_error();
    const int64_t r = PyLong_AsLongLong(v);
    if (r == -1 && PyErr_Occurred()) throw python_error();
    return r;
}

// An exact torch.Tensor or Parameter (subclasses have their own ways through the Python Functions).
const Tensor* plain_tensor(PyObject* o) {
    PyTypeObject* t = Py_TYPE(o);
    if (t != reinterpret_cast<PyTypeObject*>(THPVariableClass) && t != reinterpret_cast<PyTypeObject*>(ParameterClass)) return nullptr;
    return &THPVariable_Unpack(o);
}

bool on_gpu(const Tensor& t) { return t.is_cuda() && t.layout() == at::kStrided && !t.is_neg() && !t.is_conj(); }

// Whether nothing watches or rewrites what a call does: those go through the Python Functions.
bool plain_context() {
    return !c10::impl::TorchDispatchModeTLS::any_modes_set() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !c10::impl::tls_local_dispatch_key_set().included_.has(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) &&
           !torch::jit::tracer::isTracing() && torch::autograd::ForwardADLevel::try_get_by_idx(0) == nullptr &&
           !is_true(config_dict, name_use_trace);
}

void* current_stream(const Tensor& t) {
    return reinterpret_cast<void*>(c10::hip::getCurrentHIPStreamMasqueradingAsCUDA(t.device().index()).stream());
}

bool stream_is_capturing() {  // (of the current device's stream)
    return c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None;
}

bool pow2(int64_t n) { return n != 0 && (n & (n - 1)) == 0; }

// ---------------------------------------------------------------- attention

Tensor dense_rows(const Tensor& t) {  // the kernels need unit stride along the last dimension
    return t.size(-1) != 1 && t.stride(-1) != 1 ? t.contiguous() : t;
}

void set_strides(int64_t* dst, const Tensor& t) {
    for (int i = 0; i < 4; ++i) dst[i] = t.stride(i);
    if (t.size(-1) == 1) dst[3] = 1;
}

// operation._expand_mask: the mask broadcast to `full`, unit stride along the keys.
Tensor expand_mask(const Tensor& mask, at::IntArrayRef full) {
    Tensor view = mask.detach().expand(full);
    return view.size(-1) != 1 && view.stride(-1) != 1 ? view.contiguous() : view;
}

// operation._PreparedMask
struct Prepared {
    Tensor padded, classes;
    int64_t strides[4];
    int dtype;

    void describe(TriAttnArgs& a) const {
        a.mask = padded.data_ptr();
        a.mask_dtype = dtype;
        std::copy(strides, strides + 4, a.mask_stride);
        if (classes.defined()) a.mask_classes = static_cast<uint8_t*>(classes.data_ptr());
    }
};

std::shared_ptr<Prepared> prepare(const Tensor& source, const Tensor& query) {
    const int64_t B = query.size(0), H = query.size(1), S = query.size(2);
    const int64_t full[4] = {B, H, S, S};
    const int missing = 4 - static_cast<int>(source.dim());
    int64_t shape[4], from[4], kept[4];
    for (int i = 0; i < 4; ++i) {
        shape[i] = i < missing ? 1 : source.size(i - missing);
        from[i] = i < missing || shape[i] == 1 ? 0 : source.stride(i - missing);
        kept[i] = from[i] == 0 ? 1 : shape[i];  // (a dimension the source broadcasts is kept once)
    }
    if (missing < 0 || !std::equal(shape, shape + 4, full, [](int64_t n, int64_t m) { return n == 1 || n == m; }))
        source.expand(full);  // (raises)
    const int64_t pitch = (S + 63) / 64 * 64, blocks = pitch / 64;
    const bool boolean = source.scalar_type() == at::kBool;
    const auto dtype = boolean ? query.scalar_type() : source.scalar_type();
    auto m = std::make_shared<Prepared>();
    m->padded = at::empty({kept[0] * kept[1] * kept[2] * pitch}, query.options().dtype(dtype));
    m->strides[0] = kept[0] > 1 ? kept[1] * kept[2] * pitch : 0;
    m->strides[1] = kept[1] > 1 ? kept[2] * pitch : 0;
    m->strides[2] = kept[2] > 1 ? pitch : 0;
    m->strides[3] = 1;
    m->dtype = dtype_code(dtype) | TRI_ATTN_MASK_PADDED | (boolean ? TRI_ATTN_MASK_BINARY : 0);
    if (query.scalar_type() != at::kFloat)
        m->classes = at::empty({kept[0] * kept[1] * (kept[2] > 1 ? blocks : 1) * blocks}, query.options().dtype(at::kByte));
    TriAttnArgs a{};
    a.struct_size = sizeof(a);
    a.B = static_cast<int32_t>(B);
    a.H = static_cast<int32_t>(H);
    a.S = static_cast<int32_t>(S);
    a.stream = current_stream(query);
    m->describe(a);
    check(lib.prepare_mask(&a, source.data_ptr(), boolean ? TRI_ATTN_BOOL : dtype_code(dtype), from));
    return m;
}

constexpr int64_t kPadsLong = int64_t{1} << 28;  // operation._PADS_LONG
constexpr int64_t kKeptBytes = int64_t{1} << 22;

// operation._worth_padding
bool worth_padding(const Tensor& query, int64_t pads_from) {
    const int64_t S = query.size(2), work = query.size(0) * query.size(1) * S * S * std::max<int64_t>(query.size(3), 32);
    return std::max(work, S > 128 ? kPadsLong : int64_t{0}) >= pads_from;
}

// operation._sums_mask_gradient
bool sums_mask_gradient(const Tensor& mask, const Tensor& query, int64_t pads_from) {
    const int64_t S = query.size(2);
    if (query.scalar_type() == at::kFloat || mask.dim() < 2 || mask.size(-1) != S || mask.size(-2) != S) return false;
    const int64_t b = mask.dim() >= 4 ? mask.size(-4) : 1, h = mask.dim() >= 3 ? mask.size(-3) : 1;
    return b != query.size(0) || h != query.size(1) || (S % 128 != 0 && (S % 64 == 0 || worth_padding(query, pads_from)));
}

// What a call was asked for, kept for its backward.
struct Call : torch::CustomClassHolder {
    Tensor mask;                         // as given; of a boolean one the prepared mask is kept in its place
    std::shared_ptr<Prepared> prepared;  // a boolean mask, or a small padded one, on its way through forward and backward
    bool boolean = false;
    double dropout_p = 0.0, scale = 1.0;
    bool causal = false;
    uint64_t seed = 0, offset = 0;
};

// operation._prepared_mask
std::shared_ptr<Prepared> prepared_mask(const Call& call, const Tensor& query, int64_t pads_from) {
    if (call.prepared) return call.prepared;
    const Tensor& mask = call.mask;
    if (query.size(2) % 64 == 0 || !worth_padding(query, pads_from)) return nullptr;
    if (query.scalar_type() == at::kFloat || (mask.scalar_type() != at::kFloat && mask.scalar_type() != query.scalar_type())) return nullptr;
    if (mask.requires_grad() && !sums_mask_gradient(mask, query, pads_from)) return nullptr;
    try {
        return prepare(mask.detach(), query);
    } catch (const c10::OutOfMemoryError&) {
        return nullptr;
    }
}

// Classes of a mask's 64 x 64 blocks, kept per mask tensor: the rules stand at operation._mask_classes.
struct ClassesEntry {
    c10::weak_intrusive_ptr<c10::TensorImpl> owner;
    uint32_t version;
    std::vector<int64_t> signature;
    Tensor classes;
};
std::mutex classes_lock;
std::unordered_map<const c10::TensorImpl*, ClassesEntry>& classes_cache() {
    static auto* cache = new std::unordered_map<const c10::TensorImpl*, ClassesEntry>;  // (never destroyed: it holds device memory)
    return *cache;
}
constexpr size_t kMaxClasses = 64;

std::vector<int64_t> classes_signature(const Tensor& mask, const TriAttnArgs& a) {
    std::vector<int64_t> s(mask.sizes().begin(), mask.sizes().end());
    s.insert(s.end(), mask.strides().begin(), mask.strides().end());
    for (int64_t v : {static_cast<int64_t>(mask.scalar_type()), static_cast<int64_t>(a.B), static_cast<int64_t>(a.H), static_cast<int64_t>(a.S),
                      reinterpret_cast<int64_t>(a.mask), reinterpret_cast<int64_t>(a.stream)})
        s.push_back(v);
    return s;
}

Tensor mask_classes(const Tensor& mask, TriAttnArgs& a, bool may_cache) {
    if (a.dtype == TRI_ATTN_F32) return Tensor();  // (no fp32 kernel looks at them)
    const int64_t size = lib.mask_classes_size(&a);
    if (size <= 0) return Tensor();
    const bool use_cache = may_cache && !stream_is_capturing() && !mask.is_inference();
    const c10::TensorImpl* key = mask.unsafeGetTensorImpl();
    std::vector<int64_t> signature;
    uint32_t version = 0;
    if (use_cache) {
        signature = classes_signature(mask, a);
        version = mask._version();
        std::lock_guard<std::mutex> guard(classes_lock);
        auto it = classes_cache().find(key);
        if (it != classes_cache().end() && !it->second.owner.expired() && it->second.version == version && it->second.signature == signature) {
            a.mask_classes = static_cast<uint8_t*>(it->second.classes.data_ptr());
            return it->second.classes;
        }
    }
    Tensor classes = at::empty({size}, mask.options().dtype(at::kByte).requires_grad(false));
    a.mask_classes = static_cast<uint8_t*>(classes.data_ptr());
    const int status = lib.classify_mask(&a);
    if (status == TRI_ATTN_ENOFUSE || status == TRI_ATTN_EALIGN) {
        a.mask_classes = nullptr;
        return Tensor();
    }
    check(status);
    if (use_cache) {
        std::vector<Tensor> freed;  // (released outside the lock)
        std::lock_guard<std::mutex> guard(classes_lock);
        auto& cache = classes_cache();
        // (also what this entry replaces: a tensor that Python has seen takes the interpreter's lock to go, which a thread
        // waiting for this one may hold)
        if (const auto old = cache.find(key); old != cache.end()) {
            freed.push_back(std::move(old->second.classes));
            cache.erase(old);
        }
        for (auto it = cache.begin(); it != cache.end();) {  // entries of tensors that are gone; all of them when it is full
            if (it->second.owner.expired() || cache.size() >= kMaxClasses) {
                freed.push_back(std::move(it->second.classes));
                it = cache.erase(it);
            } else ++it;
        }
        cache.insert_or_assign(key, ClassesEntry{c10::weak_intrusive_ptr<c10::TensorImpl>(mask.getIntrusivePtr()), version, std::move(signature), classes});
    }
    return classes;
}

struct MaskSwitches {
    bool cache = false;
    int64_t pads_from = 0;
};
MaskSwitches mask_switches() {
    py::gil_scoped_acquire gil;
    return {is_true(config_dict, name_cache), int_of(operation_dict, name_pads_from)};
}

TriAttnArgs make_args(const Call& call, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& lse, const Tensor& mask_view) {
    TriAttnArgs a{};
    a.struct_size = sizeof(a);
    a.dtype = dtype_code(q.scalar_type());
    a.B = static_cast<int32_t>(q.size(0));
    a.H = static_cast<int32_t>(q.size(1));
    a.S = static_cast<int32_t>(q.size(2));
    a.D = static_cast<int32_t>(q.size(3));
    a.is_causal = call.causal;
    a.softmax_scale = static_cast<float>(call.scale);
    a.dropout_p = static_cast<float>(call.dropout_p);
    a.seed = call.seed;
    a.offset = call.offset;
    a.q = q.data_ptr();
    a.k = k.data_ptr();
    a.v = v.data_ptr();
    a.o = o.data_ptr();
    a.lse = static_cast<float*>(lse.data_ptr());
    set_strides(a.q_stride, q);
    set_strides(a.k_stride, k);
    set_strides(a.v_stride, v);
    set_strides(a.o_stride, o);
    if (mask_view.defined()) {
        a.mask = mask_view.data_ptr();
        a.mask_dtype = dtype_code(mask_view.scalar_type());
        set_strides(a.mask_stride, mask_view);
    }
    a.stream = current_stream(q);
    return a;
}

// operation._take_workspace
template <typename Args>
Tensor give_workspace(Args& a, int64_t size, const Tensor& q) {
    if (size <= 0) return Tensor();
    try {
        Tensor workspace = at::empty({size}, q.options().dtype(at::kByte).requires_grad(false));
        a.workspace = workspace.data_ptr();
        a.workspace_size = size;
        return workspace;
    } catch (const c10::OutOfMemoryError&) {
        return Tensor();
    }
}
Tensor take_workspace(TriAttnArgs& a, int pass, const Tensor& q) { return give_workspace(a, lib.workspace_size(&a, pass), q); }

// operation.Attention._forward
std::pair<Tensor, Tensor> attention_forward(Call& call, const Tensor& query, const Tensor& key, const Tensor& value) {
    const c10::DeviceGuard device(query.device());
    const Tensor q = dense_rows(query), k = dense_rows(key), v = dense_rows(value);
    const int64_t B = q.size(0), H = q.size(1), S = q.size(2);
    const Tensor output = at::empty(q.sizes(), q.options().requires_grad(false));
    const Tensor lse = at::empty({B, H, S}, q.options().dtype(at::kFloat).requires_grad(false));
    MaskSwitches switches;
    std::shared_ptr<Prepared> prepared;
    Tensor mask_view;
    if (call.mask.defined()) {
        switches = mask_switches();
        if (call.boolean) {
            call.prepared = prepare(call.mask, q);
            call.mask.reset();
        }
        prepared = prepared_mask(call, q, switches.pads_from);
        if (prepared == nullptr) mask_view = expand_mask(call.mask, {B, H, S, S});
        // (for the backward, which pads a larger mask again instead of holding the memory until then)
        else if (prepared->padded.nbytes() <= kKeptBytes) call.prepared = prepared;
    }
    TriAttnArgs a = make_args(call, q, k, v, output, lse, mask_view);
    if (prepared) prepared->describe(a);
    Tensor classes;  // (kept alive until the call is enqueued)
    if (mask_view.defined()) classes = mask_classes(call.mask, a, switches.cache);
    const Tensor workspace = take_workspace(a, 0, q);
    check(lib.fwd(&a));
    return {output, lse};
}

// operation._require_same_gpu and rowops._require_gpu, for what a backward finds: a saved tensor may come back from a hook of the
// caller's as something else, and the kernels take raw pointers.
void require_saved_as(const Tensor& saved, const char* name, const Tensor& like, at::IntArrayRef sizes, at::ScalarType dtype) {
    TORCH_CHECK(on_gpu(saved) && saved.device() == like.device(), "trident_amd: ", name, " is on ", saved.device(), ", expected ", like.device(),
                " (all tensors of a call must be on the same GPU)");
    TORCH_CHECK(saved.sizes() == sizes && saved.scalar_type() == dtype, "trident_amd: the saved ", name, " has come back with another shape or dtype");
}

// operation.Attention._backward
std::array<Tensor, 4> attention_backward(const Call& call, const Tensor& grad_out, const Tensor& query, const Tensor& key, const Tensor& value,
                                         const Tensor& output, const Tensor& saved_lse, bool want_grad_mask) {
    require_saved_as(query, "query", grad_out, grad_out.sizes(), grad_out.scalar_type());
    require_saved_as(key, "key", query, query.sizes(), query.scalar_type());
    require_saved_as(value, "value", query, query.sizes(), query.scalar_type());
    require_saved_as(output, "output", query, query.sizes(), query.scalar_type());
    require_saved_as(saved_lse, "log_sum_exp", query, query.sizes().slice(0, 3), at::kFloat);
    const c10::DeviceGuard device(query.device());
    const Tensor lse = saved_lse.contiguous();
    const Tensor q = dense_rows(query), k = dense_rows(key), v = dense_rows(value), grad_output = dense_rows(grad_out);
    const int64_t B = q.size(0), H = q.size(1), S = q.size(2);
    const std::array<int64_t, 4> full = {B, H, S, S};
    auto dense = [](const Tensor& t) { return at::empty(t.sizes(), t.options().requires_grad(false)); };
    const Tensor dq = dense(q), dk = dense(k), dv = dense(v);
    const Tensor delta = at::empty({B, H, S}, lse.options());
    const bool masked = call.mask.defined() || call.prepared;
    MaskSwitches switches;
    if (masked) switches = mask_switches();
    const Tensor& mask = call.mask;
    bool summed = want_grad_mask && sums_mask_gradient(mask, q, switches.pads_from);  // (a mask whose gradient the dQ pass writes was not padded)
    std::shared_ptr<Prepared> prepared;
    if (masked && !want_grad_mask) prepared = prepared_mask(call, q, switches.pads_from);
    Tensor mask_view, grad_mask_buf, grad_mask_view;
    if (masked && prepared == nullptr) mask_view = expand_mask(mask, full);
    std::array<int64_t, 4> shape4 = {1, 1, 1, 1};
    if (want_grad_mask) {
        for (int i = 0; i < mask.dim(); ++i) shape4[4 - mask.dim() + i] = mask.size(i);
        if (shape4 == full || summed) {
            grad_mask_buf = at::empty(shape4, mask.options().requires_grad(false));
            grad_mask_view = shape4 == full ? grad_mask_buf : grad_mask_buf.expand(full);
        }
    }
    TriAttnArgs a = make_args(call, q, k, v, output, lse, mask_view);
    a.d_o = grad_output.data_ptr();
    a.dq = dq.data_ptr();
    a.dk = dk.data_ptr();
    a.dv = dv.data_ptr();
    a.delta = static_cast<float*>(delta.data_ptr());
    set_strides(a.do_stride, grad_output);
    set_strides(a.dq_stride, dq);
    set_strides(a.dk_stride, dk);
    set_strides(a.dv_stride, dv);
    auto set_grad_mask = [&](const Tensor& t) {
        a.dmask = t.data_ptr();
        set_strides(a.dmask_stride, t);
    };
    auto set_mask = [&](const Tensor& t) {
        a.mask = t.data_ptr();
        a.mask_dtype = dtype_code(t.scalar_type());
        set_strides(a.mask_stride, t);
    };
    if (grad_mask_view.defined()) set_grad_mask(grad_mask_view);
    Tensor classes;  // (kept alive until the call is enqueued, as `prepared`)
    if (summed) {
        summed = lib.uses_matrix_cores(&a, 3) == 1;
        if (summed) {  // (else the dQ pass writes it: in place, or below, into what broadcast dimensions are added up in)
            a.dmask = nullptr;
            prepared = prepared_mask(call, q, switches.pads_from);
        }
    }
    if (prepared) {
        prepared->describe(a);
    } else if (masked && (summed || !want_grad_mask)) {
        if (!summed || mask.scalar_type() == at::kFloat || !stream_is_capturing()) classes = mask_classes(mask, a, switches.cache);
    } else if (want_grad_mask) {
        if (shape4 != full) {
            grad_mask_buf = at::zeros(shape4, mask.options().dtype(at::kFloat).requires_grad(false));
            grad_mask_view = grad_mask_buf.expand(full);
            set_grad_mask(grad_mask_view);
            if (mask_view.scalar_type() != at::kFloat) {  // (mask and dmask share one dtype field)
                mask_view = expand_mask(mask.detach().to(at::kFloat), full);
                set_mask(mask_view);
            }
        }
        if (mask_view.scalar_type() == mask.scalar_type()) classes = mask_classes(mask, a, switches.cache);
    }
    const Tensor workspace = take_workspace(a, 3, q);
    check(lib.bwd(&a));
    if (summed) {
        set_mask(mask_view);
        a.dmask = grad_mask_buf.data_ptr();
        a.workspace = nullptr;
        a.workspace_size = 0;
        const Tensor sums = take_workspace(a, 4, q);
        check(lib.bwd_dmask(&a));
    }
    Tensor grad_mask;
    if (grad_mask_buf.defined()) grad_mask = grad_mask_buf.to(mask.scalar_type()).reshape(mask.sizes());
    return {dq, dk, dv, grad_mask};
}

struct AttentionBackward : torch::autograd::Function<AttentionBackward> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& query, const Tensor& key, const Tensor& value,
                          const std::optional<Tensor>& /*mask: call->mask*/, const c10::intrusive_ptr<Call>& call) {
        const auto [output, lse] = attention_forward(*call, query, key, value);
        ctx->save_for_backward({query, key, value, output, lse});
        ctx->saved_data["call"] = c10::IValue::make_capsule(call);
        return output;
    }

    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const auto capsule = ctx->saved_data["call"].toCapsule();
        const Call& call = static_cast<const Call&>(*capsule);
        const auto g = attention_backward(call, grads[0], saved[0], saved[1], saved[2], saved[3], saved[4],
                                          call.mask.defined() && ctx->needs_input_grad(3));
        return {g[0], g[1], g[2], g[3], Tensor()};
    }
};

// attention(query, key, value, mask, dropout_p, is_causal, softmax_scale) -> output, or None
PyObject* attention(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 7, "attention takes 7 arguments");
    const Tensor *q = plain_tensor(args[0]), *k = plain_tensor(args[1]), *v = plain_tensor(args[2]);
    const Tensor* mask = args[3] == Py_None ? nullptr : plain_tensor(args[3]);
    if (q == nullptr || k == nullptr || v == nullptr || (mask == nullptr && args[3] != Py_None)) Py_RETURN_NONE;
    if (q->dim() != 4 || !on_gpu(*q) || !on_gpu(*k) || !on_gpu(*v) || dtype_code(q->scalar_type()) < 0) Py_RETURN_NONE;
    if (k->sizes() != q->sizes() || v->sizes() != q->sizes() || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() ||
        k->device() != q->device() || v->device() != q->device())
        Py_RETURN_NONE;
    const int64_t S = q->size(2), D = q->size(3);
    if ((D != 16 && D != 32 && D != 64 && D != 128) || q->numel() == 0 || !plain_context()) Py_RETURN_NONE;
    for (int i = 0; i < 3; ++i)
        if (q->size(i) > std::numeric_limits<int32_t>::max()) Py_RETURN_NONE;
    if (!PyFloat_CheckExact(args[4]) && !PyLong_CheckExact(args[4])) Py_RETURN_NONE;
    if (!PyBool_Check(args[5]) || !PyFloat_CheckExact(args[6])) Py_RETURN_NONE;
    const bool limits = is_true(config_dict, name_reference_limits);
    if (limits && !pow2(S)) Py_RETURN_NONE;
    auto call = c10::make_intrusive<Call>();
    call->causal = args[5] == Py_True;
    if (mask != nullptr) {
        call->boolean = mask->scalar_type() == at::kBool;
        if (call->causal || !on_gpu(*mask) || mask->device() != q->device() || mask->dim() > 4 || (call->boolean && limits) ||
            (!call->boolean && dtype_code(mask->scalar_type()) < 0))
            Py_RETURN_NONE;
        call->mask = *mask;
    }
    call->scale = PyFloat_AS_DOUBLE(args[6]);
    call->dropout_p = PyFloat_AsDouble(args[4]);
    if (call->dropout_p == -1.0 && PyErr_Occurred()) throw python_error();
    if (call->dropout_p > 0.0) {  // operation._next_seed() -> (seed, offset)
        PyObject* next_seed = PyDict_GetItemWithError(operation_dict, name_next_seed);
        if (next_seed == nullptr) throw python_error();
        const py::object pair = py::reinterpret_steal<py::object>(PyObject_CallNoArgs(next_seed));
        if (!pair) throw python_error();
        call->seed = PyLong_AsUnsignedLongLongMask(PyTuple_GetItem(pair.ptr(), 0));
        call->offset = PyLong_AsUnsignedLongLongMask(PyTuple_GetItem(pair.ptr(), 1));
        if (PyErr_Occurred()) throw python_error();
    }
    Tensor output;
    {
        const Tensor query = *q, key = *k, value = *v;
        const std::optional<Tensor> given = mask ? std::optional<Tensor>(*mask) : std::nullopt;
        py::gil_scoped_release no_gil;
        const bool wanted = at::GradMode::is_enabled() && (query.requires_grad() || key.requires_grad() || value.requires_grad() ||
                                                           (given && given->requires_grad()));
        output = wanted ? AttentionBackward::apply(query, key, value, given, call) : attention_forward(*call, query, key, value).first;
    }
    return THPVariable_Wrap(std::move(output));
    END_HANDLE_TH_ERRORS
}

// mask_classes(mask, address of a TriAttnArgs, may_cache) -> tensor or None (sets args.mask_classes)
PyObject* py_mask_classes(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 3 && THPVariable_Check(args[0]), "mask_classes takes a tensor, an address and a flag");
    auto* a = reinterpret_cast<TriAttnArgs*>(PyLong_AsVoidPtr(args[1]));
    if (PyErr_Occurred()) throw python_error();
    TORCH_CHECK(a != nullptr && a->struct_size == sizeof(*a), "TriAttnArgs of another size");
    const Tensor& mask = THPVariable_Unpack(args[0]);
    const c10::DeviceGuard device(mask.device());
    Tensor classes = mask_classes(mask, *a, args[2] == Py_True);
    if (!classes.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(classes));
    END_HANDLE_TH_ERRORS
}

PyObject* forget_mask_classes(PyObject*, PyObject*) {
    HANDLE_TH_ERRORS
    std::unordered_map<const c10::TensorImpl*, ClassesEntry> freed;
    {
        std::lock_guard<std::mutex> guard(classes_lock);
        freed.swap(classes_cache());
    }
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// ---------------------------------------------------------------- row operations

// rowops._same_layout
Tensor same_layout(const Tensor& t, const Tensor& like) {
    if (t.sizes() == like.sizes() && t.strides() == like.strides()) return t;
    Tensor out = at::empty_strided(like.sizes(), like.strides(), t.options().requires_grad(false));
    out.copy_(t.expand(like.sizes()));
    return out;
}

// rowops._dense
Tensor dense_matrix(const Tensor& t) {
    return t.is_contiguous() || (t.dim() == 2 && t.t().is_contiguous()) ? t : t.contiguous();
}

// rowops._row_args of a dense tensor (columns: the operation runs down dimension 0 of a matrix)
TriRowArgs row_args(const Tensor& t, bool columns) {
    TriRowArgs a{};
    a.struct_size = sizeof(a);
    a.dtype = dtype_code(t.scalar_type());
    if (columns) {
        a.x_size = t.size(0);
        a.y_size = t.size(1);
        a.y_stride = t.stride(1);
        a.x_stride = t.stride(0);
    } else if (t.dim() == 2) {
        a.y_size = t.size(0);
        a.x_size = t.size(1);
        a.y_stride = t.stride(0);
        a.x_stride = t.stride(1);
    } else {
        a.x_size = t.size(-1);
        a.y_size = t.numel() / a.x_size;
        a.y_stride = a.x_size;
        a.x_stride = 1;
    }
    a.stream = current_stream(t);
    return a;
}

int row_mask_code(at::ScalarType t) {
    switch (t) {
        case at::kLong: return TRI_ROW_MASK_I64;
        case at::kInt: return TRI_ROW_MASK_I32;
        case at::kByte:
        case at::kBool: return TRI_ROW_MASK_U8;
        default: return dtype_code(t);
    }
}

Tensor softmax_forward(const Tensor& given, const std::optional<Tensor>& given_mask, bool columns) {
    const c10::DeviceGuard device(given.device());
    const Tensor input = dense_matrix(given);
    const Tensor output = at::empty_like(input);
    TriRowArgs a = row_args(input, columns);
    a.input = input.data_ptr();
    a.output = output.data_ptr();
    Tensor mask;
    if (given_mask) {
        mask = same_layout(*given_mask, input);
        a.mask = mask.data_ptr();
        a.mask_dtype = row_mask_code(mask.scalar_type());
    }
    const Tensor workspace = give_workspace(a, lib.softmax_workspace_size(&a, 0), input);  // (rowops._take_workspace)
    check(lib.softmax_fwd(&a));
    return output;
}

struct SoftmaxBackward : torch::autograd::Function<SoftmaxBackward> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& input, const std::optional<Tensor>& mask, bool columns) {
        const Tensor output = softmax_forward(input, mask, columns);
        ctx->save_for_backward({output});
        ctx->saved_data["columns"] = columns;
        return output;
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const Tensor saved = ctx->get_saved_variables()[0];
        require_saved_as(saved, "output", grads[0], grads[0].sizes(), grads[0].scalar_type());
        const c10::DeviceGuard device(saved.device());
        const Tensor output = dense_matrix(saved);  // (a hook may have laid it out anew)
        const Tensor grad_output = same_layout(grads[0], output);
        const Tensor grad_input = at::empty_like(output);
        TriRowArgs a = row_args(output, ctx->saved_data["columns"].toBool());
        a.output = output.data_ptr();
        a.grad_output = grad_output.data_ptr();
        a.grad_input = grad_input.data_ptr();
        const Tensor workspace = give_workspace(a, lib.softmax_workspace_size(&a, 1), output);
        check(lib.softmax_bwd(&a));
        return {grad_input, Tensor(), Tensor()};
    }
};

// softmax(input, mask or None, dim) -> output, or None
PyObject* softmax(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 3, "softmax takes 3 arguments");
    const Tensor* x = plain_tensor(args[0]);
    const Tensor* mask = args[1] == Py_None ? nullptr : plain_tensor(args[1]);
    if (x == nullptr || (mask == nullptr && args[1] != Py_None)) Py_RETURN_NONE;
    if (!on_gpu(*x) || x->dim() < 2 || x->numel() == 0 || dtype_code(x->scalar_type()) < 0 || !plain_context()) Py_RETURN_NONE;
    if (mask != nullptr && (!on_gpu(*mask) || mask->device() != x->device() || row_mask_code(mask->scalar_type()) < 0 || mask->requires_grad()))
        Py_RETURN_NONE;
    bool columns = false;
    if (x->dim() != 2 || args[2] != Py_None) {
        if (!PyLong_CheckExact(args[2])) Py_RETURN_NONE;
        const int64_t dim = PyLong_AsLongLong(args[2]);
        if (dim == -1 && PyErr_Occurred()) {
            PyErr_Clear();
            Py_RETURN_NONE;
        }
        if (x->dim() != 2 && dim != -1 && dim != x->dim() - 1) Py_RETURN_NONE;
        columns = x->dim() == 2 && dim == 0;
    }
    Tensor output;
    {
        const Tensor input = *x;
        const std::optional<Tensor> given = mask ? std::optional<Tensor>(*mask) : std::nullopt;
        py::gil_scoped_release no_gil;
        output = at::GradMode::is_enabled() && input.requires_grad() ? SoftmaxBackward::apply(input, given, columns)
                                                                     : softmax_forward(input, given, columns);
    }
    return THPVariable_Wrap(std::move(output));
    END_HANDLE_TH_ERRORS
}

Tensor dropout_launch(const Tensor& given, double p, uint64_t seed, uint64_t offset, bool backward) {
    const c10::DeviceGuard device(given.device());
    const Tensor source = given.contiguous();
    const Tensor result = at::empty_like(source);
    if (source.numel() == 0) return result;
    TriRowArgs a{};
    a.struct_size = sizeof(a);
    a.dtype = dtype_code(source.scalar_type());
    a.y_size = 1;
    a.x_size = source.numel();
    a.p = static_cast<float>(p);
    a.seed = seed;
    a.offset = offset;
    a.stream = current_stream(source);
    if (backward) {
        a.grad_output = source.data_ptr();
        a.grad_input = result.data_ptr();
        check(lib.dropout_bwd(&a));
    } else {
        a.input = source.data_ptr();
        a.output = result.data_ptr();
        check(lib.dropout_fwd(&a));
    }
    return result;
}

struct DropoutBackward : torch::autograd::Function<DropoutBackward> {
    static Tensor forward(torch::autograd::AutogradContext* ctx, const Tensor& input, double p, int64_t seed, int64_t offset) {
        ctx->saved_data["p"] = p;
        ctx->saved_data["seed"] = seed;
        ctx->saved_data["offset"] = offset;
        return dropout_launch(input, p, seed, offset, false);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext* ctx, torch::autograd::variable_list grads) {
        const Tensor grad_input = dropout_launch(grads[0], ctx->saved_data["p"].toDouble(), ctx->saved_data["seed"].toInt(),
                                                 ctx->saved_data["offset"].toInt(), true);
        return {grad_input, Tensor(), Tensor(), Tensor()};
    }
};

// dropout(input, p) -> output, or None
PyObject* dropout(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 2, "dropout takes 2 arguments");
    const Tensor* x = plain_tensor(args[0]);
    if (x == nullptr || !on_gpu(*x) || x->numel() == 0 || dtype_code(x->scalar_type()) < 0 || !plain_context()) Py_RETURN_NONE;
    if (!PyFloat_CheckExact(args[1]) && !PyLong_CheckExact(args[1])) Py_RETURN_NONE;
    const double p = PyFloat_AsDouble(args[1]);
    if (p == -1.0 && PyErr_Occurred()) throw python_error();
    PyObject* next_seed = PyDict_GetItemWithError(operation_dict, name_next_seed);
    if (next_seed == nullptr) throw python_error();
    const py::object pair = py::reinterpret_steal<py::object>(PyObject_CallNoArgs(next_seed));
    if (!pair) throw python_error();
    const int64_t seed = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(PyTuple_GetItem(pair.ptr(), 0)));
    const int64_t offset = static_cast<int64_t>(PyLong_AsUnsignedLongLongMask(PyTuple_GetItem(pair.ptr(), 1)));
    if (PyErr_Occurred()) throw python_error();
    Tensor output;
    {
        const Tensor input = *x;
        py::gil_scoped_release no_gil;
        output = at::GradMode::is_enabled() && input.requires_grad() ? DropoutBackward::apply(input, p, seed, offset)
                                                                     : dropout_launch(input, p, seed, offset, false);
    }
    return THPVariable_Wrap(std::move(output));
    END_HANDLE_TH_ERRORS
}

// bind(config module's dict, operation module's dict, {name: address of the library's entry point})
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    TORCH_CHECK(n == 3 && PyDict_Check(args[0]) && PyDict_Check(args[1]) && PyDict_Check(args[2]), "bind takes three dicts");
    auto entry = [&](const char* name, auto& fn) {
        PyObject* v = PyDict_GetItemString(args[2], name);
        TORCH_CHECK(v != nullptr, "no address of ", name);
        fn = reinterpret_cast<std::remove_reference_t<decltype(fn)>>(PyLong_AsVoidPtr(v));
        if (PyErr_Occurred()) throw python_error();
    };
    entry("tri_attn_strerror", lib.strerror);
    entry("tri_attn_fwd", lib.fwd);
    entry("tri_attn_bwd", lib.bwd);
    entry("tri_attn_bwd_dmask", lib.bwd_dmask);
    entry("tri_attn_uses_matrix_cores", lib.uses_matrix_cores);
    entry("tri_attn_workspace_size", lib.workspace_size);
    entry("tri_attn_mask_classes_size", lib.mask_classes_size);
    entry("tri_attn_classify_mask", lib.classify_mask);
    entry("tri_attn_prepare_mask", lib.prepare_mask);
    entry("tri_softmax_fwd", lib.softmax_fwd);
    entry("tri_softmax_bwd", lib.softmax_bwd);
    entry("tri_softmax_workspace_size", lib.softmax_workspace_size);
    entry("tri_dropout_fwd", lib.dropout_fwd);
    entry("tri_dropout_bwd", lib.dropout_bwd);
    Py_INCREF(args[0]);
    Py_INCREF(args[1]);
    config_dict = args[0];
    operation_dict = args[1];
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

PyCFunction fast(PyObject* (*f)(PyObject*, PyObject* const*, Py_ssize_t)) { return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)); }

}  // namespace

PyMODINIT_FUNC PyInit__torch_ops() {
    static PyMethodDef methods[] = {
        {"bind", fast(bind), METH_FASTCALL, nullptr},
        {"attention", fast(attention), METH_FASTCALL, nullptr},
        {"mask_classes", fast(py_mask_classes), METH_FASTCALL, nullptr},
        {"forget_mask_classes", forget_mask_classes, METH_NOARGS, nullptr},
        {"softmax", fast(softmax), METH_FASTCALL, nullptr},
        {"dropout", fast(dropout), METH_FASTCALL, nullptr},
        {nullptr, nullptr, 0, nullptr},
    };
    static PyModuleDef module = {PyModuleDef_HEAD_INIT, "_torch_ops", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};
    name_use_trace = PyUnicode_InternFromString("use_trace");
    name_reference_limits = PyUnicode_InternFromString("reference_limits");
    name_cache = PyUnicode_InternFromString("cache_mask_classes");
    name_pads_from = PyUnicode_InternFromString("_PADS_FROM");
    name_next_seed = PyUnicode_InternFromString("_next_seed");
    return PyModule_Create(&module);
}
