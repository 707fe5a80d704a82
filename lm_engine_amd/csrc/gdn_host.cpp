// The host path of the entry points and of their backward passes: from torch tensors to the calls of the C ABI (include/gdn_hip.h).
//
// On a decode step, a short prompt or a short training sequence the GPU needs a few microseconds per kernel, and reading shapes,
// strides and pointers out of tensors, allocating the results and filling the argument structs takes 10 to 60 in Python per call.
// Here it takes 1 to 6.  Every function is a fast path only: it takes well-formed operands that need no conversion and no
// gradient, and returns None for everything else, so that the Python code behind it converts, differentiates or reports.
// The library itself stays independent of torch: its entry points come in as addresses (bind), from the one loaded copy.

#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <algorithm>
#include <cmath>
#include <initializer_list>

#include "gdn_hip.h"

namespace {

decltype(&gdn_layer_step) layer_step_fn = nullptr;
decltype(&gdn_layer_step_tiles) layer_step_tiles_fn = nullptr;
decltype(&gdn_causal_conv1d_fwd) conv_fn = nullptr;
decltype(&gdn_gates_fwd) gates_fn = nullptr;
decltype(&gdn_gated_rmsnorm_fwd) norm_fn = nullptr;
decltype(&gdn_recurrent_fwd) recurrent_fn = nullptr;
decltype(&gdn_chunk_fwd) chunk_fn = nullptr;
decltype(&gdn_workspace_bytes) workspace_bytes_fn = nullptr;
decltype(&gdn_chunk_fwd_is_one_launch) one_launch_fn = nullptr;
decltype(&gdn_chunk_bwd_sweeps) sweeps_fn = nullptr;
decltype(&gdn_chunk_bwd_sweeps_workspace_bytes) sweeps_workspace_fn = nullptr;
decltype(&gdn_chunk_bwd_local) local_fn = nullptr;
decltype(&gdn_causal_conv1d_bwd) conv_bwd_fn = nullptr;
decltype(&gdn_gates_bwd) gates_bwd_fn = nullptr;
decltype(&gdn_gated_rmsnorm_bwd) norm_bwd_fn = nullptr;
decltype(&gdn_column_sums) column_sums_fn = nullptr;
decltype(&gdn_fold_heads) fold_heads_fn = nullptr;
decltype(&gdn_layer_front) layer_front_fn = nullptr;
PyObject* check_status = nullptr;  // _lib.check_status: raises what a status stands for

// bind(check_status, addresses...)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    void** slots[] = {(void**)&layer_step_fn, (void**)&layer_step_tiles_fn, (void**)&conv_fn, (void**)&gates_fn, (void**)&norm_fn,
                      (void**)&recurrent_fn, (void**)&chunk_fn, (void**)&workspace_bytes_fn, (void**)&one_launch_fn,
                      (void**)&sweeps_fn, (void**)&sweeps_workspace_fn, (void**)&local_fn, (void**)&conv_bwd_fn, (void**)&gates_bwd_fn,
                      (void**)&norm_bwd_fn, (void**)&column_sums_fn, (void**)&fold_heads_fn, (void**)&layer_front_fn};
    constexpr Py_ssize_t count = sizeof(slots) / sizeof(slots[0]);
    if (n != count + 1) return PyErr_Format(PyExc_TypeError, "bind takes a function and %zd addresses, got %zd arguments", count, n);
    for (Py_ssize_t i = 0; i < count; i++) {
        *slots[i] = PyLong_AsVoidPtr(args[i + 1]);
        if (PyErr_Occurred()) return nullptr;
    }
    Py_XDECREF(check_status);
    check_status = Py_NewRef(args[0]);
    Py_RETURN_NONE;
}

// What disqualifies an operand ends the fast path: the caller's Python code takes over.
struct NotHere {};
void need(bool ok) {
    if (!ok) throw NotHere{};
}

// The operands of one call: all on one device, which is the current one, plain tensors, no gradient wanted.
struct Operands {
    c10::Device device{c10::DeviceType::CPU};
    bool grad = c10::GradMode::is_enabled();

    const at::Tensor& operator()(PyObject* x) {
        need(THPVariable_Check(x));
        const at::Tensor& t = THPVariable_Unpack(x);
        need(t.defined() && t.device().type() == c10::DeviceType::CUDA && !(grad && t.requires_grad()) && t.layout() == at::kStrided);
        need(!t.unsafeGetTensorImpl()->key_set().has(c10::DispatchKey::Python) && t.unsafeGetTensorImpl()->has_storage() && !t.is_conj() && !t.is_neg());
        if (device.type() == c10::DeviceType::CPU) {
            device = t.device();
            need(c10::impl::VirtualGuardImpl(c10::DeviceType::CUDA).getDevice().index() == device.index());
        }
        need(t.device() == device);
        return t;
    }
    const at::Tensor* optional(PyObject* x) { return x == Py_None ? nullptr : &(*this)(x); }
};

int32_t code_of(const at::Tensor& t) {
    if (t.scalar_type() == at::kBFloat16) return GDN_BF16;
    need(t.scalar_type() == at::kFloat);
    return GDN_F32;
}
// Runs `body`, which touches no Python object, while other Python threads may run: around the allocations of a call, which
// may wait for the device, and around the library's entry point.
template <typename F>
auto without_interpreter_lock(F&& body) {
    struct Released {
        PyThreadState* const state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
    } released;
    return body();
}

void* ptr(const at::Tensor& t) { return t.data_ptr(); }
void* ptr(const at::Tensor* t) { return t == nullptr ? nullptr : t->data_ptr(); }
bool aligned(const void* p, size_t n) { return reinterpret_cast<uintptr_t>(p) % n == 0; }
int64_t integer(PyObject* x) {
    const int64_t v = PyLong_AsLongLong(x);
    if (v == -1 && PyErr_Occurred()) PyErr_Clear(), need(false);
    return v;
}
double number(PyObject* x) {
    const double v = PyFloat_AsDouble(x);
    if (v == -1.0 && PyErr_Occurred()) PyErr_Clear(), need(false);
    return v;
}
bool truth(PyObject* x) { return PyObject_IsTrue(x) == 1; }
void* stream_of(PyObject* x) { return reinterpret_cast<void*>(integer(x)); }
int32_t size32(int64_t n) {
    need(n >= 0 && n <= INT32_MAX);
    return (int32_t)n;
}

// [.., width] as rows with one stride between them, when the leading dims collapse
int64_t row_stride(const at::Tensor& t, int64_t width) {
    const int64_t d = t.dim();
    need(d >= 2 && t.size(d - 1) == width && (t.stride(d - 1) == 1 || width == 1));
    int64_t stride = 0, count = 1;  // of the rows so far, from the innermost dim out
    for (int64_t i = d - 2; i >= 0; i--) {
        if (t.size(i) == 1) continue;
        if (count == 1) stride = t.stride(i);
        else need(t.stride(i) == stride * count);
        count *= t.size(i);
    }
    return count > 1 ? stride : width;
}

// taps per channel of a convolution weight [C, 1, taps] or [C, taps]
int64_t taps_of(const at::Tensor& weight, int64_t C) {
    const int64_t d = weight.dim();
    need((d == 2 || (d == 3 && weight.size(1) == 1)) && weight.size(0) == C && weight.is_contiguous());
    const int64_t taps = weight.size(d - 1);
    need(taps >= 2 && taps <= 4);
    return taps;
}

template <typename F>
PyObject* fast_path(Py_ssize_t n, Py_ssize_t wanted, F&& body) {
    if (n != wanted) return PyErr_Format(PyExc_TypeError, "takes %zd arguments, got %zd", wanted, n);
    try {
        return body();
    } catch (const NotHere&) {
    } catch (const std::exception&) {  // (out of memory, say: the Python path meets it too and raises torch's own error)
    }
    Py_RETURN_NONE;
}

PyObject* pack_results(std::initializer_list<at::Tensor> tensors) {
    PyObject* out = PyTuple_New((Py_ssize_t)tensors.size());
    if (out == nullptr) return nullptr;
    Py_ssize_t i = 0;
    for (const at::Tensor& t : tensors) {
        PyObject* x = t.defined() ? THPVariable_Wrap(t) : Py_NewRef(Py_None);
        if (x == nullptr) {
            Py_DECREF(out);
            return nullptr;
        }
        PyTuple_SET_ITEM(out, i++, x);
    }
    return out;
}

// The last step of a call: launches and hands the results on, which it takes over.  They are made before the launch, so that
// nothing can fail behind it.  A refused argument (a negative status: nothing was launched) ends the fast path.  A HIP error
// (positive) may be that of an earlier call beside a launch that did go through: it is raised, the call is never tried again.
template <typename F>
PyObject* launch(const char* what, PyObject* made, F&& entry) {
    THPObjectPtr results(made);
    if (!results) return nullptr;
    const int status = without_interpreter_lock(entry);
    if (status == GDN_OK) return results.release();
    need(status > 0);
    return PyObject_CallFunction(check_status, "is", status, what);
}

at::Tensor fresh(const at::Tensor& like, at::IntArrayRef sizes) { return at::empty(sizes, like.options()); }
at::Tensor fresh_f32(const at::Tensor& like, at::IntArrayRef sizes) { return at::empty(sizes, like.options().dtype(at::kFloat)); }

// layer_step(stream, qkv, a, b, gate, conv_weight, conv_bias, A_log, dt_bias, norm_weight, eps, HK, H, K, V, conv_state, h,
//            beta_scale, scale, activation, workspace) -> (o [B, 1, H V], conv_state, h)
// workspace(pairs, V) -> (owner, tickets, scratch): called when more than one workgroup works on a head
PyObject* layer_step(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 21, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &qkv = operand(args[1]), &a = operand(args[2]), &b = operand(args[3]), &weight = operand(args[5]);
        const at::Tensor &A_log = operand(args[7]), &dt_bias = operand(args[8]);
        const at::Tensor *gate = operand.optional(args[4]), *bias = operand.optional(args[6]), *norm_w = operand.optional(args[9]);
        const at::Tensor *conv_state = operand.optional(args[15]), *h0 = operand.optional(args[16]);
        gdn_layer_step_args s{};
        const int64_t HK = integer(args[11]), H = integer(args[12]), K = integer(args[13]), V = integer(args[14]);
        need(HK > 0 && H > 0 && K > 0 && V > 0 && H % HK == 0 && V <= 512 && V % 32 == 0 && (K == 64 || K == 128 || K == 256));
        const int64_t C = 2 * HK * K + H * V;
        s.dtype = code_of(qkv);
        need(qkv.dim() == 3 && qkv.size(1) == 1 && qkv.size(2) == C && qkv.stride(2) == 1 && C % (s.dtype == GDN_BF16 ? 8 : 4) == 0);
        const int64_t B = qkv.size(0);
        need(B > 0 && B <= 65535 && H <= 65535);
        const at::Tensor* scalars[] = {&a, &b};
        for (const at::Tensor* t : scalars)
            need(t->scalar_type() == qkv.scalar_type() && t->dim() == 3 && t->size(0) == B && t->size(1) == 1 && t->size(2) == H && (t->stride(2) == 1 || H == 1));
        const at::Tensor* decay[] = {&A_log, &dt_bias};
        for (const at::Tensor* t : decay) need(t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == H && t->is_contiguous());
        const int64_t ks = taps_of(weight, C);
        s.conv_w_dtype = code_of(weight);
        need(s.dtype == GDN_BF16 || s.conv_w_dtype == GDN_F32);
        // (the kernel reads by elements; what the convolution and the norm on their own refuse for its place in memory goes to them)
        const int64_t vec = s.dtype == GDN_BF16 ? 8 : 4;
        need(aligned(ptr(qkv), 16) && qkv.stride(0) % vec == 0 && qkv.stride(1) % vec == 0 && qkv.stride(1) >= C && aligned(ptr(weight), 16));
        need(aligned(ptr(bias), 16) && aligned(ptr(norm_w), 16));
        if (bias != nullptr) need(bias->scalar_type() == weight.scalar_type() && bias->dim() == 1 && bias->size(0) == C && bias->is_contiguous());
        if (conv_state != nullptr) need(conv_state->scalar_type() == qkv.scalar_type() && conv_state->sizes() == at::IntArrayRef({B, C, ks - 1}) && conv_state->is_contiguous());
        if (h0 != nullptr) need(h0->scalar_type() == at::kFloat && h0->sizes() == at::IntArrayRef({B, H, K, V}) && h0->is_contiguous() && aligned(ptr(h0), 16));
        if (gate != nullptr) {
            need(gate->scalar_type() == qkv.scalar_type() && gate->dim() == 3 && gate->size(0) == B && gate->size(1) == 1 && gate->size(2) == H * V && gate->stride(2) == 1);
            s.gate_stride_b = gate->stride(0);
        }
        s.norm_w_dtype = s.dtype;
        if (norm_w != nullptr) {
            s.norm_w_dtype = code_of(*norm_w);
            need(norm_w->dim() == 1 && norm_w->size(0) == V && norm_w->is_contiguous());
        }
        s.B = (int32_t)B, s.HK = size32(HK), s.H = (int32_t)H, s.K = (int32_t)K, s.V = (int32_t)V, s.kernel_size = (int32_t)ks;
        THPObjectPtr workspace;  // keeps it alive until the launch is in the stream
        if (layer_step_tiles_fn(s.B, s.H, s.V) > 1) {
            workspace = PyObject_CallFunction(args[20], "LL", (long long)(B * H), (long long)V);
            if (!workspace) return nullptr;
            s.tickets = static_cast<int32_t*>(PyLong_AsVoidPtr(PyTuple_GetItem(workspace.get(), 1)));
            s.scratch = static_cast<float*>(PyLong_AsVoidPtr(PyTuple_GetItem(workspace.get(), 2)));
        }
        at::Tensor out, state_out, ht;
        without_interpreter_lock([&] { out = fresh(qkv, {B, 1, H * V}), state_out = fresh(qkv, {B, C, ks - 1}), ht = fresh_f32(qkv, {B, H, K, V}); });
        s.qkv = ptr(qkv), s.conv_weight = ptr(weight), s.conv_bias = ptr(bias), s.conv_state = ptr(conv_state), s.conv_state_out = ptr(state_out);
        s.a = ptr(a), s.b = ptr(b), s.A_log = static_cast<const float*>(ptr(A_log)), s.dt_bias = static_cast<const float*>(ptr(dt_bias));
        s.h0 = static_cast<const float*>(ptr(h0)), s.ht = static_cast<float*>(ptr(ht)), s.gate = ptr(gate), s.norm_weight = ptr(norm_w), s.out = ptr(out);
        s.qkv_stride_b = qkv.stride(0), s.a_stride_b = a.stride(0), s.b_stride_b = b.stride(0);
        s.beta_scale = (float)number(args[17]), s.scale = (float)number(args[18]), s.eps = (float)number(args[10]);
        s.activation = (int32_t)integer(args[19]);
        return launch("gdn_layer_step", pack_results({out, state_out, ht}), [&] { return layer_step_fn(&s, stream); });
    });
}

// the convolution's arguments, but for its mask and results: (batch, tokens, channels, taps)
struct ConvOperands {
    gdn_conv_args s{};
    int64_t B, S, C, ks;
    ConvOperands(const at::Tensor& x, const at::Tensor& weight, const at::Tensor* bias, const at::Tensor* state, PyObject* activation) {
        s.dtype = code_of(x), s.w_dtype = code_of(weight);
        need(x.dim() == 3 && x.stride(2) == 1 && (s.dtype == GDN_BF16 || s.w_dtype == GDN_F32));
        B = x.size(0), S = x.size(1), C = x.size(2), ks = taps_of(weight, C);
        need(B > 0 && S > 0);
        if (bias != nullptr) need(bias->scalar_type() == weight.scalar_type() && bias->dim() == 1 && bias->size(0) == C && bias->is_contiguous());
        if (state != nullptr) need(state->scalar_type() == x.scalar_type() && state->sizes() == at::IntArrayRef({B, C, ks - 1}) && state->is_contiguous());
        s.x = ptr(x), s.weight = ptr(weight), s.bias = ptr(bias), s.input_state = ptr(state);
        s.x_stride_b = x.stride(0), s.x_stride_s = x.stride(1), s.y_stride_b = S * C, s.y_stride_s = C;
        s.B = size32(B), s.S = size32(S), s.C = size32(C), s.kernel_size = (int32_t)ks;
        s.activation = (int32_t)integer(activation);
    }
    void results(const at::Tensor& x, bool output_state, at::Tensor& y, at::Tensor& final_state) {
        y = fresh(x, {B, S, C}), s.y = ptr(y);
        if (output_state) final_state = fresh(x, {B, C, ks - 1}), s.final_state = ptr(final_state);
    }
};

// conv(stream, x, weight, bias, input_state, mask, output_state, activation) -> (y, final_state or None)
PyObject* conv(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 8, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &x = operand(args[1]), &weight = operand(args[2]);
        const at::Tensor *bias = operand.optional(args[3]), *state = operand.optional(args[4]), *mask = operand.optional(args[5]);
        ConvOperands c(x, weight, bias, state, args[7]);
        at::Tensor kept_mask;
        bool masked = false;
        if (mask != nullptr) need(mask->dim() == 2);
        if (mask != nullptr && mask->size(0) > 1 && mask->size(1) > 1) {
            need(mask->size(0) == c.B && mask->size(1) == c.S);
            masked = true;
        }
        const bool output_state = truth(args[6]);
        at::Tensor y, final_state;
        without_interpreter_lock([&] {
            if (masked) kept_mask = mask->to(x.scalar_type()).contiguous(), c.s.mask = ptr(kept_mask);
            c.results(x, output_state, y, final_state);
        });
        return launch("gdn_causal_conv1d_fwd", pack_results({y, final_state}), [&] { return conv_fn(&c.s, stream); });
    });
}

// the gates' arguments, but for their results
gdn_gate_args gate_args(const at::Tensor& a, const at::Tensor& b, const at::Tensor& A_log, const at::Tensor& dt_bias, PyObject* beta_scale) {
    gdn_gate_args s{};
    s.dtype = code_of(a);
    need(a.dim() >= 2 && b.scalar_type() == a.scalar_type() && b.sizes() == a.sizes() && a.numel() > 0);
    const int64_t H = a.size(-1);
    const at::Tensor* decay[] = {&A_log, &dt_bias};
    for (const at::Tensor* t : decay) need(t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == H && t->is_contiguous());
    s.a_stride = row_stride(a, H), s.b_stride = row_stride(b, H);
    s.tokens = a.numel() / H, s.H = size32(H);
    s.a = ptr(a), s.b = ptr(b), s.A_log = static_cast<const float*>(ptr(A_log)), s.dt_bias = static_cast<const float*>(ptr(dt_bias));
    s.beta_scale = (float)number(beta_scale);
    return s;
}

// gates(stream, a, b, A_log, dt_bias, beta_scale) -> (g, beta)
PyObject* gates(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 6, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &a = operand(args[1]), &b = operand(args[2]), &A_log = operand(args[3]), &dt_bias = operand(args[4]);
        gdn_gate_args s = gate_args(a, b, A_log, dt_bias, args[5]);
        at::Tensor g, beta;
        without_interpreter_lock([&] { g = fresh_f32(a, a.sizes()), beta = fresh(a, a.sizes()); });
        s.g = static_cast<float*>(ptr(g)), s.beta = ptr(beta);
        return launch("gdn_gates_fwd", pack_results({g, beta}), [&] { return gates_fn(&s, stream); });
    });
}

// layer_front(stream, qkv, weight, bias, input_state, mask, output_state, activation, a, b, A_log, dt_bias, beta_scale)
//   -> (y, final_state or None, g, beta, prefix sums of the mask's rows or None)
// The convolution and the gates in one launch.  mask: [B, S] of integers or None.
PyObject* layer_front(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 13, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &x = operand(args[1]), &weight = operand(args[2]), &a = operand(args[8]), &b = operand(args[9]), &A_log = operand(args[10]), &dt_bias = operand(args[11]);
        const at::Tensor *bias = operand.optional(args[3]), *state = operand.optional(args[4]), *mask = operand.optional(args[5]);
        ConvOperands c(x, weight, bias, state, args[7]);
        gdn_gate_args s = gate_args(a, b, A_log, dt_bias, args[12]);
        need(s.dtype == c.s.dtype);
        int element_bytes = 0;
        if (mask != nullptr) {
            // (the masks that _one_launch_mask takes, layer_ops.py)
            need(mask->dim() == 2 && mask->size(0) == c.B && mask->size(1) == c.S && c.B <= 64 && c.B * c.S <= 1 << 16);
            const at::ScalarType type = mask->scalar_type();
            need(type == at::kLong || type == at::kInt || type == at::kByte || type == at::kBool);
            element_bytes = (int)mask->element_size();
        }
        const bool output_state = truth(args[6]);
        at::Tensor y, final_state, g, beta, prefix;
        without_interpreter_lock([&] {
            c.results(x, output_state, y, final_state);
            g = fresh_f32(a, a.sizes()), beta = fresh(a, a.sizes());
            if (mask != nullptr) prefix = at::empty({c.B + 1}, x.options().dtype(at::kInt));
        });
        s.g = static_cast<float*>(ptr(g)), s.beta = ptr(beta);
        return launch("gdn_layer_front", pack_results({y, final_state, g, beta, prefix}), [&] {
            return layer_front_fn(&c.s, &s, ptr(mask), element_bytes, mask == nullptr ? 0 : mask->stride(0), mask == nullptr ? 0 : mask->stride(1),
                                  prefix.defined() ? static_cast<int32_t*>(ptr(prefix)) : nullptr, stream);
        });
    });
}

// o and gate of the gated norm, forward and backward: (heads, columns, elements between the gate's tokens)
struct NormOperands {
    int64_t H, V, gate_stride = 0;
    NormOperands(const at::Tensor& o, const at::Tensor* gate) {
        need(o.dim() >= 2 && o.is_contiguous() && o.numel() > 0);
        H = o.size(-2), V = o.size(-1);
        need(V % 8 == 0 && V <= 512);
        if (gate == nullptr) return;
        need(gate->scalar_type() == o.scalar_type() && gate->numel() == o.numel() && gate->dim() >= 2);
        if (gate->size(-1) == H * V && gate->dim() == o.dim() - 1) {
            gate_stride = row_stride(*gate, H * V);
        } else {
            need(gate->sizes() == o.sizes() && gate->is_contiguous());
            gate_stride = H * V;
        }
    }
};

// norm(stream, o, gate, weight, eps) -> y
PyObject* norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 5, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor& o = operand(args[1]);
        const at::Tensor *gate = operand.optional(args[2]), *weight = operand.optional(args[3]);
        gdn_norm_args s{};
        s.dtype = code_of(o);
        const NormOperands x(o, gate);
        const int64_t H = x.H, V = x.V;
        s.tokens = o.numel() / (H * V), s.gate_stride_t = x.gate_stride;
        s.w_dtype = GDN_F32;
        if (weight != nullptr) {
            s.w_dtype = code_of(*weight);
            need(weight->dim() == 1 && weight->size(0) == V && weight->is_contiguous());
        }
        s.w_dtype |= GDN_NORM_GATE_DWORDS;
        const at::Tensor y = without_interpreter_lock([&] { return fresh(o, o.sizes()); });
        s.o = ptr(o), s.gate = ptr(gate), s.weight = ptr(weight), s.y = ptr(y);
        s.o_stride_t = s.y_stride_t = H * V, s.H = size32(H), s.V = (int32_t)V, s.eps = (float)number(args[4]);
        return launch("gdn_gated_rmsnorm_fwd", THPVariable_Wrap(y), [&] { return norm_fn(&s, stream); });
    });
}

// delta_rule(stream, chunked, q, k, v, g, beta, scale or None, initial_state, output_final_state, cu_seqlens, flags, inplace)
//   -> (o, final_state or None)
// flags: GDN_FLAG_*.  Not here: what runs as one launch (its workspaces are kept by the Python side) and empty tensors.
PyObject* delta_rule(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 13, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const bool chunked = truth(args[1]), output_final = truth(args[9]), inplace = truth(args[12]);
        const at::Tensor &q = operand(args[2]), &k = operand(args[3]), &v = operand(args[4]);
        const at::Tensor *g = operand.optional(args[5]), *beta = operand.optional(args[6]), *h0 = operand.optional(args[8]), *cu = operand.optional(args[10]);
        gdn_args s{};
        s.dtype = code_of(q), s.flags = (int32_t)integer(args[11]);
        const bool padded = (s.flags & GDN_FLAG_LEFT_PADDED) != 0;
        need(q.dim() == 4 && k.sizes() == q.sizes() && v.dim() == 4 && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type());
        const int64_t B = q.size(0), T = q.size(1), HK = q.size(2), K = q.size(3), H = v.size(2), V = v.size(3);
        need(v.size(0) == B && v.size(1) == T && B > 0 && T > 0 && HK > 0 && H > 0 && H % HK == 0 && q.stride(3) == 1 && k.stride(3) == 1 && v.stride(3) == 1);
        int64_t N = B;
        if (padded) need(cu != nullptr && cu->dim() == 1 && cu->numel() == B + 1);
        else if (cu != nullptr) {
            need(B == 1 && cu->dim() == 1 && cu->numel() >= 2);
            N = cu->numel() - 1;
        }
        if (cu != nullptr) need(cu->scalar_type() == at::kInt && cu->is_contiguous());
        if (g != nullptr) need(g->scalar_type() == at::kFloat && g->sizes() == at::IntArrayRef({B, T, H}) && g->is_contiguous());
        s.beta_dtype = GDN_F32;
        if (beta != nullptr) {
            s.beta_dtype = code_of(*beta);
            need(beta->sizes() == at::IntArrayRef({B, T, H}) && beta->is_contiguous());
        }
        if (h0 != nullptr) need(h0->scalar_type() == at::kFloat && h0->sizes() == at::IntArrayRef({N, H, K, V}) && h0->is_contiguous());
        s.B = size32(B), s.T = size32(T), s.H = size32(H), s.K = size32(K), s.V = size32(V), s.N = size32(N), s.chunk = 64;
        s.qk_heads = HK == H ? 0 : (int32_t)HK;
        s.cu_seqlens = static_cast<const int32_t*>(ptr(cu));
        uint64_t workspace_bytes = 0;
        if (chunked) {
            need(s.dtype == GDN_BF16 && one_launch_fn(&s) == 0);
            workspace_bytes = workspace_bytes_fn(&s);
            need(workspace_bytes > 0);
        }
        at::Tensor workspace, o, ht;
        if (output_final && inplace) need(h0 != nullptr), ht = *h0, s.flags |= GDN_FLAG_STATE_INPLACE;
        without_interpreter_lock([&] {
            if (chunked) workspace = at::empty({(int64_t)workspace_bytes}, q.options().dtype(at::kByte)), s.workspace = ptr(workspace), s.workspace_bytes = workspace_bytes;
            // (padding positions of a left-padded batch read as zeros: gdn_chunk_fwd writes them on request, the token kernels do not)
            if (padded && chunked) s.flags |= GDN_FLAG_ZERO_PADDING;
            o = padded && !chunked ? at::zeros({B, T, H, V}, v.options()) : fresh(v, {B, T, H, V});
            if (output_final && !inplace) ht = fresh_f32(v, {N, H, K, V});
        });
        if (output_final) s.ht = static_cast<float*>(ptr(ht));
        s.q = ptr(q), s.k = ptr(k), s.v = ptr(v), s.beta = ptr(beta), s.o = ptr(o);
        s.g = static_cast<const float*>(ptr(g)), s.h0 = static_cast<const float*>(ptr(h0));
        s.q_stride_b = q.stride(0), s.q_stride_t = q.stride(1), s.q_stride_h = q.stride(2);
        s.k_stride_b = k.stride(0), s.k_stride_t = k.stride(1), s.k_stride_h = k.stride(2);
        s.v_stride_b = v.stride(0), s.v_stride_t = v.stride(1), s.v_stride_h = v.stride(2);
        s.o_stride_b = o.stride(0), s.o_stride_t = o.stride(1), s.o_stride_h = o.stride(2);
        s.scale = args[7] == Py_None ? (float)std::pow((double)K, -0.5) : (float)number(args[7]);
        THPObjectPtr results(pack_results({o, ht}));
        if (results && output_final && inplace) PyTuple_SetItem(results.get(), 1, Py_NewRef(args[8]));  // the caller's own tensor object
        return launch(chunked ? "gdn_chunk_fwd" : "gdn_recurrent_fwd", results.release(),
                      [&] { return (chunked ? chunk_fn : recurrent_fn)(&s, stream); });
    });
}

// ---- backward passes.  Like the forward: what needs a conversion or a copy, and what is itself differentiated, is not here. ----

// the sums over the first dim of one or two partial arrays, in the dtypes of the parameters they are the gradients of
struct ColumnSums {
    gdn_column_sums_args s{};
    void add(const at::Tensor& partial, const at::Tensor& out) {
        const int j = s.arrays++;
        s.partial[j] = static_cast<const float*>(ptr(partial)), s.out[j] = ptr(out), s.cols[j] = out.numel(), s.out_dtype[j] = code_of(out);
        s.rows = (int32_t)partial.size(0);
    }
};

// a gradient that a kernel reads as it lies: what kernel_rows (_autograd.py) would not copy
void need_rows(const at::Tensor& t, int64_t stride_elements, size_t address_bytes) {
    need(t.stride(-1) == 1 && aligned(ptr(t), address_bytes));
    for (int64_t i = 0; i + 1 < t.dim(); i++) need(t.stride(i) % stride_elements == 0);
}

// delta_rule_bwd(stream, q, k, v, g, beta, initial_state, cu_seqlens, do, dht, scale, flags, seq_start, seq_len, NC, tokens, joined)
//   -> (dq, dk, dv, dg, dbeta, dh0)
// Rows of a batch: without seq_start and seq_len.  Else NC chunks for the longest sequence; tokens: how many belong to one.
// joined: dq, dk and dv as column blocks of one tensor, where v has no more heads than q and k.
PyObject* delta_rule_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 17, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &q = operand(args[1]), &k = operand(args[2]), &v = operand(args[3]), &d = operand(args[8]);
        const at::Tensor *g = operand.optional(args[4]), *beta = operand.optional(args[5]), *h0 = operand.optional(args[6]), *cu = operand.optional(args[7]);
        const at::Tensor *dht = operand.optional(args[9]), *seq_start = operand.optional(args[12]), *seq_len = operand.optional(args[13]);
        const int64_t tokens = integer(args[15]);
        const bool joined = truth(args[16]);
        gdn_args s{};
        gdn_chunk_local_args l{};
        s.dtype = code_of(q), s.flags = (int32_t)integer(args[11]);
        const bool padded = (s.flags & GDN_FLAG_LEFT_PADDED) != 0;
        need(s.dtype == GDN_BF16 && q.dim() == 4 && k.sizes() == q.sizes() && v.dim() == 4 && k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type());
        const int64_t B = q.size(0), T = q.size(1), HK = q.size(2), K = q.size(3), H = v.size(2), V = v.size(3);
        need(v.size(0) == B && v.size(1) == T && B > 0 && T > 0 && HK > 0 && H > 0 && H % HK == 0 && H / HK < 0x8000 && q.stride(3) == 1 && k.stride(3) == 1 && v.stride(3) == 1);
        need((K == 64 || K == 128 || K == 256) && V % 64 == 0);
        need(d.scalar_type() == at::kBFloat16 && d.sizes() == v.sizes() && d.stride(1) <= (int64_t)1 << 24);
        need_rows(d, 8, 16);
        int64_t N = B, NC = (T + 63) / 64;
        need((cu == nullptr) == (seq_start == nullptr) && (cu == nullptr) == (seq_len == nullptr));
        if (cu != nullptr) {
            need(cu->scalar_type() == at::kInt && cu->dim() == 1 && cu->is_contiguous() && cu->numel() >= 2);
            if (padded) need(cu->numel() == B + 1);
            else need(B == 1), N = cu->numel() - 1;
            NC = integer(args[14]);
            const at::Tensor* places[] = {seq_start, seq_len};
            for (const at::Tensor* t : places) need(t->scalar_type() == at::kInt && t->dim() == 1 && t->numel() == N && t->is_contiguous());
            l.seq_start = static_cast<const int32_t*>(ptr(seq_start)), l.seq_len = static_cast<const int32_t*>(ptr(seq_len));
        } else {
            need(!padded);
        }
        need(NC > 0 && tokens >= 0 && tokens <= B * T);
        const bool covers = tokens == B * T;
        l.T_rows = size32(T);
        if (g != nullptr) need(g->scalar_type() == at::kFloat && g->sizes() == at::IntArrayRef({B, T, H}) && g->is_contiguous());
        s.beta_dtype = GDN_F32;
        if (beta != nullptr) {
            s.beta_dtype = code_of(*beta);
            need(beta->sizes() == at::IntArrayRef({B, T, H}) && beta->is_contiguous());
        }
        const at::Tensor* states[] = {h0, dht};
        for (const at::Tensor* t : states)
            if (t != nullptr) need(t->scalar_type() == at::kFloat && t->sizes() == at::IntArrayRef({N, H, K, V}) && t->is_contiguous() && aligned(ptr(t), 16));
        s.B = size32(B), s.T = size32(T), s.H = size32(H), s.K = (int32_t)K, s.V = size32(V), s.N = size32(N), s.chunk = 64;
        if (cu != nullptr && !padded && !covers) s.T = std::max((int32_t)tokens, 1);  // (tokens behind the last sequence are no work to count on)
        s.qk_heads = HK == H ? 0 : (int32_t)HK;
        s.cu_seqlens = static_cast<const int32_t*>(ptr(cu));
        s.scale = (float)number(args[10]);
        s.q = ptr(q), s.k = ptr(k), s.v = ptr(v), s.o = ptr(v), s.beta = ptr(beta);  // (no output is written)
        s.g = static_cast<const float*>(ptr(g)), s.h0 = static_cast<const float*>(ptr(h0));
        s.q_stride_b = l.q_stride_b = q.stride(0), s.q_stride_t = l.q_stride_t = q.stride(1), s.q_stride_h = l.q_stride_h = q.stride(2);
        s.k_stride_b = l.k_stride_b = k.stride(0), s.k_stride_t = l.k_stride_t = k.stride(1), s.k_stride_h = l.k_stride_h = k.stride(2);
        s.v_stride_b = l.v_stride_b = v.stride(0), s.v_stride_t = l.v_stride_t = v.stride(1), s.v_stride_h = l.v_stride_h = v.stride(2);
        s.o_stride_b = s.v_stride_b, s.o_stride_t = s.v_stride_t, s.o_stride_h = s.v_stride_h;
        s.workspace_bytes = sweeps_workspace_fn(&s);
        need(s.workspace_bytes > 0);

        at::Tensor workspace, scalars, S0, dS1, Vn, Y, dq, dk, dv, dg, dbeta, dh0;
        at::Tensor dq_each, dk_each;  // per value head, where value heads share those of q and k
        without_interpreter_lock([&] {
            scalars = fresh_f32(q, {4, N * H, NC, 64});
            S0 = fresh(q, {N * H, NC, K, V}), dS1 = fresh(q, {N * H, NC, K, V}), Vn = fresh(q, {N * H, NC, 64, V}), Y = fresh(q, {N * H, NC, 64, V});
            if (h0 != nullptr) dh0 = fresh_f32(q, {N, H, K, V});
            workspace = at::empty({(int64_t)s.workspace_bytes}, q.options().dtype(at::kByte));
        });
        s.workspace = ptr(workspace);
        float* const f = static_cast<float*>(ptr(scalars));
        const int64_t each = N * H * NC * 64;
        l.gamma = f, l.beta = f + each, l.rq = f + 2 * each, l.rk = f + 3 * each;
        l.states = ptr(S0), l.dstates = ptr(dS1), l.v_new = ptr(Vn), l.y_chunks = ptr(Y);
        l.saves_dtype = l.dstates_dtype = GDN_BF16, l.saves_sliced = 1;
        l.chunks = N * H * NC, l.K = (int32_t)K, l.V = (int32_t)V, l.H = (int32_t)H, l.NC = size32(NC), l.scale = s.scale;
        l.q_raw = s.q, l.k_raw = s.k, l.v_raw = s.v, l.dout_raw = ptr(d);
        l.dout_stride_b = d.stride(0), l.dout_stride_t = d.stride(1), l.dout_stride_h = d.stride(2);
        const int status = without_interpreter_lock([&] {
            return sweeps_fn(&s, &l, static_cast<const float*>(ptr(dht)), dh0.defined() ? static_cast<float*>(ptr(dh0)) : nullptr, stream);
        });
        need(status >= 0);
        if (status != GDN_OK) return PyObject_CallFunction(check_status, "is", status, "gdn_chunk_bwd_sweeps");

        // The results are allocated behind the sweeps' launch, where the workspace can go: they then take its place, in memory and
        // in the caches (4 x 4096 tokens, 16 heads, K = V = 128: the chunk-local kernel 208 us, 216 beside the workspace).  Should an
        // allocation fail here, the Python path starts over: nothing so far has changed an operand.
        without_interpreter_lock([&] {
            workspace.reset();
            // tokens outside every sequence are not written
            auto made = [&](at::IntArrayRef sizes, at::ScalarType dtype) {
                return covers || cu == nullptr ? at::empty(sizes, q.options().dtype(dtype)) : at::zeros(sizes, q.options().dtype(dtype));
            };
            if (HK != H) dq_each = made({B, T, H, K}, at::kBFloat16), dk_each = made({B, T, H, K}, at::kBFloat16);
            if (joined && HK == H) {
                const int64_t row = H * (2 * K + V);
                const at::Tensor rows = made({B, T, row}, at::kBFloat16);
                dq = rows.as_strided({B, T, H, K}, {T * row, row, K, 1}, 0);
                dk = rows.as_strided({B, T, H, K}, {T * row, row, K, 1}, H * K);
                dv = rows.as_strided({B, T, H, V}, {T * row, row, V, 1}, 2 * H * K);
                l.out_stride_t = size32(row);
            } else {
                dq = made({B, T, HK, K}, at::kBFloat16), dk = made({B, T, HK, K}, at::kBFloat16), dv = made({B, T, H, V}, at::kBFloat16);
            }
            dg = made({B, T, H}, at::kFloat), dbeta = made({B, T, H}, beta == nullptr ? at::kFloat : beta->scalar_type());
        });
        l.dq_out = ptr(dq), l.dk_out = ptr(dk), l.dv_out = ptr(dv), l.dg_out = static_cast<float*>(ptr(dg)), l.dbeta_out = static_cast<float*>(ptr(dbeta));
        if (!(s.flags & GDN_FLAG_L2NORM)) l.rq = l.rk = nullptr;
        if (dbeta.scalar_type() == at::kBFloat16) l.saves_dtype |= GDN_LOCAL_DBETA_BF16;
        if (seq_start == nullptr) l.saves_dtype |= GDN_LOCAL_RAGGED_ROWS;
        if (HK != H) l.saves_dtype |= GDN_LOCAL_SHARED_HEADS((int32_t)(H / HK)), l.dq_out = ptr(dq_each), l.dk_out = ptr(dk_each);
        return launch("gdn_chunk_bwd_local", pack_results({dq, dk, dv, g == nullptr ? at::Tensor() : dg, beta == nullptr ? at::Tensor() : dbeta, dh0}), [&] {
            const int status = local_fn(&l, stream);
            if (status != GDN_OK || HK == H) return status;
            return fold_heads_fn(l.dq_out, l.dk_out, ptr(dq), ptr(dk), B * T, (int)HK, (int)(H / HK), (int)K, dq.stride(1), stream);
        });
    });
}

// conv_bwd(stream, x, weight, bias, mask, dy, activation, tokens_per_block) -> (dx, dweight, dbias or None)
PyObject* conv_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 8, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &x = operand(args[1]), &weight = operand(args[2]), &dy = operand(args[5]);
        const at::Tensor *bias = operand.optional(args[3]), *mask = operand.optional(args[4]);
        gdn_conv_bwd_args s{};
        s.dtype = code_of(x), s.w_dtype = code_of(weight);
        need(x.dim() == 3 && x.stride(2) == 1 && dy.scalar_type() == x.scalar_type() && dy.sizes() == x.sizes());
        need_rows(dy, 2, 8);
        const int64_t B = x.size(0), S = x.size(1), C = x.size(2), ks = taps_of(weight, C), tokens = integer(args[7]);
        need(B > 0 && S > 0 && tokens > 0);
        if (bias != nullptr) need(bias->scalar_type() == weight.scalar_type() && bias->dim() == 1 && bias->size(0) == C && bias->is_contiguous());
        const int64_t blocks = B * ((S + tokens - 1) / tokens);
        at::Tensor kept_mask, dx, dw_part, db_part, dweight, dbias;
        const bool masked = mask != nullptr && mask->dim() == 2 && mask->size(0) > 1 && mask->size(1) > 1;
        need(mask == nullptr || mask->dim() == 2);
        if (masked) need(mask->size(0) == B && mask->size(1) == S);
        without_interpreter_lock([&] {
            if (masked) kept_mask = mask->to(x.scalar_type()).contiguous(), s.mask = ptr(kept_mask);
            dx = fresh(x, {B, S, C}), dw_part = fresh_f32(x, {blocks, C, ks}), db_part = fresh_f32(x, {blocks, C});
            dweight = at::empty(weight.sizes(), weight.options());
            if (bias != nullptr) dbias = at::empty({C}, bias->options());
        });
        s.x = ptr(x), s.dy = ptr(dy), s.weight = ptr(weight), s.bias = ptr(bias), s.dx = ptr(dx);
        s.dweight_partial = static_cast<float*>(ptr(dw_part)), s.dbias_partial = static_cast<float*>(ptr(db_part));
        s.x_stride_b = x.stride(0), s.x_stride_s = x.stride(1), s.dy_stride_b = dy.stride(0), s.dy_stride_s = dy.stride(1);
        s.B = size32(B), s.S = size32(S), s.C = size32(C), s.kernel_size = (int32_t)ks, s.tokens_per_block = size32(tokens);
        s.activation = (int32_t)integer(args[6]);
        ColumnSums sums;
        sums.add(dw_part, dweight);
        if (dbias.defined()) sums.add(db_part, dbias);
        return launch("gdn_causal_conv1d_bwd, gdn_column_sums", pack_results({dx, dweight, dbias}), [&] {
            const int status = conv_bwd_fn(&s, stream);
            return status == GDN_OK ? column_sums_fn(&sums.s, stream) : status;
        });
    });
}

// gates_bwd(stream, a, b, A_log, dt_bias, dg, dbeta, beta_scale) -> (da, db, dA_log, ddt_bias)
PyObject* gates_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 8, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &a = operand(args[1]), &b = operand(args[2]), &A_log = operand(args[3]), &dt_bias = operand(args[4]), &dg = operand(args[5]), &dbeta = operand(args[6]);
        gdn_gate_bwd_args s{};
        s.dtype = code_of(a);
        need(a.dim() >= 2 && b.scalar_type() == a.scalar_type() && b.sizes() == a.sizes() && a.numel() > 0);
        const int64_t H = a.size(-1);
        const at::Tensor* decay[] = {&A_log, &dt_bias};
        for (const at::Tensor* t : decay) need(t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == H && t->is_contiguous());
        need(dg.scalar_type() == at::kFloat && dg.sizes() == a.sizes() && dg.is_contiguous());
        need(dbeta.scalar_type() == a.scalar_type() && dbeta.sizes() == a.sizes() && dbeta.is_contiguous());
        s.a_stride = row_stride(a, H), s.b_stride = row_stride(b, H);
        s.tokens = a.numel() / H, s.H = size32(H);
        s.partial_blocks = (int32_t)std::min<int64_t>(1024, (a.numel() + 255) / 256);
        at::Tensor da, db, dA_part, ddt_part, dA_log, ddt_bias;
        without_interpreter_lock([&] {
            da = fresh(a, a.sizes()), db = fresh(a, a.sizes());
            dA_part = fresh_f32(a, {s.partial_blocks, H}), ddt_part = fresh_f32(a, {s.partial_blocks, H});
            dA_log = fresh_f32(a, {H}), ddt_bias = fresh_f32(a, {H});
        });
        s.a = ptr(a), s.b = ptr(b), s.A_log = static_cast<const float*>(ptr(A_log)), s.dt_bias = static_cast<const float*>(ptr(dt_bias));
        s.dg = static_cast<const float*>(ptr(dg)), s.dbeta = ptr(dbeta), s.da = ptr(da), s.db = ptr(db);
        s.dA_log_partial = static_cast<float*>(ptr(dA_part)), s.ddt_bias_partial = static_cast<float*>(ptr(ddt_part));
        s.beta_scale = (float)number(args[7]);
        ColumnSums sums;
        sums.add(dA_part, dA_log), sums.add(ddt_part, ddt_bias);
        return launch("gdn_gates_bwd, gdn_column_sums", pack_results({da, db, dA_log, ddt_bias}), [&] {
            const int status = gates_bwd_fn(&s, stream);
            return status == GDN_OK ? column_sums_fn(&sums.s, stream) : status;
        });
    });
}

// norm_bwd(stream, o, gate, weight, eps, dy) -> (d_o, d_gate or None, d_weight or None)
PyObject* norm_bwd(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 6, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &o = operand(args[1]), &dy = operand(args[5]);
        const at::Tensor *gate = operand.optional(args[2]), *weight = operand.optional(args[3]);
        gdn_norm_bwd_args s{};
        s.dtype = code_of(o);
        const NormOperands x(o, gate);
        need(dy.scalar_type() == o.scalar_type() && dy.sizes() == o.sizes() && dy.is_contiguous());
        need_rows(dy, 8, 16);
        s.tokens = o.numel() / (x.H * x.V), s.gate_stride_t = x.gate_stride;
        s.w_dtype = GDN_F32;
        if (weight != nullptr) {
            s.w_dtype = code_of(*weight);
            need(weight->dim() == 1 && weight->size(0) == x.V && weight->is_contiguous());
        }
        s.w_dtype |= GDN_NORM_GATE_DWORDS;
        s.partial_blocks = (int32_t)std::min<int64_t>(2048, std::max<int64_t>(1, (s.tokens * x.H * std::max<int64_t>(x.V / 8, 8) + 255) / 256));
        at::Tensor d_o, d_gate, part, d_weight;
        without_interpreter_lock([&] {
            d_o = fresh(o, o.sizes()), part = fresh_f32(o, {s.partial_blocks, x.V});
            if (gate != nullptr) d_gate = fresh(o, gate->sizes());
            if (weight != nullptr) d_weight = at::empty({x.V}, weight->options());
        });
        s.o = ptr(o), s.gate = ptr(gate), s.weight = ptr(weight), s.dy = ptr(dy), s.d_o = ptr(d_o), s.d_gate = d_gate.defined() ? ptr(d_gate) : nullptr;
        s.dweight_partial = static_cast<float*>(ptr(part));
        s.o_stride_t = x.H * x.V, s.H = size32(x.H), s.V = (int32_t)x.V, s.eps = (float)number(args[4]);
        ColumnSums sums;
        if (d_weight.defined()) sums.add(part, d_weight);
        return launch("gdn_gated_rmsnorm_bwd, gdn_column_sums", pack_results({d_o, d_gate, d_weight}), [&] {
            const int status = norm_bwd_fn(&s, stream);
            return status == GDN_OK && sums.s.arrays > 0 ? column_sums_fn(&sums.s, stream) : status;
        });
    });
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)())bind, METH_FASTCALL, "takes the addresses of the library's entry points"},
    {"layer_step", (PyCFunction)(void (*)())layer_step, METH_FASTCALL, "gdn_layer_step"},
    {"conv", (PyCFunction)(void (*)())conv, METH_FASTCALL, "gdn_causal_conv1d_fwd"},
    {"gates", (PyCFunction)(void (*)())gates, METH_FASTCALL, "gdn_gates_fwd"},
    {"layer_front", (PyCFunction)(void (*)())layer_front, METH_FASTCALL, "gdn_layer_front"},
    {"norm", (PyCFunction)(void (*)())norm, METH_FASTCALL, "gdn_gated_rmsnorm_fwd"},
    {"delta_rule", (PyCFunction)(void (*)())delta_rule, METH_FASTCALL, "gdn_chunk_fwd or gdn_recurrent_fwd"},
    {"delta_rule_bwd", (PyCFunction)(void (*)())delta_rule_bwd, METH_FASTCALL, "gdn_chunk_bwd_sweeps, gdn_chunk_bwd_local"},
    {"conv_bwd", (PyCFunction)(void (*)())conv_bwd, METH_FASTCALL, "gdn_causal_conv1d_bwd, gdn_column_sums"},
    {"gates_bwd", (PyCFunction)(void (*)())gates_bwd, METH_FASTCALL, "gdn_gates_bwd, gdn_column_sums"},
    {"norm_bwd", (PyCFunction)(void (*)())norm_bwd, METH_FASTCALL, "gdn_gated_rmsnorm_bwd, gdn_column_sums"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "gdn_host", "host path of the entry points and their backward passes", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_gdn_host() { return PyModule_Create(&module); }
