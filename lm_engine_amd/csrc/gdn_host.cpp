// The host path of the inference entry points: from torch tensors to one call of the C ABI (include/gdn_hip.h).
//
// On a decode step or a short prompt the GPU needs a few microseconds per kernel, and reading shapes, strides and
// pointers out of tensors, allocating the results and filling the argument struct takes 10 to 20 in Python per call.  Here
// it takes 1 to 4.  Every function is a fast path only: it takes well-formed operands that need no conversion and no
// gradient, and returns None for everything else, so that the Python code behind it converts, differentiates or reports.
// The library itself stays independent of torch: its entry points come in as addresses (bind), from the one loaded copy.

#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/GradMode.h>
#include <c10/core/impl/VirtualGuardImpl.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

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
PyObject* check_status = nullptr;  // _lib.check_status: raises what a status stands for

// bind(check_status, addresses...)
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    void** slots[] = {(void**)&layer_step_fn, (void**)&layer_step_tiles_fn, (void**)&conv_fn, (void**)&gates_fn, (void**)&norm_fn,
                      (void**)&recurrent_fn, (void**)&chunk_fn, (void**)&workspace_bytes_fn, (void**)&one_launch_fn};
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

// conv(stream, x, weight, bias, input_state, mask, output_state, activation) -> (y, final_state or None)
PyObject* conv(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 8, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &x = operand(args[1]), &weight = operand(args[2]);
        const at::Tensor *bias = operand.optional(args[3]), *state = operand.optional(args[4]), *mask = operand.optional(args[5]);
        gdn_conv_args s{};
        s.dtype = code_of(x), s.w_dtype = code_of(weight);
        need(x.dim() == 3 && x.stride(2) == 1 && (s.dtype == GDN_BF16 || s.w_dtype == GDN_F32));
        const int64_t B = x.size(0), S = x.size(1), C = x.size(2), ks = taps_of(weight, C);
        need(B > 0 && S > 0);
        if (bias != nullptr) need(bias->scalar_type() == weight.scalar_type() && bias->dim() == 1 && bias->size(0) == C && bias->is_contiguous());
        if (state != nullptr) need(state->scalar_type() == x.scalar_type() && state->sizes() == at::IntArrayRef({B, C, ks - 1}) && state->is_contiguous());
        at::Tensor kept_mask;
        bool masked = false;
        if (mask != nullptr) need(mask->dim() == 2);
        if (mask != nullptr && mask->size(0) > 1 && mask->size(1) > 1) {
            need(mask->size(0) == B && mask->size(1) == S);
            masked = true;
        }
        const bool output_state = truth(args[6]);
        at::Tensor y, final_state;
        without_interpreter_lock([&] {
            if (masked) kept_mask = mask->to(x.scalar_type()).contiguous(), s.mask = ptr(kept_mask);
            y = fresh(x, {B, S, C});
            if (output_state) final_state = fresh(x, {B, C, ks - 1}), s.final_state = ptr(final_state);
        });
        s.x = ptr(x), s.weight = ptr(weight), s.bias = ptr(bias), s.input_state = ptr(state), s.y = ptr(y);
        s.x_stride_b = x.stride(0), s.x_stride_s = x.stride(1), s.y_stride_b = S * C, s.y_stride_s = C;
        s.B = size32(B), s.S = size32(S), s.C = size32(C), s.kernel_size = (int32_t)ks;
        s.activation = (int32_t)integer(args[7]);
        return launch("gdn_causal_conv1d_fwd", pack_results({y, final_state}), [&] { return conv_fn(&s, stream); });
    });
}

// gates(stream, a, b, A_log, dt_bias, beta_scale) -> (g, beta)
PyObject* gates(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 6, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor &a = operand(args[1]), &b = operand(args[2]), &A_log = operand(args[3]), &dt_bias = operand(args[4]);
        gdn_gate_args s{};
        s.dtype = code_of(a);
        need(a.dim() >= 2 && b.scalar_type() == a.scalar_type() && b.sizes() == a.sizes() && a.numel() > 0);
        const int64_t H = a.size(-1);
        const at::Tensor* decay[] = {&A_log, &dt_bias};
        for (const at::Tensor* t : decay) need(t->scalar_type() == at::kFloat && t->dim() == 1 && t->size(0) == H && t->is_contiguous());
        s.a_stride = row_stride(a, H), s.b_stride = row_stride(b, H);
        s.tokens = a.numel() / H, s.H = size32(H);
        at::Tensor g, beta;
        without_interpreter_lock([&] { g = fresh_f32(a, a.sizes()), beta = fresh(a, a.sizes()); });
        s.a = ptr(a), s.b = ptr(b), s.A_log = static_cast<const float*>(ptr(A_log)), s.dt_bias = static_cast<const float*>(ptr(dt_bias));
        s.g = static_cast<float*>(ptr(g)), s.beta = ptr(beta), s.beta_scale = (float)number(args[5]);
        return launch("gdn_gates_fwd", pack_results({g, beta}), [&] { return gates_fn(&s, stream); });
    });
}

// norm(stream, o, gate, weight, eps) -> y
PyObject* norm(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return fast_path(n, 5, [&]() -> PyObject* {
        Operands operand;
        void* const stream = stream_of(args[0]);
        const at::Tensor& o = operand(args[1]);
        const at::Tensor *gate = operand.optional(args[2]), *weight = operand.optional(args[3]);
        gdn_norm_args s{};
        s.dtype = code_of(o);
        need(o.dim() >= 2 && o.is_contiguous() && o.numel() > 0);
        const int64_t H = o.size(-2), V = o.size(-1);
        need(V % 8 == 0 && V <= 512);
        s.tokens = o.numel() / (H * V);
        if (gate != nullptr) {
            need(gate->scalar_type() == o.scalar_type() && gate->numel() == o.numel() && gate->dim() >= 2);
            if (gate->size(-1) == H * V && gate->dim() == o.dim() - 1) {
                s.gate_stride_t = row_stride(*gate, H * V);
            } else {
                need(gate->sizes() == o.sizes() && gate->is_contiguous());
                s.gate_stride_t = H * V;
            }
        }
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

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)())bind, METH_FASTCALL, "takes the addresses of the library's entry points"},
    {"layer_step", (PyCFunction)(void (*)())layer_step, METH_FASTCALL, "gdn_layer_step"},
    {"conv", (PyCFunction)(void (*)())conv, METH_FASTCALL, "gdn_causal_conv1d_fwd"},
    {"gates", (PyCFunction)(void (*)())gates, METH_FASTCALL, "gdn_gates_fwd"},
    {"norm", (PyCFunction)(void (*)())norm, METH_FASTCALL, "gdn_gated_rmsnorm_fwd"},
    {"delta_rule", (PyCFunction)(void (*)())delta_rule, METH_FASTCALL, "gdn_chunk_fwd or gdn_recurrent_fwd"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "gdn_host", "host path of the inference entry points", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_gdn_host() { return PyModule_Create(&module); }
