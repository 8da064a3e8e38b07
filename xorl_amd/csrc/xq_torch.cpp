// The host path of the modules as native code: a CPython extension over libxq_hip.so and torch's C++ API.
//
// A decode forward is one or two kernels of 5-20 us; read from Python (parameter look-ups, the weight descriptor and its
// checks, torch.empty, ctypes) the same call cost 22 us of host time for one linear, 50 for a SwiGLU MLP or three joint
// projections and 70 for a routed expert layer, so the GPU waited for the host.  Here the module's own dictionaries are read
// directly, outputs and workspaces come from torch's caching allocator without the dispatcher, and the backward is a C++
// autograd node that runs without the interpreter.
//
// Every entry point returns None where anything is out of the ordinary (tensor subclasses, sharded or CPU state, tangents of
// forward-mode differentiation, function transforms, a trace being recorded, quantization noise, an active rank below the
// stored one, unexpected dtypes or layouts, a module that defines for itself what is read or done here): the caller then takes its Python path, which also raises the argument errors.
// Nothing is remembered from one call to the next, and a backward takes the addresses of the packed weights anew from
// their tensors: storage may have been freed and filled again between the two.
#include <Python.h>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/TracerMode.h>
#include <ATen/core/Tensor.h>
#include <ATen/EmptyTensor.h>
#include <ATen/hip/impl/HIPCachingAllocatorMasqueradingAsCUDA.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>

#include <cmath>
#include <optional>
#include <string>
#include <vector>

#include "../../include/xq.h"

namespace {

using at::Tensor;
using torch::autograd::Node;
using torch::autograd::SavedVariable;
using torch::autograd::variable_list;

// ---- names and classes handed over by the Python side (init)
PyObject* g_error = nullptr;            // xorl_amd._C.XqError
PyObject* g_functional = nullptr;       // the dict of xorl_amd.functional: SKINNY_CHECK_EVERY, skinny_status

// a module class and the methods whose work is done here in their place, as the class defines them
struct Program {
    PyTypeObject* type = nullptr;
    std::vector<PyObject*> name, method;
};
constexpr int kFormats = XQ_FMT_NF4 + 1;
Program g_linear[kFormats], g_experts[kFormats];      // by format; no type: no such class

#define XQ_NAMES(F)                                                                                                       \
    F(_parameters) F(_buffers) F(lora_A) F(lora_B) F(bias) F(packed_weight_f32) F(weight_scales) F(weight_block_scales)   \
    F(weight_global_scale) F(_scale_dtypes) F(active_r) F(active_lora_alpha) F(enable_aqn) F(training) F(quant_format)    \
    F(quant_group_size) F(in_features) F(out_features) F(num_local_experts) F(num_experts) F(hidden_size)                 \
    F(intermediate_size) F(use_rslora) F(swiglu_limit) F(moe_implementation) F(gate) F(up) F(down) F(gate_packed)         \
    F(up_packed) F(down_packed) F(gate_block_scales) F(up_block_scales) F(down_block_scales) F(gate_scales) F(up_scales)  \
    F(down_scales) F(gate_global_scale) F(up_global_scale) F(down_global_scale) F(gate_proj_lora_A) F(gate_proj_lora_B)   \
    F(up_proj_lora_A) F(up_proj_lora_B) F(down_proj_lora_A) F(down_proj_lora_B) F(SKINNY_CHECK_EVERY) F(skinny_status)     \
    F(__getattr__) F(__getattribute__)
#define XQ_DECLARE(n) PyObject* s_##n;
struct Names { XQ_NAMES(XQ_DECLARE) } N;
#undef XQ_DECLARE

PyObject* get(PyObject* dict, PyObject* name) { return dict ? PyDict_GetItem(dict, name) : nullptr; }   // borrowed, no error set

PyObject* dict_of(PyObject* module) {
    PyObject** p = _PyObject_GetDictPtr(module);
    return p ? *p : nullptr;
}

// whether the methods of `p` are the ones that run on `module` (no subclass, instance attribute or patch replaces one) and, in
// a subclass, whether what is read from the module's dictionaries is what attribute access gives (no property, no __getattr__
// of its own).  The library's own classes: 4-6 look-ups in the type's method cache and as many in the instance's dictionary.
bool as_defined(PyObject* module, PyObject* dict, const Program& p) {
    if (!p.type || !PyObject_TypeCheck(module, p.type)) return false;
    PyTypeObject* type = Py_TYPE(module);
    for (size_t i = 0; i < p.name.size(); ++i)
        if (_PyType_Lookup(type, p.name[i]) != p.method[i] || get(dict, p.name[i])) return false;
    if (type == p.type) return true;
#define XQ_SAME(n) if (_PyType_Lookup(type, N.s_##n) != _PyType_Lookup(p.type, N.s_##n)) return false;
    XQ_NAMES(XQ_SAME)
#undef XQ_SAME
    return true;
}

bool get_int(PyObject* dict, PyObject* name, int64_t* out) {
    PyObject* o = get(dict, name);
    if (!o || !PyLong_Check(o)) return false;
    *out = PyLong_AsLongLong(o);
    if (*out == -1 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}

bool get_number(PyObject* dict, PyObject* name, double* out) {
    PyObject* o = get(dict, name);
    if (!o || !(PyFloat_Check(o) || PyLong_Check(o))) return false;
    *out = PyFloat_AsDouble(o);
    if (*out == -1.0 && PyErr_Occurred()) { PyErr_Clear(); return false; }
    return true;
}

// a plain torch tensor (or Parameter) on the GPU; subclasses, fakes, functorch wrappers and tensors that carry a tangent are
// left to the Python path (whose autograd functions refuse what they do not define)
const Tensor* plain(PyObject* o) {
    if (!o || !THPVariable_CheckExact(o)) return nullptr;
    const Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || at::isTensorSubclassLike(t) || t._fw_grad(0).defined()) return nullptr;
    return &t;
}

// a recorded trace or a function transform sees the operators of the Python path only
bool under_transform() {
    return at::tracer::impl::is_dispatch_enabled() ||
           c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode);
}

// library calls launch kernels and may wait for room in the queue: other Python threads go on meanwhile
struct ReleaseGil {
    PyThreadState* state = PyEval_SaveThread();
    ~ReleaseGil() { PyEval_RestoreThread(state); }
};

int scale_code(PyObject* dtype, int* bytes) {
    if (!dtype || !THPDtype_Check(dtype)) return -1;
    switch (((THPDtype*)dtype)->scalar_type) {
        case at::kFloat: *bytes = 4; return XQ_SCALE_F32;
        case at::kBFloat16: *bytes = 2; return XQ_SCALE_BF16;
        case at::kFloat8_e4m3fn: *bytes = 1; return XQ_SCALE_E4M3;
        default: return -1;
    }
}

int format_code(PyObject* name) {
    if (!name || !PyUnicode_Check(name)) return -1;
    if (PyUnicode_CompareWithASCIIString(name, "block_fp8") == 0) return XQ_FMT_FP8;
    if (PyUnicode_CompareWithASCIIString(name, "nvfp4") == 0) return XQ_FMT_NVFP4;
    if (PyUnicode_CompareWithASCIIString(name, "int4") == 0) return XQ_FMT_INT4;
    if (PyUnicode_CompareWithASCIIString(name, "nf4") == 0) return XQ_FMT_NF4;
    return -1;
}

int64_t nbytes(const Tensor& t) { return t.numel() * (int64_t)t.element_size(); }

// packed bytes, scales and (nvfp4) the global scale of a weight, checked for size as _C.make_weight does
struct Weight {
    xq_weight w{};
    Tensor packed, scales, global_scale;
    int64_t packed_bytes = 0, scale_bytes = 0;

    bool fill(int fmt, int layout, int64_t rows, int64_t cols, int64_t group, int64_t experts, PyObject* packed_o, PyObject* scales_o,
              PyObject* scale_dtype, PyObject* global_o, PyObject* global_dtype) {
        const Tensor *p = plain(packed_o), *s = plain(scales_o);
        int sb = 0;
        const int sd = scale_code(scale_dtype, &sb);
        if (!p || !s || sd < 0 || !p->is_contiguous() || !s->is_contiguous() || rows <= 0 || cols <= 0 || group <= 0) return false;
        if (nbytes(*p) != experts * (fmt == XQ_FMT_FP8 ? rows * cols : rows * cols / 2)) return false;
        if (fmt == XQ_FMT_FP8) {
            if (sd != XQ_SCALE_F32 || nbytes(*s) != experts * ((rows + 127) / 128) * ((cols + 127) / 128) * 4) return false;
        } else if (rows * cols % group || nbytes(*s) != experts * (rows * cols / group) * sb) {
            return false;
        }
        if (fmt == XQ_FMT_NVFP4) {
            const Tensor* g = plain(global_o);
            int gb = 0;
            if (!g || scale_code(global_dtype, &gb) != XQ_SCALE_F32 || !g->is_contiguous() || nbytes(*g) < 4 * experts) return false;
            if ((uintptr_t)g->data_ptr() % 4) return false;
            global_scale = *g;
            w.global_scale = (const float*)g->data_ptr();
        }
        packed = *p;
        scales = *s;
        w.format = fmt; w.layout = layout; w.scale_dtype = sd; w.group = (int32_t)group;
        w.rows = rows; w.cols = cols; w.num_experts = (int32_t)experts;
        w.packed = p->data_ptr(); w.scales = s->data_ptr();
        packed_bytes = nbytes(*p); scale_bytes = nbytes(*s);
        return true;
    }

    // the descriptor for a later call: addresses as they are now, and storage that still holds the bytes
    const xq_weight* now() {
        auto held = [](const Tensor& t, int64_t bytes) {
            return nbytes(t) == bytes && t.is_contiguous() &&
                   (int64_t)t.storage().nbytes() >= t.storage_offset() * (int64_t)t.element_size() + bytes;
        };
        TORCH_CHECK(held(packed, packed_bytes) && held(scales, scale_bytes) &&
                        (!global_scale.defined() || held(global_scale, nbytes(global_scale))),
                    "the packed weight of a QLoRA module was freed or resized between forward and backward");
        w.packed = packed.data_ptr();
        w.scales = scales.data_ptr();
        if (global_scale.defined()) w.global_scale = (const float*)global_scale.data_ptr();
        return &w;
    }
};

// a QLoRALinear as the kernels see it
struct Linear {
    Weight q;
    Tensor A, B, bias;      // bias undefined: none
    int r = 0;
    double scaling = 0;
    bool A_grad = false, B_grad = false, bias_grad = false;

    int lora_dtype() const { return A.scalar_type() == at::kFloat ? XQ_DT_F32 : XQ_DT_BF16; }
    bool wants_grad() const { return A_grad || B_grad || bias_grad; }
    const void* bias_ptr() const { return bias.defined() ? bias.data_ptr() : nullptr; }

    bool read(PyObject* module) {
        PyObject* d = dict_of(module);
        PyObject *params = get(d, N.s__parameters), *bufs = get(d, N.s__buffers), *sdt = get(d, N.s__scale_dtypes);
        if (!params || !bufs || !sdt || !PyDict_Check(sdt)) return false;
        PyObject* aqn = get(d, N.s_enable_aqn);
        if (aqn != Py_False && !(aqn == Py_True && get(d, N.s_training) == Py_False)) return false;
        const int fmt = format_code(get(d, N.s_quant_format));
        int64_t rank, group, n, k;
        double alpha;
        if (fmt < 0 || !as_defined(module, d, g_linear[fmt]) || !get_int(d, N.s_active_r, &rank) || !get_number(d, N.s_active_lora_alpha, &alpha) ||
            !get_int(d, N.s_quant_group_size, &group) || !get_int(d, N.s_out_features, &n) || !get_int(d, N.s_in_features, &k))
            return false;
        PyObject* packed_o = get(params, N.s_packed_weight_f32);
        const Tensor* packed = plain(packed_o);
        if (!packed || packed->scalar_type() != at::kFloat) return false;      // (bytes held as fp32: anything else has been cast)
        PyObject* sname = fmt == XQ_FMT_FP8 || fmt == XQ_FMT_NVFP4 ? N.s_weight_block_scales : N.s_weight_scales;
        if (!q.fill(fmt, XQ_LAYOUT_FLAT, n, k, group, 1, packed_o, get(bufs, sname), get(sdt, sname),
                    get(bufs, N.s_weight_global_scale), get(sdt, N.s_weight_global_scale)))
            return false;
        const Tensor *a = plain(get(params, N.s_lora_A)), *b = plain(get(params, N.s_lora_B));
        if (!a || !b || rank < 1 || rank > 64 || a->dim() != 2 || b->dim() != 2 || a->size(0) != rank || b->size(1) != rank || a->size(1) != k ||
            b->size(0) != n || !a->is_contiguous() || !b->is_contiguous() || a->scalar_type() != b->scalar_type() ||
            (a->scalar_type() != at::kFloat && a->scalar_type() != at::kBFloat16))
            return false;
        PyObject* bias_o = get(params, N.s_bias);
        if (bias_o && bias_o != Py_None) {
            const Tensor* bt = plain(bias_o);
            if (!bt || bt->numel() != n) return false;
            bias_grad = bt->requires_grad();
            bias = bt->scalar_type() == at::kBFloat16 && bt->is_contiguous() ? *bt : bt->detach().to(at::kBFloat16).contiguous();
        }
        A = *a;
        B = *b;
        A_grad = a->requires_grad();
        B_grad = b->requires_grad();
        r = (int)rank;
        scaling = alpha / (double)rank;
        return true;
    }
};

// activations as rows of `width`: the pointer and pitch the library takes.  Rows that lie a fixed pitch apart over all leading
// dimensions are read where they are (a slice of a wider last dimension, any number of dimensions); other layouts, and pitches
// or addresses that are no multiple of 16 bytes, take a packed copy.
struct Rows {
    Tensor keep;
    const void* ptr = nullptr;
    int64_t ld = 0, M = 0;

    static bool pitched(const Tensor& x, int64_t* pitch) {
        if (x.stride(-1) != 1 || (uintptr_t)x.data_ptr() % 16 != 0) return false;
        int64_t rows = 1;                                          // of the dimensions looked at, the innermost first
        for (int64_t d = x.dim() - 2; d >= 0; --d) {
            if (x.size(d) == 1) continue;
            if (rows == 1) *pitch = x.stride(d);
            else if (x.stride(d) != *pitch * rows) return false;
            rows *= x.size(d);
        }
        return rows == 1 || *pitch % 8 == 0;
    }

    Rows(const Tensor& x, int64_t width) {
        M = width ? x.numel() / width : 0;
        ld = width;
        keep = x;
        if (!x.is_contiguous() && !pitched(x, &ld)) {
            keep = x.contiguous();
            ld = width;
        }
        ptr = keep.data_ptr();
    }
};

// torch's caching allocator, in the form whose tensors are "cuda" tensors
c10::Allocator* allocator() {
    static c10::Allocator* a = c10::hip::HIPCachingAllocatorMasqueradingAsCUDA::get();
    return a;
}

Tensor empty(at::IntArrayRef size, at::ScalarType dt) {
    constexpr c10::DispatchKeySet ks(c10::DispatchKey::CUDA);
    return at::detail::empty_generic(size, allocator(), ks, dt, std::nullopt);
}
Tensor empty_bf(at::IntArrayRef size) { return empty(size, at::kBFloat16); }
Tensor empty_f32(at::IntArrayRef size) { return empty(size, at::kFloat); }

// scratch of one call: back with the allocator (in stream order) when the call returns
struct Scratch {
    c10::DataPtr p;
    int64_t bytes;
    explicit Scratch(int64_t n) : p(allocator()->allocate((size_t)(n > 0 ? n : 0))), bytes(n) {}
    void* get() const { return p.get(); }
};

void* stream_of(const Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

struct ArgError : std::runtime_error { using std::runtime_error::runtime_error; };

void check(int rc) {
    if (rc == XQ_OK) return;
    if (rc == XQ_ERR_LAUNCH) throw std::runtime_error(xq_last_error());
    throw ArgError(xq_last_error());
}

std::vector<int64_t> with_last(const Tensor& x, int64_t last) {
    std::vector<int64_t> s(x.sizes().begin(), x.sizes().end());
    s.back() = last;
    return s;
}

int r_pad_of(int r) { return (r + 15) / 16 * 16; }

int shared_format(const xq_weight& a, const xq_weight& b, const xq_weight& c) { return a.format == b.format && a.format == c.format ? a.format : -1; }

// the report of the one-launch decode forwards is read after every functional.SKINNY_CHECK_EVERY forwards of up to 16 rows
bool note_decode_forward(const Tensor& x, int64_t M) {
    static int64_t calls = 0;       // (under the GIL)
    if (M > 16) return true;
    int64_t every;
    if (!get_int(g_functional, N.s_SKINNY_CHECK_EVERY, &every)) every = 1024;
    if (++calls < every) return true;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing((hipStream_t)stream_of(x), &cap) != hipSuccess || cap != hipStreamCaptureStatusNone) return true;
    calls = 0;
    PyObject* fn = get(g_functional, N.s_skinny_status);
    PyObject* dev = THPDevice_New(x.device());
    PyObject* r = fn && dev ? PyObject_CallFunctionObjArgs(fn, dev, nullptr) : nullptr;
    Py_XDECREF(dev);
    Py_XDECREF(r);
    return r != nullptr;
}

// ---- backward nodes: edges in the order of the inputs named in each
Tensor cast_to(Tensor g, at::ScalarType dt) { return g.scalar_type() == dt ? g : g.to(dt); }

struct QLoRALinearBackward : public Node {
    SavedVariable x_, su_, A_, B_;
    Weight q;
    int r = 0;
    double scaling = 0;
    at::ScalarType bias_dt = at::kBFloat16;

    std::string name() const override { return "QLoRALinearBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x_.reset_data();
        su_.reset_data();
        A_.reset_data();
        B_.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(4);
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        const Tensor x = x_.unpack(), A = A_.unpack(), B = B_.unpack(), su = su_.unpack(shared_from_this());
        const int64_t Nf = q.w.rows, K = q.w.cols;
        Tensor dy = cast_to(grads[0], at::kBFloat16);
        c10::DeviceGuard guard(x.device());
        const Rows dr(dy, Nf), xr(x, K);
        const int64_t M = dr.M;
        const bool need_dx = task_should_compute_output(0), need_dA = task_should_compute_output(1), need_dB = task_should_compute_output(2);
        if (need_dx) out[0] = empty_bf(x.sizes());
        if (need_dA) out[1] = empty_f32({r, K});
        if (need_dB) out[2] = empty_f32({Nf, r});
        Scratch ws(xq_linear_workspace_bytes_fmt(q.w.format, M, Nf, K, r));
        check(xq_linear_bwd(q.now(), xr.ptr, xr.ld, dr.ptr, dr.ld, M, A.data_ptr(), B.data_ptr(),
                            A.scalar_type() == at::kFloat ? XQ_DT_F32 : XQ_DT_BF16, r, (float)scaling, M ? su.data_ptr() : nullptr,
                            need_dx ? out[0].data_ptr() : nullptr, K, need_dA ? (float*)out[1].data_ptr() : nullptr,
                            need_dB ? (float*)out[2].data_ptr() : nullptr, ws.get(), ws.bytes, stream_of(x)));
        if (need_dA) out[1] = cast_to(out[1], A.scalar_type());
        if (need_dB) out[2] = cast_to(out[2], B.scalar_type());
        if (task_should_compute_output(3)) out[3] = cast_to(grads[0].reshape({-1, Nf}).sum(0), bias_dt);
        return out;
    }
};

void mlp_lora(xq_mlp_lora* L, const Tensor* A, const Tensor* B, int r, double scaling) {
    for (int p = 0; p < 3; ++p) {
        L->A[p] = A[p].data_ptr();
        L->B[p] = B[p].data_ptr();
        L->bias[p] = nullptr;
    }
    L->dtype = A[0].scalar_type() == at::kFloat ? XQ_DT_F32 : XQ_DT_BF16;
    L->r = r;
    L->scaling = (float)scaling;
    L->reserved = 0;
}

struct QLoRAMLPBackward : public Node {
    SavedVariable x_, kept_[4], A_[3], B_[3];     // kept: gate | up, h, su of gate and up, su of down
    Weight q[3];
    int r = 0, gate_up_fused = 0;
    double scaling = 0;

    std::string name() const override { return "QLoRAMLPBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x_.reset_data();
        for (auto& v : kept_) v.reset_data();
        for (auto& v : A_) v.reset_data();
        for (auto& v : B_) v.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(7);                      // x, gate A, gate B, up A, up B, down A, down B
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        const Tensor x = x_.unpack();
        Tensor kept[4], A[3], B[3];
        for (int i = 0; i < 4; ++i) kept[i] = kept_[i].unpack(shared_from_this());
        for (int p = 0; p < 3; ++p) { A[p] = A_[p].unpack(); B[p] = B_[p].unpack(); }
        const int64_t I = q[0].w.rows, H = q[0].w.cols;
        Tensor dy = cast_to(grads[0], at::kBFloat16);
        c10::DeviceGuard guard(x.device());
        const Rows dr(dy, H), xr(x, H);
        const bool need_dx = task_should_compute_output(0);
        if (need_dx) out[0] = empty_bf(x.sizes());
        xq_mlp_grads G;
        for (int p = 0; p < 3; ++p) {
            out[1 + 2 * p] = empty_f32(A[p].sizes());
            out[2 + 2 * p] = empty_f32(B[p].sizes());
            G.dA[p] = (float*)out[1 + 2 * p].data_ptr();
            G.dB[p] = (float*)out[2 + 2 * p].data_ptr();
        }
        xq_mlp_lora L;
        mlp_lora(&L, A, B, r, scaling);
        xq_mlp_saved S{kept[0].data_ptr(), kept[1].data_ptr(), kept[2].data_ptr(), kept[3].data_ptr(), gate_up_fused, 0};
        Scratch ws(xq_mlp_workspace_bytes_fmt(shared_format(q[0].w, q[1].w, q[2].w), dr.M, H, I, r, 1));
        check(xq_mlp_bwd(q[0].now(), q[1].now(), q[2].now(), &L, xr.ptr, xr.ld, dr.ptr, dr.ld, dr.M, &S, need_dx ? out[0].data_ptr() : nullptr, H, &G,
                         ws.get(), ws.bytes, stream_of(x)));
        for (int p = 0; p < 3; ++p) {
            out[1 + 2 * p] = cast_to(out[1 + 2 * p], A[p].scalar_type());
            out[2 + 2 * p] = cast_to(out[2 + 2 * p], B[p].scalar_type());
        }
        return out;
    }
};

// the eleven buffers of xq_grouped_saved that a forward fills, in its order
constexpr int kGroupedKept = 11;
void grouped_saved(xq_grouped_saved* S, const Tensor* kept, const Rows* x) {
    auto p = [&](int i) { return kept[i].numel() ? kept[i].data_ptr() : nullptr; };
    *S = xq_grouped_saved{};
    S->xs = p(0); S->gate_up = p(1); S->h = p(2); S->w_row = (float*)p(3); S->su_gate = p(4); S->su_up = p(5); S->su_down = p(6);
    S->scatter_index = (int32_t*)p(7); S->offsets = (int32_t*)p(8); S->tile_offsets = (int32_t*)p(9); S->counts = (int32_t*)p(10);
    if (x && x->M) { S->x_tokens = const_cast<void*>(x->ptr); S->ld_x_tokens = x->ld; }
}

void grouped_lora(xq_grouped_lora* L, const Tensor* A, const Tensor* B, int r, double scaling, double limit) {
    for (int p = 0; p < 3; ++p) {
        L->A[p] = A[p].data_ptr();
        L->B[p] = B[p].data_ptr();
        L->A_experts[p] = (int32_t)A[p].size(0);
        L->B_experts[p] = (int32_t)B[p].size(0);
    }
    L->dtype = A[0].scalar_type() == at::kFloat ? XQ_DT_F32 : XQ_DT_BF16;
    L->r = r;
    L->scaling = (float)scaling;
    L->swiglu_limit = (float)limit;
}

struct QLoRAMoeBackward : public Node {
    SavedVariable x_, kept_[kGroupedKept], A_[3], B_[3];
    Weight q[3];
    int r = 0;
    int64_t T = 0, topk = 0;
    double scaling = 0, limit = 0;
    at::ScalarType rw_dt = at::kFloat;
    std::vector<int64_t> rw_shape;

    std::string name() const override { return "QLoRAMoeBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        x_.reset_data();
        for (auto& v : kept_) v.reset_data();
        for (auto& v : A_) v.reset_data();
        for (auto& v : B_) v.reset_data();
    }
    variable_list apply(variable_list&& grads) override {
        std::lock_guard<std::mutex> lock(mutex_);
        variable_list out(8);                      // x, routing weights, then the factors as above
        if (!grads[0].defined()) grads[0] = input_metadata(0).zeros_like();
        const Tensor x = x_.unpack();
        Tensor kept[kGroupedKept], A[3], B[3];
        for (int i = 0; i < kGroupedKept; ++i) kept[i] = kept_[i].unpack(shared_from_this());
        for (int p = 0; p < 3; ++p) { A[p] = A_[p].unpack(); B[p] = B_[p].unpack(); }
        const int64_t H = q[0].w.rows, I = q[0].w.cols, E = q[0].w.num_experts;
        Tensor dy = cast_to(grads[0], at::kBFloat16);
        c10::DeviceGuard guard(x.device());
        const Rows dr(dy, H), xr(x, H);
        const bool need_dx = task_should_compute_output(0), need_drw = task_should_compute_output(1);
        if (need_dx) out[0] = empty_bf(x.sizes());
        const at::ScalarType kernel_dt = rw_dt == at::kBFloat16 ? at::kBFloat16 : at::kFloat;
        if (need_drw) out[1] = empty(rw_shape, kernel_dt);
        xq_grouped_grads G;
        for (int p = 0; p < 3; ++p) {
            out[2 + 2 * p] = empty_f32(A[p].sizes());
            out[3 + 2 * p] = empty_f32(B[p].sizes());
            G.dA[p] = (float*)out[2 + 2 * p].data_ptr();
            G.dB[p] = (float*)out[3 + 2 * p].data_ptr();
        }
        xq_grouped_lora L;
        grouped_lora(&L, A, B, r, scaling, limit);
        xq_grouped_saved S;
        grouped_saved(&S, kept, &xr);
        Scratch ws(xq_grouped_workspace_bytes(T, (int32_t)topk, (int32_t)E, H, I, r, 1));
        check(xq_grouped_bwd(q[0].now(), q[1].now(), q[2].now(), &L, dr.ptr, dr.ld, T, (int32_t)topk, &S, need_dx ? out[0].data_ptr() : nullptr, H,
                             need_drw ? out[1].data_ptr() : nullptr, kernel_dt == at::kBFloat16 ? XQ_DT_BF16 : XQ_DT_F32, &G, ws.get(),
                             ws.bytes, stream_of(x)));
        if (need_drw) out[1] = cast_to(out[1], rw_dt);
        for (int p = 0; p < 3; ++p) {
            out[2 + 2 * p] = cast_to(out[2 + 2 * p], A[p].scalar_type());
            out[3 + 2 * p] = cast_to(out[3 + 2 * p], B[p].scalar_type());
        }
        return out;
    }
};

// ---- entry points
bool usable_input(const Tensor* x, const Linear& m) {
    return x && x->scalar_type() == at::kBFloat16 && x->dim() >= 1 && x->size(-1) == m.q.w.cols && x->device() == m.q.packed.device() &&
           x->device() == m.A.device();
}

template <typename F>
PyObject* guarded(F&& f) {
    try {
        return f();
    } catch (const ArgError& e) {
        PyErr_SetString(g_error, e.what());
    } catch (const python_error& e) {
        const_cast<python_error&>(e).restore();
    } catch (const std::exception& e) {
        torch::translate_exception_to_python(std::current_exception());
    }
    return nullptr;
}

#define XQ_NONE Py_RETURN_NONE

// linear(module, x)
PyObject* linear(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (n != 2) { PyErr_SetString(PyExc_TypeError, "linear(module, x)"); return nullptr; }
        const Tensor* x = plain(args[1]);
        Linear m;
        if (under_transform() || !x || !m.read(args[0]) || !usable_input(x, m)) XQ_NONE;
        const int64_t Nf = m.q.w.rows, K = m.q.w.cols;
        const bool train = at::GradMode::is_enabled() && (x->requires_grad() || m.wants_grad());
        if (train && Nf % 64 != 0) XQ_NONE;
        c10::DeviceGuard guard(x->device());
        const Rows xr(*x, K);
        Tensor y = empty_bf(with_last(*x, Nf)), su;
        if (train) su = empty_bf({xr.M, r_pad_of(m.r)});
        Scratch ws(xq_linear_workspace_bytes_fmt(m.q.w.format, xr.M, Nf, K, m.r));
        {
            ReleaseGil nogil;
            check(xq_linear_fwd(&m.q.w, xr.ptr, xr.ld, xr.M, m.A.data_ptr(), m.B.data_ptr(), m.lora_dtype(), m.r, (float)m.scaling, m.bias_ptr(),
                  y.data_ptr(), Nf, train ? su.data_ptr() : nullptr, ws.get(), ws.bytes, stream_of(*x)));
        }
        if (!train) {
            if (!note_decode_forward(*x, xr.M)) return nullptr;
            return THPVariable_Wrap(std::move(y));
        }
        auto node = std::shared_ptr<QLoRALinearBackward>(new QLoRALinearBackward(), torch::autograd::deleteNode);
        const Tensor* bias = m.bias.defined() ? plain(get(get(dict_of(args[0]), N.s__parameters), N.s_bias)) : nullptr;
        node->set_next_edges(torch::autograd::collect_next_edges(*x, m.A, m.B, bias ? *bias : Tensor()));
        node->x_ = SavedVariable(*x, false);
        node->su_ = SavedVariable(su, false);
        node->A_ = SavedVariable(m.A, false);
        node->B_ = SavedVariable(m.B, false);
        if (bias) node->bias_dt = bias->scalar_type();
        node->q = m.q;
        node->r = m.r;
        node->scaling = m.scaling;
        torch::autograd::set_history(y, node);
        return THPVariable_Wrap(std::move(y));
    });
}

// linears(modules, x): up to XQ_LINEAR_MULTI_MAX forwards on one input, nothing differentiated
PyObject* linears(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (n != 2 || !PyList_Check(args[0])) { PyErr_SetString(PyExc_TypeError, "linears([modules], x)"); return nullptr; }
        const Py_ssize_t cnt = PyList_GET_SIZE(args[0]);
        const Tensor* x = plain(args[1]);
        if (under_transform() || !x || cnt < 2 || cnt > XQ_LINEAR_MULTI_MAX) XQ_NONE;
        const bool grad = at::GradMode::is_enabled();
        if (grad && x->requires_grad()) XQ_NONE;
        Linear m[XQ_LINEAR_MULTI_MAX];
        for (Py_ssize_t i = 0; i < cnt; ++i) {
            if (!m[i].read(PyList_GET_ITEM(args[0], i)) || !usable_input(x, m[i]) || (grad && m[i].wants_grad())) XQ_NONE;
            if (m[i].lora_dtype() != m[0].lora_dtype()) XQ_NONE;
        }
        c10::DeviceGuard guard(x->device());
        const Rows xr(*x, m[0].q.w.cols);
        xq_linear_job jobs[XQ_LINEAR_MULTI_MAX];
        Tensor y[XQ_LINEAR_MULTI_MAX];
        for (Py_ssize_t i = 0; i < cnt; ++i) {
            y[i] = empty_bf(with_last(*x, m[i].q.w.rows));
            jobs[i] = xq_linear_job{&m[i].q.w, m[i].A.data_ptr(), m[i].B.data_ptr(), m[i].r, (float)m[i].scaling, m[i].bias_ptr(),
                                    y[i].data_ptr(), m[i].q.w.rows};
        }
        Scratch ws(xq_linear_fwd_multi_workspace_bytes(jobs, (int)cnt, xr.M));
        {
            ReleaseGil nogil;
            check(xq_linear_fwd_multi(jobs, (int)cnt, xr.ptr, xr.ld, xr.M, m[0].lora_dtype(), ws.get(), ws.bytes, stream_of(*x)));
        }
        if (!note_decode_forward(*x, xr.M)) return nullptr;
        PyObject* out = PyList_New(cnt);
        if (!out) return nullptr;
        for (Py_ssize_t i = 0; i < cnt; ++i) PyList_SET_ITEM(out, i, THPVariable_Wrap(std::move(y[i])));
        return out;
    });
}

// mlp(gate, up, down, x)
PyObject* mlp(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (n != 4) { PyErr_SetString(PyExc_TypeError, "mlp(gate, up, down, x)"); return nullptr; }
        const Tensor* x = plain(args[3]);
        if (under_transform() || !x) XQ_NONE;
        Linear m[3];
        for (int p = 0; p < 3; ++p)
            if (!m[p].read(args[p])) XQ_NONE;
        const int64_t I = m[0].q.w.rows, H = m[0].q.w.cols;
        if (!usable_input(x, m[0]) || m[1].q.w.rows != I || m[1].q.w.cols != H || m[2].q.w.rows != H || m[2].q.w.cols != I || H % 64 || I % 64)
            XQ_NONE;
        for (int p = 0; p < 3; ++p)
            if (m[p].r != m[0].r || m[p].scaling != m[0].scaling || m[p].bias_grad || m[p].lora_dtype() != m[0].lora_dtype() ||
                m[p].q.packed.device() != x->device() || m[p].A.device() != x->device())
                XQ_NONE;
        const bool train = at::GradMode::is_enabled() && (x->requires_grad() || m[0].wants_grad() || m[1].wants_grad() || m[2].wants_grad());
        const int r = m[0].r, rp = r_pad_of(r), fmt = shared_format(m[0].q.w, m[1].q.w, m[2].q.w);
        c10::DeviceGuard guard(x->device());
        const Rows xr(*x, H);
        const int64_t M = xr.M;
        Tensor A[3] = {m[0].A, m[1].A, m[2].A}, B[3] = {m[0].B, m[1].B, m[2].B};
        xq_mlp_lora L;
        mlp_lora(&L, A, B, r, m[0].scaling);
        for (int p = 0; p < 3; ++p) L.bias[p] = m[p].bias_ptr();
        Tensor y = empty_bf(x->sizes());
        if (!train) {
            Scratch ws(xq_mlp_infer_workspace_bytes_fmt(fmt, M, H, I, r));
            {
                ReleaseGil nogil;
                check(xq_mlp_fwd_infer(&m[0].q.w, &m[1].q.w, &m[2].q.w, &L, xr.ptr, xr.ld, M, y.data_ptr(), H, ws.get(), ws.bytes, stream_of(*x)));
            }
            if (!note_decode_forward(*x, M)) return nullptr;
            return THPVariable_Wrap(std::move(y));
        }
        Tensor kept[4] = {empty_bf({M, 2 * I}), empty_bf({M, I}), empty_bf({M, 2 * rp}), empty_bf({M, rp})};
        // gate and up in one launch or two: settled once, for this forward and its backward
        const int gu = xq_get_mlp_gate_up_fused() && m[0].q.w.format == XQ_FMT_FP8 && m[1].q.w.format == XQ_FMT_FP8;
        xq_mlp_saved S{kept[0].data_ptr(), kept[1].data_ptr(), kept[2].data_ptr(), kept[3].data_ptr(), gu, 0};
        Scratch ws(xq_mlp_workspace_bytes_fmt(fmt, M, H, I, r, 0));
        {
            ReleaseGil nogil;
            check(xq_mlp_fwd(&m[0].q.w, &m[1].q.w, &m[2].q.w, &L, xr.ptr, xr.ld, M, y.data_ptr(), H, &S, ws.get(), ws.bytes, stream_of(*x)));
        }
        TORCH_CHECK(S.gate_up_fused == gu, "xq_mlp_fwd ran gate and up in form ", S.gate_up_fused, ", asked for ", gu);
        auto node = std::shared_ptr<QLoRAMLPBackward>(new QLoRAMLPBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(*x, A[0], B[0], A[1], B[1], A[2], B[2]));
        node->x_ = SavedVariable(*x, false);
        for (int i = 0; i < 4; ++i) node->kept_[i] = SavedVariable(kept[i], false);
        for (int p = 0; p < 3; ++p) {
            node->A_[p] = SavedVariable(A[p], false);
            node->B_[p] = SavedVariable(B[p], false);
            node->q[p] = m[p].q;
        }
        node->r = r;
        node->gate_up_fused = gu;
        node->scaling = m[0].scaling;
        torch::autograd::set_history(y, node);
        return THPVariable_Wrap(std::move(y));
    });
}

// moe(module, x, routing_weights, selected_experts, streaming): the routed forward; `streaming` asks for the weight-streaming
// form for a handful of tokens and nothing else (None where the call is differentiated or does not fit it)
PyObject* moe(PyObject*, PyObject* const* args, Py_ssize_t n) {
    return guarded([&]() -> PyObject* {
        if (n != 5) { PyErr_SetString(PyExc_TypeError, "moe(module, x, routing_weights, selected_experts, streaming)"); return nullptr; }
        const bool streaming = args[4] == Py_True;
        const Tensor *x = plain(args[1]), *rw = plain(args[2]), *sel = plain(args[3]);
        if (under_transform() || !x || !rw || !sel) XQ_NONE;
        PyObject* d = dict_of(args[0]);
        PyObject *params = get(d, N.s__parameters), *bufs = get(d, N.s__buffers), *sdt = get(d, N.s__scale_dtypes);
        PyObject* impl = get(d, N.s_moe_implementation);
        const int fmt = format_code(get(d, N.s_quant_format));
        int64_t rank, group, E, local, H, I;
        double alpha, limit = 0;
        if (!params || !bufs || !sdt || !PyDict_Check(sdt) || fmt < 0 || !as_defined(args[0], d, g_experts[fmt]) || !impl || !PyUnicode_Check(impl) ||
            PyUnicode_CompareWithASCIIString(impl, "eager") == 0 || !get_int(d, N.s_active_r, &rank) ||
            !get_number(d, N.s_active_lora_alpha, &alpha) || !get_int(d, N.s_quant_group_size, &group) || !get_int(d, N.s_num_experts, &E) ||
            !get_int(d, N.s_num_local_experts, &local) || local != E || !get_int(d, N.s_hidden_size, &H) ||
            !get_int(d, N.s_intermediate_size, &I) || rank < 1 || rank > 64)
            XQ_NONE;
        if (!get_number(d, N.s_swiglu_limit, &limit)) XQ_NONE;
        PyObject* rs = get(d, N.s_use_rslora);
        if (rs != Py_True && rs != Py_False) XQ_NONE;
        const double scaling = rs == Py_True ? alpha / std::sqrt((double)rank) : alpha / (double)rank;
        if (limit < 0) limit = 0;

        PyObject* const proj[3] = {N.s_gate, N.s_up, N.s_down};
        PyObject* const packed[3] = {N.s_gate_packed, N.s_up_packed, N.s_down_packed};
        PyObject* const bscales[3] = {N.s_gate_block_scales, N.s_up_block_scales, N.s_down_block_scales};
        PyObject* const scales[3] = {N.s_gate_scales, N.s_up_scales, N.s_down_scales};
        PyObject* const gscale[3] = {N.s_gate_global_scale, N.s_up_global_scale, N.s_down_global_scale};
        PyObject* const fA[3] = {N.s_gate_proj_lora_A, N.s_up_proj_lora_A, N.s_down_proj_lora_A};
        PyObject* const fB[3] = {N.s_gate_proj_lora_B, N.s_up_proj_lora_B, N.s_down_proj_lora_B};
        Weight q[3];
        Tensor A[3], B[3];
        bool factor_grad = false;
        for (int p = 0; p < 3; ++p) {
            PyObject* dts = get(sdt, proj[p]);
            if (!dts || !PyDict_Check(dts)) XQ_NONE;
            const bool blocks = fmt == XQ_FMT_FP8 || fmt == XQ_FMT_NVFP4;
            const int64_t K = p == 2 ? I : H, Nf = p == 2 ? H : I;
            if (!q[p].fill(fmt, XQ_LAYOUT_GKN, K, Nf, group, E, get(bufs, packed[p]), get(bufs, blocks ? bscales[p] : scales[p]),
                           get(dts, blocks ? N.s_weight_block_scales : N.s_weight_scales), get(bufs, gscale[p]),
                           get(dts, N.s_weight_global_scale)))
                XQ_NONE;
            const Tensor *a = plain(get(params, fA[p])), *b = plain(get(params, fB[p]));
            if (!a) a = plain(get(bufs, fA[p]));           // a projection that is not a LoRA target holds frozen zero factors
            if (!b) b = plain(get(bufs, fB[p]));
            if (!a || !b || a->dim() != 3 || b->dim() != 3 || a->size(2) != rank || b->size(1) != rank || a->size(1) != K || b->size(2) != Nf ||
                !a->is_contiguous() || !b->is_contiguous() || (a->scalar_type() != at::kFloat && a->scalar_type() != at::kBFloat16) ||
                a->scalar_type() != b->scalar_type() || q[p].packed.device() != x->device() || a->device() != x->device())
                XQ_NONE;
            A[p] = *a;
            B[p] = *b;
            if (A[p].scalar_type() != A[0].scalar_type()) XQ_NONE;
            factor_grad = factor_grad || a->requires_grad() || b->requires_grad();
        }
        if (x->scalar_type() != at::kBFloat16 || x->dim() < 1 || x->size(-1) != H || sel->dim() < 1) XQ_NONE;
        const int64_t topk = sel->size(-1);
        if (rw->scalar_type() != at::kFloat && rw->scalar_type() != at::kBFloat16) XQ_NONE;
        if (sel->scalar_type() != at::kLong && sel->scalar_type() != at::kInt) XQ_NONE;
        c10::DeviceGuard guard(x->device());
        const Rows xr(*x, H);
        const int64_t T = xr.M;
        if (topk < 1 || T < 1 || sel->numel() != T * topk || rw->numel() != T * topk || (uintptr_t)xr.ptr % 16 ||
            rw->device() != x->device() || sel->device() != x->device())
            XQ_NONE;
        const int r = (int)rank, rp = r_pad_of(r);
        const bool train = at::GradMode::is_enabled() && (x->requires_grad() || rw->requires_grad() || factor_grad);
        if (streaming && (train || !xq_grouped_infer_supported(&q[0].w, &q[1].w, &q[2].w, T, (int32_t)topk, r) || !xq_grouped_infer_shorter(&q[0].w, T, (int32_t)topk)))
            XQ_NONE;
        Tensor ids = sel->is_contiguous() ? *sel : sel->detach().contiguous();       // 64-bit ids as they are: a conversion would be a launch
        const int id_bytes = (int)ids.element_size();
        Tensor w = rw->is_contiguous() ? *rw : rw->detach().contiguous();
        const int rw_code = w.scalar_type() == at::kFloat ? XQ_DT_F32 : XQ_DT_BF16;
        xq_grouped_lora L;
        grouped_lora(&L, A, B, r, scaling, limit);
        Tensor out = empty_bf(x->sizes());
        void* stream = stream_of(*x);
        if (streaming) {
            Scratch ws(xq_grouped_infer_workspace_bytes(T, (int32_t)topk, (int32_t)E, H, I, r));
            {
                ReleaseGil nogil;
                check(xq_grouped_fwd_infer_ids(&q[0].w, &q[1].w, &q[2].w, &L, xr.ptr, xr.ld, T, w.data_ptr(), rw_code, ids.data_ptr(), id_bytes,
                      (int32_t)topk, out.data_ptr(), H, ws.get(), ws.bytes, stream));
            }
            return THPVariable_Wrap(std::move(out));
        }
        const int64_t R = T * topk;
        // where the banks allow it the routed rows are read in place: no [R, H] copy is kept for the backward
        const bool in_place = xq_grouped_in_place(&q[0].w, &q[1].w, &q[2].w);
        auto i32 = [](int64_t c) { return empty({c}, at::kInt); };
        Tensor kept[kGroupedKept] = {in_place ? empty_bf({0, H}) : empty_bf({R, H}), empty_bf({R, 2 * I}), empty_bf({R, I}), empty_f32({R}),
                                     empty_bf({R, rp}), empty_bf({R, rp}), empty_bf({R, rp}), i32(R), i32(E + 1), i32(2 * (E + 1)), i32(E)};
        xq_grouped_saved S;
        grouped_saved(&S, kept, nullptr);
        Scratch ws(xq_grouped_workspace_bytes(T, (int32_t)topk, (int32_t)E, H, I, r, 0));
        {
            ReleaseGil nogil;
            check((train ? xq_grouped_fwd_ids : xq_grouped_fwd_eval_ids)(&q[0].w, &q[1].w, &q[2].w, &L, xr.ptr, xr.ld, T, w.data_ptr(), rw_code,
                  ids.data_ptr(), id_bytes, (int32_t)topk, out.data_ptr(), H, &S, ws.get(), ws.bytes, stream));
        }
        if (!train) return THPVariable_Wrap(std::move(out));
        auto node = std::shared_ptr<QLoRAMoeBackward>(new QLoRAMoeBackward(), torch::autograd::deleteNode);
        node->set_next_edges(torch::autograd::collect_next_edges(*x, *rw, A[0], B[0], A[1], B[1], A[2], B[2]));
        node->x_ = SavedVariable(*x, false);
        for (int i = 0; i < kGroupedKept; ++i) node->kept_[i] = SavedVariable(kept[i], false);
        for (int p = 0; p < 3; ++p) {
            node->A_[p] = SavedVariable(A[p], false);
            node->B_[p] = SavedVariable(B[p], false);
            node->q[p] = q[p];
        }
        node->r = r;
        node->T = T;
        node->topk = topk;
        node->scaling = scaling;
        node->limit = limit;
        node->rw_dt = rw->scalar_type();
        node->rw_shape.assign(rw->sizes().begin(), rw->sizes().end());
        torch::autograd::set_history(out, node);
        return THPVariable_Wrap(std::move(out));
    });
}

// {format: (class, ((method name, method), ...))} -> programs by format
bool fill_programs(PyObject* table, Program* out) {
    PyObject *key, *entry;
    for (Py_ssize_t at = 0; PyDict_Next(table, &at, &key, &entry);) {
        const int fmt = format_code(key);
        PyObject *type, *methods;
        if (fmt < 0 || !PyArg_ParseTuple(entry, "O!O!", &PyType_Type, &type, &PyTuple_Type, &methods)) return false;
        Program p;
        p.type = (PyTypeObject*)type;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(methods); ++i) {
            PyObject *name, *method;
            if (!PyArg_ParseTuple(PyTuple_GET_ITEM(methods, i), "UO", &name, &method)) return false;
            Py_INCREF(name);
            PyUnicode_InternInPlace(&name);
            Py_INCREF(method);
            p.name.push_back(name);
            p.method.push_back(method);
        }
        Py_INCREF(type);
        out[fmt] = p;
    }
    return true;
}

// init(XqError, dict of xorl_amd.functional, programs of the linear modules, programs of the expert modules)
PyObject* init(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 4 || !PyDict_Check(args[1]) || !PyDict_Check(args[2]) || !PyDict_Check(args[3]) || !fill_programs(args[2], g_linear) ||
        !fill_programs(args[3], g_experts)) {
        PyErr_SetString(PyExc_TypeError, "init(error class, dict, linear programs, expert programs)");
        return nullptr;
    }
    for (Py_ssize_t i = 0; i < 2; ++i) Py_INCREF(args[i]);
    g_error = args[0];
    g_functional = args[1];
#define XQ_INTERN(m) N.s_##m = PyUnicode_InternFromString(#m);
    XQ_NAMES(XQ_INTERN)
#undef XQ_INTERN
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"init", (PyCFunction)(void (*)())init, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)())linear, METH_FASTCALL, nullptr},
    {"linears", (PyCFunction)(void (*)())linears, METH_FASTCALL, nullptr},
    {"mlp", (PyCFunction)(void (*)())mlp, METH_FASTCALL, nullptr},
    {"moe", (PyCFunction)(void (*)())moe, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "xq_torch", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_xq_torch() { return PyModule_Create(&module_def); }
