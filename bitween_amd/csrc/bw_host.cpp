// Host path of the Python package in native code: from a module call to the launch without the interpreter in between.
//
// A decode kernel runs for 3 ... 12 us, so what a call costs on the host decides how fast eager code decodes.  The same
// steps written in Python (views, checks, the output tensor, a ctypes call with sixteen arguments) took 8 ... 9 us a
// call, and an autograd node written in Python about 50 us per forward + backward.  Here: a layer's buffers are looked at
// on every call (dtype, shape, strides, device, address: about 0.1 us, so nothing about them has to be remembered), the
// output comes straight from the caching allocator, and the node that backward runs is a C++ node.
//
// The kernels are reached through function pointers of the C ABI (bind(), called once by hip_loader), so this file
// neither links the kernel library nor knows where it lies.  Anything a function here does not take - CPU tensors,
// tensor subclasses, buffers of another dtype or layout - it answers with None, and the Python code that it stands in
// front of deals with the call and raises what has to be raised.
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/function.h>
#include <torch/csrc/autograd/functions/utils.h>
#include <torch/csrc/autograd/python_cpp_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/autograd/saved_variable.h>
#include <torch/csrc/autograd/variable.h>

#include "../../include/bitween_hip.h"

namespace {

using at::Tensor;

struct Library {
    decltype(&bw_qlinear_ws) qlinear = nullptr;
    decltype(&bw_qlinear_workspace_bytes) qlinear_ws_bytes = nullptr;
    decltype(&bw_cast_bf16_f16) cast = nullptr;
    decltype(&bw_qdgrad) qdgrad = nullptr;
    decltype(&bw_qdgrad_workspace_bytes) qdgrad_ws_bytes = nullptr;
    decltype(&bw_qdgrad_tile_rows) qdgrad_tile_rows = nullptr;
    decltype(&bw_quantize_pack_add) quantize = nullptr;
    decltype(&bw_dequantize) dequantize = nullptr;
} lib;

PyObject* g_check = nullptr;          // Python: check(status, entry point's name) raises for a status other than 0
PyObject* g_limits = nullptr;         // Python: the dict with the row limits of the fused input gradient

PyObject *s_fused_rows, *s_fused_large_rows;
PyObject *s_buffers, *s_qweight, *s_scale, *s_zero, *s_bias, *s_bits, *s_group;

int dtype_code(at::ScalarType t) {
    switch (t) {
        case at::kHalf: return BW_F16;
        case at::kBFloat16: return BW_BF16;
        case at::kFloat: return BW_F32;
        case at::kInt: return BW_I32;
        case at::kDouble: return BW_F64;
        default: return -1;
    }
}

at::ScalarType dtype_of(int code) {
    switch (code) {
        case BW_F16: return at::kHalf;
        case BW_BF16: return at::kBFloat16;
        case BW_F32: return at::kFloat;
        case BW_F64: return at::kDouble;
        default: return at::kInt;
    }
}

inline bool aligned16(const void* p) { return ((uintptr_t)p & 15) == 0; }

inline Tensor empty(at::IntArrayRef sizes, at::ScalarType t, const at::Device& dev) {
    return Tensor(at::detail::empty_cuda(sizes, t, dev, std::nullopt));
}

inline void* stream_of(at::DeviceIndex index) { return (void*)c10::hip::getCurrentHIPStream(index).stream(); }

// The device of a call made current, only where it is not already.
struct OnDevice {
    std::optional<c10::DeviceGuard> guard;
    explicit OnDevice(const at::Device& d) {
        if (c10::hip::current_device() != d.index()) guard.emplace(d);
    }
};

// The interpreter lock given up while a call allocates, plans and launches: a full queue or an allocator that goes to the driver would
// hold every other Python thread up.  Nothing between here and the end of its scope touches a Python object.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    Unlocked() = default;
    Unlocked(const Unlocked&) = delete;
    ~Unlocked() { PyEval_RestoreThread(state); }
};

// The row limits as they are now (0 = not a number: no row runs fused); takes the interpreter lock where the thread does not hold it.
struct FusedRows {
    int64_t always = 0, large = 0;
    FusedRows() {
        const PyGILState_STATE state = PyGILState_Ensure();
        always = read(s_fused_rows);
        large = read(s_fused_large_rows);
        PyGILState_Release(state);
    }
    static int64_t read(PyObject* name) {
        PyObject* v = g_limits ? PyDict_GetItemWithError(g_limits, name) : nullptr;
        const long long rows = v && PyLong_Check(v) ? PyLong_AsLongLong(v) : 0;
        if (PyErr_Occurred()) PyErr_Clear();
        return rows < 0 ? 0 : rows;
    }
};

struct Layer {
    const void *qweight, *scale, *zero, *bias;
    int64_t n, k;
    int bits, group;
    at::DeviceIndex device;
};

// What the kernels ask of a layer's buffers; false = the general Python path has to look at them.
bool layer_of(const Tensor& qweight, const Tensor& scale, const Tensor& zero, const Tensor* bias, int64_t bits, int64_t group, Layer& l) {
    if (!lib.qlinear || (bits != 2 && bits != 4 && bits != 8) || group < 1) return false;
    if (!qweight.is_cuda() || !qweight.has_storage() || qweight.scalar_type() != at::kInt || qweight.dim() != 2 || !qweight.is_contiguous()) return false;
    const int64_t n = qweight.size(0), k = qweight.size(1) * (32 / bits);
    if (n < 1 || k < 1 || k % group) return false;
    for (const Tensor* t : {&scale, &zero})
        if (t->device() != qweight.device() || t->scalar_type() != at::kHalf || t->dim() != 2 || !t->is_contiguous() || t->size(0) != n ||
            t->size(1) != k / group)
            return false;
    if (bias && (bias->device() != qweight.device() || bias->scalar_type() != at::kHalf || bias->dim() != 1 || bias->size(0) != n ||
                 !bias->is_contiguous()))
        return false;
    l = {qweight.const_data_ptr(), scale.const_data_ptr(), zero.const_data_ptr(), bias ? bias->const_data_ptr() : nullptr,
         n, k, (int)bits, (int)group, qweight.device().index()};
    return true;
}

// x.to(float16) of a bfloat16 matrix [m, k] with row pitch ldx: the library's streaming kernel where the layout qualifies.
Tensor cast_to_f16(const Tensor& x, int64_t m, int64_t k, int64_t ldx, void* stream) {
    if (k % 8 == 0 && ldx % 8 == 0 && aligned16(x.const_data_ptr())) {
        Tensor y = empty({m, k}, at::kHalf, x.device());
        if (lib.cast(x.const_data_ptr(), m, k, ldx, y.mutable_data_ptr(), k, stream) == BW_OK) return y;
    }
    return x.to(at::kHalf).contiguous();
}

// y = x W16^T (+ bias); the result keeps x's leading dimensions.  An undefined tensor with status 0 = not taken here.
Tensor linear(const Layer& l, Tensor x, int& status, const char*& what) {
    status = 0;
    if (!x.is_cuda() || x.device().index() != l.device || x.dim() < 1 || x.size(-1) != l.k || x.numel() == 0) return {};
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = l.n;
    OnDevice on(x.device());
    at::ScalarType t = x.scalar_type();
    if (t != at::kHalf && t != at::kBFloat16) {
        x = x.to(at::kHalf);
        t = at::kHalf;
    }
    const int64_t m = x.numel() / l.k;
    int64_t ldx = l.k;
    if (!x.is_contiguous()) {
        if (x.dim() != 2) x = x.reshape({m, l.k});
        if (x.stride(1) == 1 && x.stride(0) >= l.k) ldx = x.stride(0);
        else x = x.contiguous();
    }
    if ((ldx * 2) % 16 || !aligned16(x.const_data_ptr())) {
        x = x.clone(at::MemoryFormat::Contiguous);
        ldx = l.k;
    }
    void* stream = stream_of(l.device);
    Tensor y = empty(shape, at::kHalf, x.device());
    what = "bw_qlinear_ws";
    auto launch = [&](int act) {
        const size_t bytes = lib.qlinear_ws_bytes(m, l.n, l.k, l.bits, l.group, act);
        Tensor ws;
        if (bytes) ws = empty({(int64_t)bytes}, at::kByte, x.device());
        return lib.qlinear(x.const_data_ptr(), act, m, l.k, ldx, (const int32_t*)l.qweight, l.scale, l.zero, l.bias, l.n, l.bits, l.group,
                           y.mutable_data_ptr(), l.n, bytes ? ws.mutable_data_ptr() : nullptr, bytes, stream);
    };
    status = launch(t == at::kHalf ? BW_F16 : BW_BF16);
    if (t == at::kBFloat16 && (status == BW_EUNSUPPORTED || status == BW_EALIGN || status == BW_EWORKSPACE)) {
        x = cast_to_f16(x, m, l.k, ldx, stream);               // a shape or layout that wants float16 in memory
        ldx = l.k;
        status = launch(BW_F16);
    }
    return y;
}

// grad_x = grad_y @ W, W the dequantised weight in grad_y's dtype (bitween/modules.py:108-141).  float16 / bfloat16
// gradients run the fused kernel - up to `fused.always` rows always, up to `fused.large` where the library plans its
// 256 x 256 kernel - and dequantise + library GEMM beyond, which is faster there; so does a backward that is itself
// recorded (create_graph).
Tensor input_grad(const Tensor& go, const Tensor& qweight, const Tensor& scale, const Tensor& zero, int bits, int group, const FusedRows& fused) {
    const int64_t n = qweight.size(0), k = qweight.size(1) * (32 / bits);
    OnDevice on(go.device());
    void* stream = stream_of(go.device().index());
    const at::ScalarType t = go.scalar_type();
    const int64_t m = go.numel() / n;
    const bool recorded = c10::GradMode::is_enabled() && go.requires_grad();
    if ((t == at::kHalf || t == at::kBFloat16) && !recorded && m > 0 &&
        (m <= fused.always || (m <= fused.large && lib.qdgrad_tile_rows(m, n, k, bits, group) == 257))) {
        Tensor g = go;
        int64_t ldg = n;
        if (!g.is_contiguous()) {
            if (g.dim() != 2) g = g.reshape({m, n});
            if (g.stride(1) == 1 && g.stride(0) >= n) ldg = g.stride(0);
            else g = g.contiguous();
        }
        if (n >= 32) {
            c10::SmallVector<int64_t, 5> shape(go.sizes().begin(), go.sizes().end());
            shape.back() = k;
            Tensor gx = empty(shape, t, go.device());
            const size_t bytes = lib.qdgrad_ws_bytes(m, n, k, bits, group);
            Tensor ws;
            if (bytes) ws = empty({(int64_t)bytes}, at::kByte, go.device());
            const int st = lib.qdgrad(g.const_data_ptr(), dtype_code(t), m, n, ldg, (const int32_t*)qweight.const_data_ptr(),
                                      scale.const_data_ptr(), zero.const_data_ptr(), k, bits, group, gx.mutable_data_ptr(), k,
                                      bytes ? ws.mutable_data_ptr() : nullptr, bytes, stream);
            if (st == BW_OK) return gx;
            TORCH_CHECK(st == BW_EUNSUPPORTED || st == BW_EALIGN, "bw_qdgrad failed (status ", st, ")");
        }
    }
    // W = scale * (q - zp) in float32, cast to grad_output's dtype: the float32 product is exact, so dequantising straight
    // to that dtype gives the same bits
    const at::ScalarType wt = (t == at::kHalf || t == at::kBFloat16 || t == at::kFloat) ? t : at::kFloat;
    Tensor w = empty({n, k}, wt, go.device());
    const int st = lib.dequantize((const int32_t*)qweight.const_data_ptr(), scale.const_data_ptr(), BW_F16, zero.const_data_ptr(), BW_F16, n, k,
                                  bits, group, w.mutable_data_ptr(), dtype_code(wt), k, stream);
    TORCH_CHECK(st == BW_OK, "bw_dequantize failed (status ", st, ")");
    return at::matmul(go, wt == t ? w : w.to(t));
}

// The node of a recorded forward, in the likeness of QuantizedLinearFunction's: its name, what it saves (x too, so that a change of x in
// place is noticed, and saved-tensor hooks see it) and the edges it has.
struct QuantizedLinearBackward : public torch::autograd::Node {
    enum { X, QWEIGHT, SCALE, ZERO, BIAS };
    torch::autograd::SavedVariable saved[5];
    bool has_bias = false;
    int bits = 0, group = 0;
    std::string name() const override { return "QuantizedLinearFunctionBackward"; }
    void release_variables() override {
        std::lock_guard<std::mutex> lock(mutex_);
        for (auto& v : saved) v.reset_data();
    }
    std::array<Tensor, 5> unpack() const {
        std::array<Tensor, 5> t;
        for (int i = 0; i < (has_bias ? 5 : 4); i++) t[i] = saved[i].unpack();
        return t;
    }
    torch::autograd::variable_list apply(torch::autograd::variable_list&& grads) override {
        const FusedRows fused;
        std::lock_guard<std::mutex> lock(mutex_);
        const auto t = unpack();
        torch::autograd::variable_list out(has_bias ? 5 : 4);
        if (!task_should_compute_output(0)) return out;
        const Tensor go = grads[0].defined() ? grads[0] : input_metadata(0).zeros_like();
        out[0] = input_grad(go, t[QWEIGHT].contiguous(), t[SCALE].contiguous(), t[ZERO].contiguous(), bits, group, fused);
        return out;
    }
};

QuantizedLinearBackward* node_of(PyObject* self) {
    return static_cast<QuantizedLinearBackward*>(reinterpret_cast<torch::autograd::THPCppFunction*>(self)->cdata.get());
}

PyObject* node_saved_tensors(PyObject* self, void*) {
    HANDLE_TH_ERRORS
    QuantizedLinearBackward* node = node_of(self);
    const auto t = node->unpack();
    PyObject* r = PyTuple_New(5);
    if (!r) return nullptr;
    for (int i = 0; i < 5; i++) PyTuple_SET_ITEM(r, i, THPVariable_Wrap(t[i]));   // (an undefined tensor is None)
    return r;
    END_HANDLE_TH_ERRORS
}

PyObject* node_needs_input_grad(PyObject* self, void*) {
    QuantizedLinearBackward* node = node_of(self);
    PyObject* r = PyTuple_New(7);
    if (!r) return nullptr;
    for (uint32_t i = 0; i < 7; i++)
        PyTuple_SET_ITEM(r, i, PyBool_FromLong(i < node->num_outputs() && node->task_should_compute_output(i)));
    return r;
}

using namespace torch::autograd;                              // (the names of the next macro)
PyGetSetDef node_properties[] = {THP_FUNCTION_DEFAULT_PROPERTIES,
                                 {"saved_tensors", node_saved_tensors, nullptr, nullptr, nullptr},
                                 {"needs_input_grad", node_needs_input_grad, nullptr, nullptr, nullptr},
                                 {"bits", [](PyObject* self, void*) { return PyLong_FromLong(node_of(self)->bits); }, nullptr, nullptr, nullptr},
                                 {"group_size", [](PyObject* self, void*) { return PyLong_FromLong(node_of(self)->group); }, nullptr, nullptr, nullptr},
                                 {nullptr, nullptr, nullptr, nullptr, nullptr}};
PyTypeObject node_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- Python side ----

// A plain tensor or parameter; subclasses have their own ideas of every operation and go through Python.
inline bool plain(PyObject* o) { return THPVariable_CheckExact(o); }
inline const Tensor& unpack(PyObject* o) { return THPVariable_Unpack(o); }

PyObject* none() { Py_RETURN_NONE; }

PyObject* checked(Tensor y, int status, const char* what) {
    if (status == 0) return y.defined() ? THPVariable_Wrap(std::move(y)) : none();
    PyObject* r = PyObject_CallFunction(g_check, "is", status, what);   // raises
    Py_XDECREF(r);
    if (!PyErr_Occurred()) PyErr_SetString(PyExc_RuntimeError, what);
    return nullptr;
}

// The C++ exceptions of torch as Python ones.
template <class F>
PyObject* guarded(F&& f) {
    HANDLE_TH_ERRORS
    return f();
    END_HANDLE_TH_ERRORS
}

// The module's buffers as they are now; false = the general path (or, with a Python error set, none).
struct Module {
    Tensor qweight, scale, zero, bias;                         // held: the interpreter may run while a call is under way
    Layer layer;
};

bool module_of(PyObject* dict, Module& m) {
    PyObject* buffers = PyDict_GetItemWithError(dict, s_buffers);
    PyObject *bits = PyDict_GetItemWithError(dict, s_bits), *group = PyDict_GetItemWithError(dict, s_group);
    if (!buffers || !PyDict_Check(buffers) || !bits || !group || !PyLong_Check(bits) || !PyLong_Check(group)) return false;
    PyObject* names[4] = {s_qweight, s_scale, s_zero, s_bias};
    Tensor* out[4] = {&m.qweight, &m.scale, &m.zero, &m.bias};
    for (int i = 0; i < 4; i++) {
        PyObject* t = PyDict_GetItemWithError(buffers, names[i]);
        if (i == 3 && (!t || t == Py_None)) break;
        if (!t || !plain(t)) return false;
        *out[i] = unpack(t);
    }
    const long b = PyLong_AsLong(bits), g = PyLong_AsLong(group);
    return !PyErr_Occurred() && layer_of(m.qweight, m.scale, m.zero, m.bias.defined() ? &m.bias : nullptr, b, g, m.layer);
}

// forward(module.__dict__, x) -> y or None
PyObject* py_forward(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject* {
        if (nargs != 2 || !PyDict_Check(args[0]) || !plain(args[1])) return none();
        const Tensor x = unpack(args[1]);
        if (!x.is_cuda() || !x.has_storage()) return none();    // (no storage: a wrapper of vmap or torch.func)
        Module l;
        if (!module_of(args[0], l)) {
            if (PyErr_Occurred()) return nullptr;
            return none();
        }
        int status = 0;
        const char* what = "";
        const bool recorded = c10::GradMode::is_enabled() && x.requires_grad();
        if (recorded && x._fw_grad(0).defined()) return none();   // the Python function refuses forward-mode derivatives
        Tensor y;
        {
            Unlocked unlocked;
            c10::AutoGradMode off(false);
            y = linear(l.layer, x, status, what);
        }
        if (recorded && status == 0 && y.defined()) {
            std::shared_ptr<QuantizedLinearBackward> node(new QuantizedLinearBackward(), torch::autograd::deleteNode);
            const Tensor* inputs[5] = {&x, &l.qweight, &l.scale, &l.zero, &l.bias};
            node->has_bias = l.bias.defined();
            node->set_next_edges(node->has_bias ? torch::autograd::collect_next_edges(x, l.qweight, l.scale, l.zero, l.bias)
                                                : torch::autograd::collect_next_edges(x, l.qweight, l.scale, l.zero));
            for (int i = 0; i < (node->has_bias ? 5 : 4); i++) node->saved[i] = torch::autograd::SavedVariable(*inputs[i], false);
            node->bits = l.layer.bits;
            node->group = l.layer.group;
            torch::autograd::set_history(y, node);
        }
        return checked(std::move(y), status, what);
    });
}

// matmul(x, qweight, scale, zero_point, bias, bits, group_size) -> y or None
PyObject* py_matmul(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject* {
        if (nargs != 7 || !PyLong_Check(args[5]) || !PyLong_Check(args[6])) return none();
        for (int i = 0; i < 5; i++)
            if (!plain(args[i]) && !(i == 4 && args[i] == Py_None)) return none();
        const Tensor x = unpack(args[0]);
        if (!x.has_storage() || (x.scalar_type() != at::kHalf && x.scalar_type() != at::kBFloat16)) return none();
        const Tensor qweight = unpack(args[1]), scale = unpack(args[2]), zero = unpack(args[3]), bias = args[4] == Py_None ? Tensor() : unpack(args[4]);
        const int64_t bits = PyLong_AsLong(args[5]), group = PyLong_AsLong(args[6]);
        if (PyErr_Occurred()) return nullptr;
        Layer l;
        if (!layer_of(qweight, scale, zero, bias.defined() ? &bias : nullptr, bits, group, l)) return none();
        int status = 0;
        const char* what = "";
        Tensor y;
        {
            Unlocked unlocked;
            c10::AutoGradMode off(false);
            y = linear(l, x, status, what);
        }
        return checked(std::move(y), status, what);
    });
}

// input_grad(grad_output, qweight, scale, zero_point, bits, group_size) -> grad_input or None
PyObject* py_input_grad(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject* {
        if (nargs != 6 || !PyLong_Check(args[4]) || !PyLong_Check(args[5])) return none();
        for (int i = 0; i < 4; i++)
            if (!plain(args[i])) return none();
        const Tensor go = unpack(args[0]), qweight = unpack(args[1]), scale = unpack(args[2]), zero = unpack(args[3]);
        const int64_t bits = PyLong_AsLong(args[4]), group = PyLong_AsLong(args[5]);
        if (PyErr_Occurred()) return nullptr;
        Layer l;
        if (!go.is_cuda() || !go.has_storage() || !layer_of(qweight, scale, zero, nullptr, bits, group, l)) return none();
        if (go.dim() < 1 || go.size(-1) != l.n || !go.is_floating_point() || go.device().index() != l.device) return none();
        const FusedRows fused;
        Tensor gx;
        {
            Unlocked unlocked;
            gx = input_grad(go, qweight, scale, zero, l.bits, l.group, fused);
        }
        return THPVariable_Wrap(std::move(gx));
    });
}

// quantize(weight, delta or None, bits, group_size, math code with flags, scale code, zero-point code) -> (qweight, scale, zero_point) or None
PyObject* py_quantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject* {
        if (nargs != 7 || !plain(args[0]) || !(args[1] == Py_None || plain(args[1]))) return none();
        Tensor w = unpack(args[0]), delta = args[1] == Py_None ? Tensor() : unpack(args[1]);
        const int64_t bits = PyLong_AsLong(args[2]), group = PyLong_AsLong(args[3]);
        const int math = (int)PyLong_AsLong(args[4]), sc = (int)PyLong_AsLong(args[5]), zc = (int)PyLong_AsLong(args[6]);
        if (PyErr_Occurred()) return nullptr;
        const int code = dtype_code(w.scalar_type());
        if (!lib.quantize || !w.is_cuda() || w.dim() != 2 || code < 0 || (bits != 2 && bits != 4 && bits != 8) || group < 1) return none();
        if (delta.defined() && (delta.device() != w.device() || delta.sizes() != w.sizes() || delta.scalar_type() != w.scalar_type())) return none();
        Tensor q, s, z;
        int st;
        {
            Unlocked unlocked;
            c10::AutoGradMode off(false);
            if (w.stride(1) != 1) w = w.contiguous();
            if (delta.defined() && delta.stride(1) != 1) delta = delta.contiguous();
            const int64_t n = w.size(0), k = w.size(1);
            OnDevice on(w.device());
            q = empty({n, k / (32 / bits)}, at::kInt, w.device());
            s = empty({n, k / group}, dtype_of(sc), w.device());
            z = empty({n, k / group}, dtype_of(zc), w.device());
            st = lib.quantize(w.const_data_ptr(), delta.defined() ? delta.const_data_ptr() : nullptr, code, math, n, k, w.stride(0),
                              delta.defined() ? delta.stride(0) : 0, (int)bits, (int)group, (int32_t*)q.mutable_data_ptr(),
                              s.mutable_data_ptr(), sc, z.mutable_data_ptr(), zc, stream_of(w.device().index()));
        }
        if (st) return checked({}, st, "bw_quantize_pack");
        PyObject* r = PyTuple_New(3);
        if (!r) return nullptr;
        PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(q)));
        PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(s)));
        PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(std::move(z)));
        return r;
    });
}

// dequantize(qweight, scale, zero_point, group_size, bits, output code) -> weight or None
PyObject* py_dequantize(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&]() -> PyObject* {
        if (nargs != 6 || !plain(args[0]) || !plain(args[1]) || !plain(args[2])) return none();
        const int64_t group = PyLong_AsLong(args[3]), bits = PyLong_AsLong(args[4]);
        const int oc = (int)PyLong_AsLong(args[5]);
        if (PyErr_Occurred()) return nullptr;
        Tensor q = unpack(args[0]), s = unpack(args[1]), z = unpack(args[2]), w;
        const int sc = dtype_code(s.scalar_type()), zc = dtype_code(z.scalar_type());
        if (!lib.dequantize || !q.is_cuda() || s.device() != q.device() || z.device() != q.device() || q.scalar_type() != at::kInt || q.dim() != 2 ||
            sc < 0 || zc < 0 || (bits != 2 && bits != 4 && bits != 8) || group < 1)
            return none();
        const int64_t n = q.size(0), k = q.size(1) * (32 / bits);
        if (s.numel() < n * (k / group) || z.numel() < n * (k / group)) return none();
        int st;
        {
            Unlocked unlocked;
            c10::AutoGradMode off(false);
            q = q.contiguous();
            s = s.contiguous();
            z = z.contiguous();
            OnDevice on(q.device());
            w = empty({n, k}, dtype_of(oc), q.device());
            st = lib.dequantize((const int32_t*)q.const_data_ptr(), s.const_data_ptr(), sc, z.const_data_ptr(), zc, n, k, (int)bits, (int)group,
                                w.mutable_data_ptr(), oc, k, stream_of(q.device().index()));
        }
        return checked(std::move(w), st, "bw_dequantize");
    });
}

// bind({entry point name: address}, check, dict with the fused gradient's row limits): once, after the kernel library is loaded
PyObject* py_bind(PyObject*, PyObject* args) {
    PyObject *table, *check, *limits;
    if (!PyArg_ParseTuple(args, "O!OO!", &PyDict_Type, &table, &check, &PyDict_Type, &limits)) return nullptr;
    bool ok = true;
    auto get = [&](auto& fn, const char* name) {
        PyObject* v = PyDict_GetItemString(table, name);
        void* p = v ? PyLong_AsVoidPtr(v) : nullptr;
        if (!p) ok = false;
        fn = reinterpret_cast<std::decay_t<decltype(fn)>>(p);
    };
    Library l;
    get(l.qlinear, "bw_qlinear_ws");
    get(l.qlinear_ws_bytes, "bw_qlinear_workspace_bytes");
    get(l.cast, "bw_cast_bf16_f16");
    get(l.qdgrad, "bw_qdgrad");
    get(l.qdgrad_ws_bytes, "bw_qdgrad_workspace_bytes");
    get(l.qdgrad_tile_rows, "bw_qdgrad_tile_rows");
    get(l.quantize, "bw_quantize_pack_add");
    get(l.dequantize, "bw_dequantize");
    if (PyErr_Occurred()) return nullptr;
    if (!ok) {
        PyErr_SetString(PyExc_RuntimeError, "bind: an entry point is missing");
        return nullptr;
    }
    lib = l;
    Py_INCREF(check);
    Py_XSETREF(g_check, check);
    Py_INCREF(limits);
    Py_XSETREF(g_limits, limits);
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", py_bind, METH_VARARGS, nullptr},
    {"forward", (PyCFunction)(void*)py_forward, METH_FASTCALL, nullptr},
    {"matmul", (PyCFunction)(void*)py_matmul, METH_FASTCALL, nullptr},
    {"input_grad", (PyCFunction)(void*)py_input_grad, METH_FASTCALL, nullptr},
    {"quantize", (PyCFunction)(void*)py_quantize, METH_FASTCALL, nullptr},
    {"dequantize", (PyCFunction)(void*)py_dequantize, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_bw_host", "Native host path of bitween_amd", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__bw_host() {
    s_fused_rows = PyUnicode_InternFromString("FUSED_DGRAD_MAX_ROWS");
    s_fused_large_rows = PyUnicode_InternFromString("FUSED_DGRAD_LARGE_MAX_ROWS");
    s_buffers = PyUnicode_InternFromString("_buffers");
    s_qweight = PyUnicode_InternFromString("qweight");
    s_scale = PyUnicode_InternFromString("scale");
    s_zero = PyUnicode_InternFromString("zero_point");
    s_bias = PyUnicode_InternFromString("bias");
    s_bits = PyUnicode_InternFromString("bits");
    s_group = PyUnicode_InternFromString("group_size");
    HANDLE_TH_ERRORS
    torch::autograd::_initFunctionPyTypeObject(node_type, "QuantizedLinearFunctionBackward", node_properties, nullptr);
    torch::autograd::registerCppFunction(typeid(QuantizedLinearBackward), &node_type);
    return PyModule_Create(&module_def);
    END_HANDLE_TH_ERRORS
}
