// native_calls.cpp -- the Python module innova_amd._native: the ordinary form of the package's calls without the interpreter.
//
// A small call is bound by the host.  Of a GEMV call's 6.3 to 6.8 us (1000 x 1280, one row, eager) the launch takes 3.6; the rest is Python:
// the output through Tensor.new_empty 1.55, the checks 0.3, ctypes and attribute look-ups 0.7.  Here the checks, the output, the current
// stream and the call are one C function.  It takes only the ordinary form: exact torch tensors on the GPU, of the right type,
// contiguous, plain ints, no torch mode in force, no graph capture that needs a workspace.  Anything else, and any C++ exception, makes it return None,
// and the caller in Python does what it always did, with its own checks and errors.
#include <Python.h>
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>

#include <algorithm>
#include <type_traits>

#include "../../include/oilhip.h"

namespace {

// what makes a function return None
struct NotOrdinary {};
inline void need(bool ok) { if (!ok) throw NotOrdinary{}; }

void need_no_modes() {
    need(!at::impl::torch_function_mode_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set());
}
const at::Tensor& tensor(PyObject* o) {
    need(THPVariable_CheckExact(o));
    const at::Tensor& t = THPVariable_Unpack(o);
    need(t.is_cuda() && t.is_contiguous());
    return t;
}
const at::Tensor& tensor(PyObject* o, at::ScalarType type) {
    const at::Tensor& t = tensor(o);
    need(t.scalar_type() == type);
    return t;
}
long long integer(PyObject* o) {
    need(PyLong_CheckExact(o));
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); throw NotOrdinary{}; }
    return v;
}
long long size(PyObject* o) {
    const long long v = integer(o);
    need(v >= 0 && v <= 0x7FFFFFFF);
    return v;
}
template <class T>
T* handle(PyObject* o) {
    need(PyLong_CheckExact(o));
    void* p = PyLong_AsVoidPtr(o);
    if (!p) { PyErr_Clear(); throw NotOrdinary{}; }
    return static_cast<T*>(p);
}
void* stream() { return c10::hip::getCurrentHIPStream().stream(); }
// a call of several rows under capture gets a workspace from the graph's pool, which the caller in Python arranges
void need_no_capture(void* s) {
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    need(hipStreamIsCapturing(static_cast<hipStream_t>(s), &status) == hipSuccess && status == hipStreamCaptureStatusNone);
}
at::Tensor empty(at::IntArrayRef sizes, const at::Tensor& like) { return at::empty(sizes, like.options().dtype(at::kFloat)); }
// activations of whole rows of `cols`: how many
int64_t rows_of(const at::Tensor& x, int64_t cols) {
    need(cols > 0 && x.numel() > 0 && x.numel() % cols == 0 && x.numel() / cols <= 0x7FFFFFFF);
    return x.numel() / cols;
}
// `out` when the caller brought one, else a new tensor
at::Tensor output(PyObject* out, at::IntArrayRef sizes, const at::Tensor& like) {
    if (out == Py_None) return empty(sizes, like);
    const at::Tensor& t = tensor(out, at::kFloat);
    int64_t n = 1;
    for (int64_t s : sizes) n *= s;
    need(t.numel() == n);
    return t;
}
float* f32(const at::Tensor& t) { return static_cast<float*>(t.data_ptr()); }
uint8_t* u8(const at::Tensor& t) { return static_cast<uint8_t*>(t.data_ptr()); }

PyObject* raise(int rc) {
    PyObject* m = PyImport_ImportModule("innova_amd._lib");
    PyObject* cls = m ? PyObject_GetAttrString(m, "OilHipError") : nullptr;
    if (cls) PyErr_Format(cls, "liboilhip error %d: %s", rc, oilhip_last_error());
    Py_XDECREF(cls);
    Py_XDECREF(m);
    return nullptr;
}
// The library's `f` without the interpreter's lock.  Its arguments are plain values, worked out while the lock is held: data_ptr() raises
// for a tensor without storage (those of torch.func's transforms), and nothing may be thrown past a lock that is not taken again.
struct Unlocked {
    PyThreadState* state = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(state); }
};
template <class... P, class... A>
int without_gil(int (*f)(P...), A... a) {
    static_assert((std::is_scalar_v<A> && ...), "pointers and numbers, not what they are read from");
    const Unlocked unlocked;
    return f(a...);
}
// `f` as a Python function: None for what it does not take, an OilHipError for a failed call
template <class F>
PyObject* ordinary(Py_ssize_t n, Py_ssize_t want, F&& f) {
    if (n != want) { PyErr_Format(PyExc_TypeError, "%zd arguments, %zd wanted", n, want); return nullptr; }
    try {
        need_no_modes();
        return f();
    } catch (...) {
    }
    Py_RETURN_NONE;
}
PyObject* result(int rc, PyObject* given, const at::Tensor& t) {
    if (rc) return raise(rc);
    if (given == Py_None) return THPVariable_Wrap(t);
    Py_INCREF(given);
    return given;
}

// gemv(weights, x, out, rows, cols)
PyObject* gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 5, [&]() -> PyObject* {
        const auto* w = handle<oilhip_weights>(a[0]);
        const at::Tensor& x = tensor(a[1], at::kFloat);
        const int64_t M = rows_of(x, size(a[4]));
        void* s = stream();
        if (M > 1) need_no_capture(s);
        const at::Tensor y = output(a[2], {M, size(a[3])}, x);
        return result(without_gil(oilhip_gemv_f32, w, f32(x), f32(y), (int)M, s), a[2], y);
    });
}
// gemm(weights, x, out, rows, cols, bf16)
PyObject* gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 6, [&]() -> PyObject* {
        const auto* w = handle<oilhip_weights>(a[0]);
        const bool bf16 = integer(a[5]) != 0;
        const at::Tensor& x = tensor(a[1], bf16 ? at::kBFloat16 : at::kFloat);
        const int64_t M = rows_of(x, size(a[4]));
        const at::Tensor y = output(a[2], {M, size(a[3])}, x);
        void* s = stream();
        const int rc = bf16 ? without_gil(oilhip_gemm_bf16, w, static_cast<const uint16_t*>(x.data_ptr()), f32(y), (int)M, s)
                            : without_gil(oilhip_gemm_f32, w, f32(x), f32(y), (int)M, s);
        return result(rc, a[2], y);
    });
}
// dequant(weights, rows, cols) into a new tensor
PyObject* dequant(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 3, [&]() -> PyObject* {
        const auto* w = handle<oilhip_weights>(a[0]);
        const at::Tensor y = at::empty({size(a[1]) * size(a[2])}, at::TensorOptions().dtype(at::kFloat).device(at::kCUDA, c10::hip::current_device()));
        void* s = stream();
        return result(without_gil(oilhip_dequant_f32, w, f32(y), s), Py_None, y);
    });
}
// embed_rows(weights, ids, cols) into a new tensor
PyObject* embed_rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 3, [&]() -> PyObject* {
        const auto* w = handle<oilhip_weights>(a[0]);
        const at::Tensor& ids = tensor(a[1], at::kInt);
        need(ids.numel() <= 0x7FFFFFFF);
        const at::Tensor y = empty({ids.numel(), size(a[2])}, ids);
        void* s = stream();
        return result(without_gil(oilhip_embed_rows_f32, w, static_cast<const int*>(ids.data_ptr()), (int)ids.numel(), f32(y), s), Py_None, y);
    });
}
// gemv_rmsnorm(weights, x, norm_w, out, rows, cols)
PyObject* gemv_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 6, [&]() -> PyObject* {
        const auto* w = handle<oilhip_weights>(a[0]);
        const at::Tensor &x = tensor(a[1], at::kFloat), &nw = tensor(a[2], at::kFloat);
        const int64_t M = rows_of(x, size(a[5]));
        void* s = stream();
        if (M > 1) need_no_capture(s);
        const at::Tensor y = output(a[3], {M, size(a[4])}, x), xn = empty(x.sizes(), x);
        return result(without_gil(oilhip_gemv_rmsnorm_f32, w, f32(x), f32(nw), f32(y), (int)M, f32(xn), s), a[3], y);
    });
}
// mlp_step(gate_up, down, x, norm_w or None, out, rows of down, cols of gate_up, cols of down)
PyObject* mlp_step(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 8, [&]() -> PyObject* {
        const auto *gu = handle<oilhip_weights>(a[0]), *down = handle<oilhip_weights>(a[1]);
        const at::Tensor& x = tensor(a[2], at::kFloat);
        const float* nw = a[3] == Py_None ? nullptr : f32(tensor(a[3], at::kFloat));
        const int64_t D = size(a[6]), F = size(a[7]), M = rows_of(x, D);
        void* s = stream();
        if (M > 1) need_no_capture(s);
        const at::Tensor y = output(a[4], {M, size(a[5])}, x), scratch = empty({(3 * F + D) * M}, x);
        return result(without_gil(oilhip_mlp_step_f32, gu, down, f32(x), nw, f32(y), (int)M, f32(scratch), s), a[4], y);
    });
}
// oil8_gemm / oil4_gemm(codes, codebook, activations, M, N, K)
template <class Book>
PyObject* flat_gemm(PyObject* const* a, Py_ssize_t n, int (*f)(const uint8_t*, const Book*, const float*, float*, int, int, int, void*)) {
    return ordinary(n, 6, [&]() -> PyObject* {
        const at::Tensor &codes = tensor(a[0]), &cb = tensor(a[1]), &x = tensor(a[2]);
        const int M = (int)size(a[3]), N = (int)size(a[4]), K = (int)size(a[5]);
        const at::Tensor y = empty({M, N}, x);
        void* s = stream();
        return result(without_gil(f, u8(codes), static_cast<const Book*>(cb.data_ptr()), f32(x), f32(y), M, N, K, s), Py_None, y);
    });
}
PyObject* oil8_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) { return flat_gemm(a, n, oilhip_flat_oil8_gemm); }
PyObject* oil4_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) { return flat_gemm(a, n, oilhip_flat_oil4_gemm); }
// prod(bits, codes, codebook or None, scale, activations, M, N, K): M weight rows, N activation rows
PyObject* prod(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 8, [&]() -> PyObject* {
        const long long bits = integer(a[0]);
        const at::Tensor &w = tensor(a[1]), &x = tensor(a[4]);
        void* cb = a[2] == Py_None ? nullptr : tensor(a[2]).data_ptr();
        need(PyFloat_CheckExact(a[3]) && (bits == 2 || (cb && (bits == 4 || bits == 8))));
        const float scale = (float)PyFloat_AS_DOUBLE(a[3]);
        const int M = (int)size(a[5]), N = (int)size(a[6]), K = (int)size(a[7]);
        const at::Tensor y = empty({N, M}, x);
        void* s = stream();
        const int rc = bits == 2 ? without_gil(oilhip_prod_gemv_spark, u8(w), scale, f32(x), f32(y), M, K, N, s)
                     : bits == 4 ? without_gil(oilhip_prod_gemv_oil4, u8(w), static_cast<uint16_t*>(cb), scale, f32(x), f32(y), M, K, N, s)
                                 : without_gil(oilhip_prod_gemv_oil8, u8(w), static_cast<float*>(cb), scale, f32(x), f32(y), M, K, N, s);
        return result(rc, Py_None, y);
    });
}
// engine_quant_gemm(bits, a, codes, codebook, M, N, K)
PyObject* engine_quant_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 7, [&]() -> PyObject* {
        const long long bits = integer(a[0]);
        const at::Tensor &x = tensor(a[1]), &codes = tensor(a[2]), &cb = tensor(a[3]);
        need(bits >= 0 && bits < 16 && cb.numel() >= (1ll << bits));
        const int64_t M = size(a[4]), N = size(a[5]), K = size(a[6]);
        const at::Tensor y = empty({M, N}, x);
        void* s = stream();
        return result(without_gil(oilhip_engine_quant_gemm, (int)bits, f32(x), u8(codes), f32(cb), f32(y), M, N, K, s), Py_None, y);
    });
}
// kv_append(cache, layer, k, v, values of a token): True
PyObject* kv_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 5, [&]() -> PyObject* {
        auto* c = handle<oilhip_kv>(a[0]);
        const int layer = (int)size(a[1]);
        const at::Tensor &k = tensor(a[2], at::kFloat), &v = tensor(a[3], at::kFloat);
        need(k.dim() == 4 && v.dim() == 4);
        const int64_t seq = k.size(2), token = size(a[4]);
        need(k.numel() == seq * token && v.numel() == k.numel());
        void* s = stream();
        if (const int rc = without_gil(oilhip_kv_append, c, layer, f32(k), f32(v), seq, s)) return raise(rc);
        Py_RETURN_TRUE;
    });
}
// kv_get_range(cache, layer, start, end, max_seq, heads, dim): (k, v) of the tokens of the range that the layer holds
PyObject* kv_get_range(PyObject*, PyObject* const* a, Py_ssize_t n) {
    return ordinary(n, 7, [&]() -> PyObject* {
        auto* c = handle<oilhip_kv>(a[0]);
        const int layer = (int)size(a[1]);
        const int64_t start = size(a[2]), end = std::min(size(a[3]), size(a[4])), heads = size(a[5]), dim = size(a[6]);
        need(end > start);
        int64_t held = 0;
        need(oilhip_kv_held(c, layer, &held) == OILHIP_OK);
        const int64_t len = std::min(end, held) - start;
        need(len > 0);
        const auto options = at::TensorOptions().dtype(at::kFloat).device(at::kCUDA, c10::hip::current_device());
        const at::Tensor k = at::empty({1, heads, len, dim}, options), v = at::empty({1, heads, len, dim}, options);
        int64_t got = 0;
        void* s = stream();
        if (const int rc = without_gil(oilhip_kv_get_range, c, layer, start, start + len, f32(k), f32(v), &got, s)) return raise(rc);
        need(got == len);
        PyObject *pk = THPVariable_Wrap(k), *pv = THPVariable_Wrap(v), *pair = pk && pv ? PyTuple_Pack(2, pk, pv) : nullptr;
        Py_XDECREF(pk);
        Py_XDECREF(pv);
        return pair;
    });
}

PyMethodDef methods[] = {
#define CALL(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
    CALL(gemv), CALL(gemm), CALL(dequant), CALL(embed_rows), CALL(gemv_rmsnorm), CALL(mlp_step), CALL(oil8_gemm), CALL(oil4_gemm), CALL(prod),
    CALL(engine_quant_gemm), CALL(kv_append), CALL(kv_get_range), {nullptr, nullptr, 0, nullptr}
#undef CALL
};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "innova_amd._native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native() { return PyModule_Create(&module_def); }
