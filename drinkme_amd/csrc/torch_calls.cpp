// The per-call path of the torch launchers (drinkme_amd/radix_ops.py) as a
// CPython extension: one call checks the activation, allocates the output
// with torch and launches through the C ABI. What bounds a decode step's
// small calls is the host: through ctypes and Python's own checks a call of
// one Linear took 10.1 us on the host for a 5.5 us kernel (k_proj of 1024 x
// 4096, M = 1), a grouped attention block 33.6 us for 20.6 us of kernels.
//
// Every function takes the plain case alone (dense contiguous GPU tensors of
// the types, shapes and device the launcher was built for, and a descriptor
// whose buffers are still its runtime dict's) and returns None for anything
// else, having launched nothing: the caller's general path then copies,
// rebuilds its descriptor or raises.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <string>

#include "dmx_radix.h"

namespace {

constexpr int kMaxRows = 8, kMaxGroup = 16;

// A dense strided tensor of the GPU that no torch wrapper (functorch, a
// dispatch subclass, a lazy negation) stands in front of.
bool plain(const at::Tensor& t) {
    using K = c10::DispatchKey;
    return t.defined() && t.is_cuda() && t.layout() == at::kStrided && t.has_storage() &&
           !t.key_set().has_any(c10::DispatchKeySet({K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Functionalize,
                                                     K::Python, K::Negative, K::Conjugate, K::ZeroTensor})) &&
           t.is_contiguous();
}

// The tensor of an exact torch.Tensor or Parameter, null for anything else.
const at::Tensor* exact(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

int code(at::ScalarType t) { return t == at::kBFloat16 ? DMX_BF16 : t == at::kFloat ? DMX_F32 : -1; }

// Rows of x [..., C], 0 where x is not a plain [..., C] of 1..8 rows on
// device `index` in a type that the kernels take.
uint32_t rows_of(const at::Tensor* x, int64_t C, int64_t index) {
    if (!x || !plain(*x) || x->get_device() != index || code(x->scalar_type()) < 0) return 0;
    if (x->dim() == 0 || C <= 0 || x->size(-1) != C) return 0;
    const int64_t m = x->numel() / C;
    return m >= 1 && m <= kMaxRows ? (uint32_t)m : 0;
}

// Whether `o` (None or a bias of R elements) is taken; its address and type.
bool bias_of(PyObject* o, int64_t R, int64_t index, const void*& at, int& dtype) {
    at = nullptr;
    dtype = 0;
    if (o == Py_None) return true;
    const at::Tensor* b = exact(o);
    if (!b || !plain(*b) || b->get_device() != index || b->numel() != R || code(b->scalar_type()) < 0) return false;
    at = b->const_data_ptr();
    dtype = code(b->scalar_type());
    return true;
}

// Whether the descriptor's buffers are those in the runtime dict p.
PyObject* g_keys[4];  // "rx_data", "rx_offsets", "rx_palette", "rx_schedule"
bool current(const dmx_radix_tensor* t, PyObject* p) {
    const void* held[4] = {t->data, t->offsets, t->palette, t->schedule};
    if (!PyDict_Check(p)) return false;
    for (int i = 0; i < 4; ++i) {
        PyObject* o = PyDict_GetItem(p, g_keys[i]);  // borrowed
        const at::Tensor* b = o && o != Py_None ? exact(o) : nullptr;
        if (!b ? i != 3 || (o && o != Py_None) : !plain(*b)) return false;
        const void* at = b && b->numel() ? b->const_data_ptr() : nullptr;
        if (at != held[i]) return false;
    }
    return true;
}

at::ScalarType dtype_of(PyObject* o) {
    return THPDtype_Check(o) ? reinterpret_cast<THPDtype*>(o)->scalar_type : at::ScalarType::Undefined;
}

at::Tensor output(const at::Tensor& x, int64_t R, at::ScalarType dtype) {
    c10::SmallVector<int64_t, 6> sizes(x.sizes().begin(), x.sizes().end());
    sizes.back() = R;
    return at::empty(sizes, at::TensorOptions().device(x.device()).dtype(dtype));
}

PyObject* launch_failed(const char* what, const char* err) {
    PyErr_SetString(PyExc_RuntimeError, (std::string(what) + ": " + err).c_str());
    return nullptr;
}

bool modes_off() { return !at::impl::torch_function_mode_enabled(); }

// rows(descriptor address, p, x, bias, out dtype, R, C, device index, stream)
PyObject* rows(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 9) return launch_failed("rows", "nine arguments");
    const auto* t = static_cast<const dmx_radix_tensor*>(PyLong_AsVoidPtr(a[0]));
    const at::Tensor* x = exact(a[2]);
    const at::ScalarType od = dtype_of(a[4]);
    const int64_t R = PyLong_AsLongLong(a[5]), C = PyLong_AsLongLong(a[6]), index = PyLong_AsLongLong(a[7]);
    void* stream = PyLong_AsVoidPtr(a[8]);
    if (PyErr_Occurred()) return nullptr;
    const uint32_t m = rows_of(x, C, index);
    const void* bias;
    int bd;
    if (!t || !m || code(od) < 0 || !modes_off() || !bias_of(a[3], R, index, bias, bd) || !current(t, a[1]))
        Py_RETURN_NONE;
    at::Tensor out;
    char err[512];
    int st;
    {
        pybind11::gil_scoped_release no_gil;
        out = output(*x, R, od);
        st = dmx_radix_gemv(t, x->const_data_ptr(), code(x->scalar_type()), m, bias, bd, out.mutable_data_ptr(), code(od),
                            stream, err, sizeof err);
    }
    return st ? launch_failed("dmx_radix_gemv", err) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// group(descriptor table address, [p, ...], x, bias table address, bias dtype
// code, out dtype, (R, ...), C, device index, stream)
PyObject* group(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 10 || !PyList_Check(a[1]) || !PyTuple_Check(a[6])) return launch_failed("group", "ten arguments");
    const auto* const* ts = static_cast<const dmx_radix_tensor* const*>(PyLong_AsVoidPtr(a[0]));
    const Py_ssize_t k = PyTuple_GET_SIZE(a[6]);
    const at::Tensor* x = exact(a[2]);
    const void* const* bias = static_cast<const void* const*>(PyLong_AsVoidPtr(a[3]));
    const long bd = PyLong_AsLong(a[4]);
    const at::ScalarType od = dtype_of(a[5]);
    const int64_t C = PyLong_AsLongLong(a[7]), index = PyLong_AsLongLong(a[8]);
    void* stream = PyLong_AsVoidPtr(a[9]);
    if (PyErr_Occurred()) return nullptr;
    const uint32_t m = rows_of(x, C, index);
    if (!ts || !m || code(od) < 0 || !modes_off() || k < 1 || k > kMaxGroup || PyList_GET_SIZE(a[1]) != k) Py_RETURN_NONE;
    int64_t R[kMaxGroup];
    for (Py_ssize_t i = 0; i < k; ++i) {
        if (!current(ts[i], PyList_GET_ITEM(a[1], i))) Py_RETURN_NONE;
        R[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(a[6], i));
    }
    if (PyErr_Occurred()) return nullptr;
    at::Tensor outs[kMaxGroup];
    void* at_out[kMaxGroup];
    char err[512];
    int st;
    {
        pybind11::gil_scoped_release no_gil;
        for (Py_ssize_t i = 0; i < k; ++i) {
            outs[i] = output(*x, R[i], od);
            at_out[i] = outs[i].mutable_data_ptr();
        }
        st = dmx_radix_gemv_group(ts, (uint32_t)k, x->const_data_ptr(), code(x->scalar_type()), m, bias, (int)bd, at_out,
                                  code(od), stream, err, sizeof err);
    }
    if (st) return launch_failed("dmx_radix_gemv_group", err);
    PyObject* list = PyList_New(k);
    if (!list) return nullptr;
    for (Py_ssize_t i = 0; i < k; ++i) {
        PyObject* o = THPVariable_Wrap(std::move(outs[i]));
        if (!o) {
            Py_DECREF(list);
            return nullptr;
        }
        PyList_SET_ITEM(list, i, o);
    }
    return list;
    END_HANDLE_TH_ERRORS
}

// narrow(w, x, bias, stream): x [..., C] against the raw bf16 w [R, C], in x's dtype
PyObject* narrow(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 4) return launch_failed("narrow", "four arguments");
    const at::Tensor *w = exact(a[0]), *x = exact(a[1]);
    void* stream = PyLong_AsVoidPtr(a[3]);
    if (PyErr_Occurred()) return nullptr;
    if (!w || !plain(*w) || w->dim() != 2 || w->scalar_type() != at::kBFloat16 || !modes_off()) Py_RETURN_NONE;
    const int64_t R = w->size(0), C = w->size(1), index = w->get_device();
    const uint32_t m = rows_of(x, C, index);
    const void* bias;
    int bd;
    if (!m || R < 1 || R >= (1ll << 31) || C >= (1ll << 32) || !bias_of(a[2], R, index, bias, bd)) Py_RETURN_NONE;
    at::Tensor out;
    char err[512];
    int st;
    {
        pybind11::gil_scoped_release no_gil;
        const int xd = code(x->scalar_type());
        out = output(*x, R, x->scalar_type());
        st = dmx_gemv_narrow(static_cast<const uint16_t*>(w->const_data_ptr()), (uint32_t)R, (uint32_t)C,
                             x->const_data_ptr(), xd, m, bias, bd, out.mutable_data_ptr(), xd, stream, err, sizeof err);
    }
    return st ? launch_failed("dmx_gemv_narrow", err) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyCFunction fast() {
    return reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(F));
}
PyMethodDef g_methods[] = {{"rows", fast<rows>(), METH_FASTCALL, nullptr},
                           {"group", fast<group>(), METH_FASTCALL, nullptr},
                           {"narrow", fast<narrow>(), METH_FASTCALL, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "dmx_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_dmx_calls(void) {
    const char* names[4] = {"rx_data", "rx_offsets", "rx_palette", "rx_schedule"};
    for (int i = 0; i < 4; ++i)
        if (!(g_keys[i] = PyUnicode_InternFromString(names[i]))) return nullptr;
    PyObject* m = PyModule_Create(&g_module);
    // (the torch whose headers this was compiled with: the loader compares)
    if (m && PyModule_AddStringConstant(m, "torch_version", DMX_TORCH_VERSION) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
