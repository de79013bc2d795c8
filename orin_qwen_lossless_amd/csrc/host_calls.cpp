// The dense products' calls from Python in native code: mmv(x, w, out_bf16, multi_col) and linear(x, w, gemv_tokens, chunk_bytes).
//
// A small product is bound by the host's call (512 x 2048, one token: the kernel takes 3 us, the call with its checks, result
// and argument block in Python 9.2).  This does the same for the plain case: a two-dimensional tensor of the plain class on the
// current device, all of the weight's buffers there.  Whatever it does not take, wrong arguments among it, it answers with
// None, and the Python layer goes its general way, whose checks and messages hold; nothing is kept from one call for the next.
#include <Python.h>

#include <algorithm>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <pybind11/gil.h>
#include <torch/csrc/autograd/python_variable.h>

#include "bf16n_c.h"

namespace {

typedef int (*mmv_fn)(const bf16n_weight *, const bf16n_mmv_args *, void *, int);
typedef int (*max_tokens_fn)(const bf16n_weight *, int *);
typedef int (*dequant_fn)(const bf16n_weight *, int64_t, int64_t, uint16_t *, void *);
mmv_fn g_mmv = nullptr; // of the library that the Python layer loaded
max_tokens_fn g_max_tokens = nullptr;
dequant_fn g_dequant = nullptr;
PyObject * s_plane, * s_aux, * s_meta, * s_format, * s_K, * s_rows, * s_R, * s_cm, * s_frag, * s_w64, * s_off[4];

// a tensor of the plain class with memory of its own on a device (no tracer, batch or gradient wrapper)
const at::Tensor * plain(PyObject * o) {
    if (!THPVariable_CheckExact(o)) {
        return nullptr;
    }
    const at::Tensor & t = THPVariable_Unpack(o);
    constexpr c10::DispatchKeySet other({c10::DispatchKey::Python, c10::DispatchKey::PythonTLSSnapshot, c10::DispatchKey::FuncTorchBatched,
                                         c10::DispatchKey::FuncTorchGradWrapper, c10::DispatchKey::Functionalize, c10::DispatchKey::Conjugate,
                                         c10::DispatchKey::Negative, c10::DispatchKey::ZeroTensor});
    if (!t.is_cuda() || t.layout() != c10::kStrided || t.key_set().has_any(other) || !t.has_storage()) {
        return nullptr;
    }
    return &t;
}

struct ref { // an owned attribute
    PyObject * o;
    ref(PyObject * of, PyObject * name) : o(PyObject_GetAttr(of, name)) {}
    ~ref() { Py_XDECREF(o); }
};
bool number(PyObject * of, PyObject * name, int64_t & out) {
    const ref a(of, name);
    if (!a.o || !PyLong_Check(a.o)) { // (bool is a number too)
        return false;
    }
    out = PyLong_AsLongLong(a.o);
    return out >= 0; // -1: an error too
}

PyObject * not_taken() {
    PyErr_Clear();
    Py_RETURN_NONE;
}

// x [tokens, K] and a weight on the current device, checked as the Python layer checks them
struct operands {
    const at::Tensor * x;
    bf16n_weight w;
    int device;
    bool x_bf16;
    bool get(PyObject * px, PyObject * pw) {
        if (!g_mmv || at::impl::torch_function_mode_enabled() || c10::impl::dispatch_mode_enabled()) {
            return false;
        }
        x = plain(px);
        if (!x || x->dim() != 2) {
            return false;
        }
        device = c10::hip::current_device();
        x_bf16 = x->scalar_type() == at::kBFloat16;
        const ref pl(pw, s_plane), au(pw, s_aux), me(pw, s_meta);
        if (!pl.o || !au.o || !me.o) {
            return false;
        }
        const at::Tensor * plane = plain(pl.o), * aux = plain(au.o);
        int64_t fmt, K, rows, R, cm, frag, w64, off[4];
        bool ok = plane && aux && x->get_device() == device && plane->get_device() == device && aux->get_device() == device &&
                  number(me.o, s_format, fmt) && number(me.o, s_K, K) && number(me.o, s_rows, rows) && number(me.o, s_R, R) &&
                  number(me.o, s_cm, cm) && number(me.o, s_frag, frag) && number(me.o, s_w64, w64);
        for (int i = 0; ok && i < 4; i++) {
            ok = number(me.o, s_off[i], off[i]) && off[i] < aux->numel();
        }
        if (!ok || plane->scalar_type() != at::kByte || aux->scalar_type() != at::kByte || !plane->is_contiguous() || !aux->is_contiguous() ||
            rows <= 0 || K <= 0 || plane->numel() != rows * K || fmt > INT32_MAX || R > INT32_MAX) {
            return false;
        }
        w = {};
        w.plane = (decltype(w.plane)) plane->data_ptr();
        w.aux = (decltype(w.aux)) aux->data_ptr();
        w.format = (int32_t) fmt;
        w.R = (int32_t) R;
        w.K = K;
        w.rows = rows;
        w.flags = (cm ? 1u : 0u) | (frag ? 2u : 0u) | (w64 ? 4u : 0u);
        w.off_a = (uint64_t) off[0];
        w.off_b = (uint64_t) off[1];
        w.off_c = (uint64_t) off[2];
        w.off_d = (uint64_t) off[3];
        return x->size(0) > 0 && x->size(0) <= 65535 && x->size(1) == K && x->stride(1) == 1 && x->stride(0) * (x_bf16 ? 2 : 4) % 16 == 0 &&
               (((uintptr_t) x->data_ptr() | (uintptr_t) w.plane | (uintptr_t) w.aux) & 15) == 0;
    }
    void * stream() const { return (void *) c10::hip::getCurrentHIPStream((c10::DeviceIndex) device).stream(); }
    PyObject * product(bool out_bf16, bool multi_col) const {
        at::Tensor y = at::empty({x->size(0), w.rows}, x->options().dtype(out_bf16 ? at::kBFloat16 : at::kFloat).requires_grad(false));
        bf16n_mmv_args a = {};
        a.x = (decltype(a.x)) x->data_ptr();
        a.y = (decltype(a.y)) y.data_ptr();
        a.x_tok = x->stride(0) * (x_bf16 ? 2 : 4);
        a.y_tok = w.rows * (out_bf16 ? 2 : 4);
        a.rows_per_matrix = w.rows;
        a.nrows = w.rows;
        a.ncols = (int32_t) x->size(0);
        a.n_used = 1;
        a.x_per_slot = 1;
        a.x_bf16 = x_bf16;
        a.y_bf16 = out_bf16;
        int status;
        {
            pybind11::gil_scoped_release free; // (the queue may be full)
            status = g_mmv(&w, &a, stream(), multi_col);
        }
        return status == 0 ? THPVariable_Wrap(y) : PyLong_FromLong(status);
    }
};

PyObject * mmv(PyObject *, PyObject * const * args, Py_ssize_t n) {
    try {
        operands o;
        if (n != 4 || !o.get(args[0], args[1]) || (!o.x_bf16 && o.x->scalar_type() != at::kFloat)) {
            return not_taken();
        }
        return o.product(args[2] == Py_True, args[3] == Py_True);
    } catch (const std::exception &) { // (out of memory: the general way meets it again and says so)
        return not_taken();
    }
}

// the GEMV up to gemv_tokens or bf16n_gemv_max_tokens tokens, beyond it the whole matrix decoded, if it is one piece of
// chunk_bytes, and torch's product
PyObject * linear(PyObject *, PyObject * const * args, Py_ssize_t n) {
    try {
        operands o;
        if (n != 4 || !o.get(args[0], args[1]) || !o.x_bf16) {
            return not_taken();
        }
        const int64_t gemv_tokens = PyLong_AsLongLong(args[2]), chunk_bytes = PyLong_AsLongLong(args[3]), T = o.x->size(0);
        if (gemv_tokens < 0 || chunk_bytes < 0) {
            return not_taken();
        }
        int most = 0;
        if (T > gemv_tokens && g_max_tokens(&o.w, &most) != 0) {
            return not_taken();
        }
        if (T <= gemv_tokens || T <= most) {
            return o.product(true, true);
        }
        const int64_t unit = o.w.format == 1 ? 1 : o.w.R; // (the 4-bit code has no units)
        if (unit <= 0 || std::max(chunk_bytes / (o.w.K * 2) / unit * unit, unit) < o.w.rows) {
            return not_taken();
        }
        at::Tensor d = at::empty({o.w.rows, o.w.K}, o.x->options().requires_grad(false)), y;
        int status;
        {
            pybind11::gil_scoped_release free;
            status = g_dequant(&o.w, 0, o.w.rows, (uint16_t *) d.data_ptr(), o.stream());
            if (status == 0) {
                y = at::linear(*o.x, d);
            }
        }
        return status == 0 ? THPVariable_Wrap(y) : PyLong_FromLong(status);
    } catch (const std::exception &) {
        return not_taken();
    }
}

PyObject * bind(PyObject *, PyObject * const * args, Py_ssize_t n) {
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "bind: three addresses");
        return nullptr;
    }
    g_mmv = (mmv_fn) PyLong_AsVoidPtr(args[0]);
    g_max_tokens = (max_tokens_fn) PyLong_AsVoidPtr(args[1]);
    g_dequant = (dequant_fn) PyLong_AsVoidPtr(args[2]);
    if (PyErr_Occurred()) {
        g_mmv = nullptr;
        return nullptr;
    }
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"mmv", (PyCFunction) (void (*)(void)) mmv, METH_FASTCALL, "the product, a status of the C ABI, or None: not taken"},
    {"linear", (PyCFunction) (void (*)(void)) linear, METH_FASTCALL, "the same for BF16 in and out and any number of tokens"},
    {"bind", (PyCFunction) (void (*)(void)) bind, METH_FASTCALL, "the addresses of bf16n_mmv, bf16n_gemv_max_tokens, bf16n_dequant"},
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject ** const names[] = {&s_plane, &s_aux, &s_meta, &s_format, &s_K, &s_rows, &s_R, &s_cm, &s_frag, &s_w64, &s_off[0], &s_off[1], &s_off[2], &s_off[3]};
    const char * const text[] = {"plane", "aux", "meta", "format", "K", "rows", "R", "chunk_major", "frag_order", "wave64", "off_a", "off_b", "off_c", "off_d"};
    for (size_t i = 0; i < sizeof(text) / sizeof(text[0]); i++) {
        if (!(*names[i] = PyUnicode_InternFromString(text[i]))) {
            return nullptr;
        }
    }
    // the release of torch whose internals are inlined above; the Python layer uses the module with no other
    PyObject * m = PyModule_Create(&g_module);
    if (m && PyModule_AddStringConstant(m, "built_for", BUILT_FOR) != 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
