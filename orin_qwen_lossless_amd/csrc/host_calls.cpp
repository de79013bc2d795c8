// The dense product's call from Python in native code: mmv(x, w, out_bf16, multi_col, bf16_only, max_tokens).
//
// A small product is bound by the host's call (512 x 2048, one token: the kernel takes 3 us, the call with its checks, result
// and argument block in Python 9.2).  This does the same for the plain case: a two-dimensional tensor of the plain class on the
// current device, all of the weight's buffers there.  Whatever it does not take, wrong arguments among it, it answers with
// None, and the Python layer goes its general way, whose checks and messages hold; nothing is kept from one call for the next.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "bf16n_c.h"

namespace {

typedef int (*mmv_fn)(const bf16n_weight *, const bf16n_mmv_args *, void *, int);
mmv_fn g_mmv = nullptr; // bf16n_mmv of the library that the Python layer loaded
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

PyObject * mmv(PyObject *, PyObject * const * args, Py_ssize_t n) {
    if (n != 6 || !g_mmv) {
        return not_taken();
    }
    const bool out_bf16 = args[2] == Py_True, multi_col = args[3] == Py_True, bf16_only = args[4] == Py_True;
    const long max_tokens = PyLong_AsLong(args[5]);
    if (max_tokens <= 0 || at::impl::torch_function_mode_enabled() || c10::impl::dispatch_mode_enabled()) {
        return not_taken();
    }
    try {
        const at::Tensor * x = plain(args[0]);
        if (!x || x->dim() != 2) {
            return not_taken();
        }
        const int device = c10::hip::current_device();
        const bool x_bf16 = x->scalar_type() == at::kBFloat16;
        if (!x_bf16 && (bf16_only || x->scalar_type() != at::kFloat)) {
            return not_taken();
        }
        const ref pl(args[1], s_plane), au(args[1], s_aux), me(args[1], s_meta);
        if (!pl.o || !au.o || !me.o) {
            return not_taken();
        }
        const at::Tensor * plane = plain(pl.o), * aux = plain(au.o);
        int64_t fmt, K, rows, R, cm, frag, w64, off[4];
        bool ok = plane && aux && x->get_device() == device && plane->get_device() == device && aux->get_device() == device && number(me.o, s_format, fmt) && number(me.o, s_K, K) && number(me.o, s_rows, rows) && number(me.o, s_R, R) &&
                  number(me.o, s_cm, cm) && number(me.o, s_frag, frag) && number(me.o, s_w64, w64);
        for (int i = 0; ok && i < 4; i++) {
            ok = number(me.o, s_off[i], off[i]) && off[i] < aux->numel();
        }
        if (!ok || plane->scalar_type() != at::kByte || aux->scalar_type() != at::kByte || !plane->is_contiguous() || !aux->is_contiguous() ||
            rows <= 0 || K <= 0 || plane->numel() != rows * K || fmt > INT32_MAX || R > INT32_MAX) {
            return not_taken();
        }
        const int64_t T = x->size(0), esz = x_bf16 ? 2 : 4, osz = out_bf16 ? 2 : 4;
        char * xp = (char *) x->data_ptr(), * pp = (char *) plane->data_ptr(), * ap = (char *) aux->data_ptr();
        if (T <= 0 || T > max_tokens || x->size(1) != K || x->stride(1) != 1 || x->stride(0) * esz % 16 != 0 ||
            (((uintptr_t) xp | (uintptr_t) pp | (uintptr_t) ap) & 15) != 0) {
            return not_taken();
        }
        at::Tensor y = at::empty({T, rows}, x->options().dtype(out_bf16 ? at::kBFloat16 : at::kFloat).requires_grad(false));
        bf16n_weight w = {};
        w.plane = (decltype(w.plane)) pp;
        w.aux = (decltype(w.aux)) ap;
        w.format = (int32_t) fmt;
        w.R = (int32_t) R;
        w.K = K;
        w.rows = rows;
        w.flags = (cm ? 1u : 0u) | (frag ? 2u : 0u) | (w64 ? 4u : 0u);
        w.off_a = (uint64_t) off[0];
        w.off_b = (uint64_t) off[1];
        w.off_c = (uint64_t) off[2];
        w.off_d = (uint64_t) off[3];
        bf16n_mmv_args a = {};
        a.x = (decltype(a.x)) xp;
        a.y = (decltype(a.y)) y.data_ptr();
        a.x_tok = x->stride(0) * esz;
        a.y_tok = rows * osz;
        a.rows_per_matrix = rows;
        a.nrows = rows;
        a.ncols = (int32_t) T;
        a.n_used = 1;
        a.x_per_slot = 1;
        a.x_bf16 = x_bf16;
        a.y_bf16 = out_bf16;
        void * stream = (void *) c10::hip::getCurrentHIPStream((c10::DeviceIndex) device).stream();
        int status;
        Py_BEGIN_ALLOW_THREADS // (the queue may be full)
        status = g_mmv(&w, &a, stream, multi_col);
        Py_END_ALLOW_THREADS
        return status == 0 ? THPVariable_Wrap(y) : PyLong_FromLong(status);
    } catch (const std::exception &) { // (out of memory: the general way meets it again and says so)
        return not_taken();
    }
}

PyObject * bind(PyObject *, PyObject * addr) {
    g_mmv = (mmv_fn) PyLong_AsVoidPtr(addr);
    if (PyErr_Occurred()) {
        return nullptr;
    }
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"mmv", (PyCFunction) (void (*)(void)) mmv, METH_FASTCALL, "the product, a status of the C ABI, or None: not taken"},
    {"bind", bind, METH_O, "the address of bf16n_mmv"},
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
    return PyModule_Create(&g_module);
}
