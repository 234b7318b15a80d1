// The host side of the operator calls that are a few microseconds on the device, as a Python module: what the wrappers of
// ../__init__.py do for tensors of the ordinary kind -- outputs allocated, pointers, sizes and the current stream handed to the
// C ABI -- without the interpreter in between.  A 5632 x 2048 GEMV takes 4 - 5 us on the device; the call took 6.3 us through
// ctypes (of which the launch itself 2), dynamic_quantize_linear and quantized_matmul behind it 13.
//
// Every function returns None for anything it does not take (other classes than Tensor, other devices, types, orders, sizes that
// do not fit together): the caller then goes the long way, which has the checks and raises what it always raised.  An error code
// of the C ABI becomes the exception that bind() was given.
#include <ATen/ATen.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include "../../include/mynn_hip.h"

namespace {

decltype(&mynn_last_error) g_last_error;
decltype(&mynn_dequant_matmul) g_dequant_matmul;
decltype(&mynn_quantized_matmul) g_quantized_matmul;
decltype(&mynn_dynamic_quantize_linear) g_dynamic_quantize_linear;
decltype(&mynn_attention) g_attention;
PyObject *g_error;

int code_of(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return MYNN_F32;
        case at::kBFloat16: return MYNN_BF16;
        case at::kHalf: return MYNN_F16;
        default: return -1;
    }
}
// a plain tensor on the GPU, its elements in order (THPVariable_CheckExact: no subclass, which may mean something else by it)
const at::Tensor *plain(PyObject *o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor &t = THPVariable_Unpack(o);
    return t.defined() && t.has_storage() && t.is_cuda() && t.layout() == at::kStrided && t.is_contiguous() ? &t : nullptr;
}
void *data(const at::Tensor &t) { return t.data_ptr(); }
mynn_stream current_stream() { return (mynn_stream)c10::hip::getCurrentHIPStream().stream(); }
at::Tensor make(at::IntArrayRef sizes, const at::Tensor &like, at::ScalarType type) { return at::empty(sizes, like.options().dtype(type)); }

PyObject *none() { Py_RETURN_NONE; }
template <typename F> int without_gil(F &&f) {
    PyThreadState *state = PyEval_SaveThread();
    const int rc = f();
    PyEval_RestoreThread(state);
    return rc;
}
PyObject *failed(int rc) {
    PyErr_Format(g_error, "mynn error %d: %s", rc, g_last_error());
    return nullptr;
}
// f() with what torch throws (a tensor without memory of its own, no memory left) answered by None
template <typename F> PyObject *guarded(F &&f) {
    try {
        at::AutoDispatchBelowADInplaceOrView guard;
        return f();
    } catch (const std::exception &) {
        return none();
    }
}

// (act [.., K], wq [N, K], scale [N]) -> [.., N]
PyObject *dequant_matmul(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 3) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *act = plain(args[0]), *wq = plain(args[1]), *scale = plain(args[2]);
        if (!act || !wq || !scale || wq->dim() != 2 || wq->scalar_type() != at::kChar || act->dim() < 1) return none();
        const int64_t N = wq->size(0), K = wq->size(1);
        const int ac = code_of(act->scalar_type()), sc = code_of(scale->scalar_type());
        if (ac < 0 || sc < 0 || K < 1 || act->size(-1) != K) return none();
        const int64_t M = act->numel() / K;
        c10::SmallVector<int64_t, 4> sizes(act->sizes().begin(), act->sizes().end());
        sizes.back() = N;
        const at::Tensor out = make(sizes, *wq, scale->scalar_type());
        void *o = data(out), *a = data(*act), *w = data(*wq), *s = data(*scale);
        const mynn_stream st = current_stream();
        const int rc = without_gil([&] { return g_dequant_matmul(o, a, (const int8_t *)w, s, (int)M, (int)N, (int)K, ac, sc, st); });
        return rc ? failed(rc) : THPVariable_Wrap(out);
    });
}

// (lhs [M, K], lhs_scale, rhs [N, K], rhs_scale) -> [M, N]
PyObject *quantized_matmul(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 4) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *lhs = plain(args[0]), *ls = plain(args[1]), *rhs = plain(args[2]), *rs = plain(args[3]);
        if (!lhs || !ls || !rhs || !rs || lhs->dim() != 2 || rhs->dim() != 2 || lhs->scalar_type() != at::kChar || rhs->scalar_type() != at::kChar) return none();
        const int64_t M = lhs->size(0), K = lhs->size(1), N = rhs->size(0);
        const int code = code_of(rs->scalar_type());
        if (code < 0 || rhs->size(1) != K) return none();
        const at::Tensor out = make({M, N}, *lhs, rs->scalar_type());
        void *o = data(out), *l = data(*lhs), *lsp = data(*ls), *r = data(*rhs), *rsp = data(*rs);
        const mynn_stream st = current_stream();
        const int rc = without_gil([&] {
            return g_quantized_matmul(o, nullptr, (const int8_t *)l, lsp, (const int8_t *)r, rsp, (int)M, (int)N, (int)K, code, st);
        });
        return rc ? failed(rc) : THPVariable_Wrap(out);
    });
}

// (x [rows, ..]) -> (int8 codes like x, scales [rows], zero points [rows]), the symmetric form
PyObject *dynamic_quantize_linear(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 1) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *x = plain(args[0]);
        if (!x || x->dim() < 1 || x->size(0) < 1) return none();
        const int code = code_of(x->scalar_type());
        if (code < 0) return none();
        const int64_t rows = x->size(0), inner = x->numel() / rows;
        const at::Tensor y = make(x->sizes(), *x, at::kChar), s = make({rows}, *x, x->scalar_type()), zp = make({rows}, *x, at::kChar);
        void *yp = data(y), *sp = data(s), *zpp = data(zp), *xp = data(*x);
        const mynn_stream st = current_stream();
        const int rc = without_gil([&] { return g_dynamic_quantize_linear(yp, sp, zpp, xp, (int)rows, (int)inner, code, 1, st); });
        if (rc) return failed(rc);
        PyObject *r = PyTuple_New(3);
        if (!r) return nullptr;
        PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(y));
        PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(s));
        PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(zp));
        return r;
    });
}

// (q [B, Hq, Sq, D], k, v [B, Hkv, rows, D], scale, is_causal, active or None, q_pos_offset or None, k_scale or None, v_scale or None)
PyObject *attention(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 9) return none();
    return guarded([&]() -> PyObject * {
        const at::Tensor *q = plain(args[0]), *k = plain(args[1]), *v = plain(args[2]);
        if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || !PyFloat_CheckExact(args[3]) || !PyBool_Check(args[4])) return none();
        const int code = code_of(q->scalar_type());
        if (code < 0) return none();
        const int64_t B = q->size(0), Hq = q->size(1), Sq = q->size(2), D = q->size(3), Hkv = k->size(1), rows = k->size(2);
        int64_t active = rows, offset = 0;
        if (args[5] != Py_None) {
            if (!PyLong_CheckExact(args[5])) return none();
            active = PyLong_AsLongLong(args[5]);
        }
        if (args[6] != Py_None) {
            if (!PyLong_CheckExact(args[6])) return none();
            offset = PyLong_AsLongLong(args[6]);
        } else offset = Sq == rows ? 0 : active - Sq;
        if (PyErr_Occurred() || active != (int)active || offset != (int)offset) {
            PyErr_Clear();
            return none();
        }
        const at::Tensor *ks = nullptr, *vs = nullptr;
        if ((args[7] != Py_None && !(ks = plain(args[7]))) || (args[8] != Py_None && !(vs = plain(args[8])))) return none();
        const at::Tensor out = make(q->sizes(), *q, q->scalar_type());
        void *o = data(out), *qp = data(*q), *kp = data(*k), *vp = data(*v), *ksp = ks ? data(*ks) : nullptr, *vsp = vs ? data(*vs) : nullptr;
        const float scale = (float)PyFloat_AS_DOUBLE(args[3]);
        const int causal = args[4] == Py_True, i8 = k->scalar_type() == at::kChar;
        const mynn_stream st = current_stream();
        const int rc = without_gil([&] {
            return g_attention(o, qp, kp, vp, ksp, vsp, scale, causal, (int)B, (int)Sq, (int)active, nullptr, (int)rows, (int)offset, (int)Hq, (int)Hkv, (int)D,
                               code, i8, st);
        });
        return rc ? failed(rc) : THPVariable_Wrap(out);
    });
}

// (exception class, addresses of mynn_last_error and of the four operators)
PyObject *bind(PyObject *, PyObject *const *args, Py_ssize_t n) {
    if (n != 6) {
        PyErr_SetString(PyExc_TypeError, "bind: six arguments");
        return nullptr;
    }
    void *p[5];
    for (int i = 0; i < 5; i++) {
        p[i] = PyLong_AsVoidPtr(args[i + 1]);
        if (!p[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "bind: null address");
            return nullptr;
        }
    }
    Py_INCREF(args[0]);
    Py_XSETREF(g_error, args[0]);
    g_last_error = (decltype(g_last_error))p[0];
    g_dequant_matmul = (decltype(g_dequant_matmul))p[1];
    g_quantized_matmul = (decltype(g_quantized_matmul))p[2];
    g_dynamic_quantize_linear = (decltype(g_dynamic_quantize_linear))p[3];
    g_attention = (decltype(g_attention))p[4];
    Py_RETURN_NONE;
}

#define MYNN_METHOD(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {MYNN_METHOD(bind), MYNN_METHOD(dequant_matmul), MYNN_METHOD(quantized_matmul), MYNN_METHOD(dynamic_quantize_linear), MYNN_METHOD(attention),
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host_ops", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_ops(void) {
    PyObject *m = PyModule_Create(&g_module);
    // (torch's classes are used as its headers lay them out: a module built against another one is not to be called)
    if (m && PyModule_AddStringConstant(m, "torch_version", TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
