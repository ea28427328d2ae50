// The operators of rocmforge_amd/ops.py from the argument checks to the library call, in one native call each.
//
// A small decode call is over on the GPU in 3 us; what bounds it is the host: the Python checks, torch.empty and ctypes around the
// launch took 3.7 us of 6.7 (4864 x 896 Q4_0; 4.3 this way, 2.7 of it the runtime's launch; the MLP block of one vector 12.4 ->
// 8.2, three arranged projections 26 -> 19).  Every function here handles the calls that need nothing said about them -
// plain tensors of the right type, shape, device and layout - and returns None for all others, which then run through the Python
// text (its errors, its order of checks).  A status other than RFQ_OK is raised by the Python `check`.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/ops/empty.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "rfq.h"

namespace {

PyObject *g_check = nullptr;                                     // rocmforge_amd._lib.check

struct NotHere {};                                               // this call is for the Python text
struct Raised {};                                                // a Python error is set

// A plain tensor (no subclass, nobody listening to torch functions).
const at::Tensor &tensor(PyObject *o)
{
    if (!THPVariable_CheckExact(o)) throw NotHere{};
    return THPVariable_Unpack(o);
}
const at::Tensor &device_tensor(PyObject *o, at::ScalarType type)
{
    const at::Tensor &t = tensor(o);
    if (!t.is_cuda() || t.scalar_type() != type || !t.is_contiguous()) throw NotHere{};
    return t;
}
int whole(PyObject *o)
{
    if (!PyLong_CheckExact(o)) throw NotHere{};
    int over = 0;
    const long v = PyLong_AsLongAndOverflow(o, &over);
    if (over != 0 || v < 0 || v > 0x7fffffffL) throw NotHere{};
    return (int)v;
}
float real(PyObject *o)
{
    if (!PyFloat_CheckExact(o)) throw NotHere{};
    return (float)PyFloat_AS_DOUBLE(o);
}
int rows_of(const at::Tensor &x, int k)
{
    if (x.dim() < 1 || x.dim() > 2 || x.size(-1) != k) throw NotHere{};
    const int64_t m = x.dim() == 1 ? 1 : x.size(0);
    if (m > 0x7fffffff) throw NotHere{};
    return (int)m;
}
// The caller's buffer, or a new one on x's device.
at::Tensor result(PyObject *out, at::IntArrayRef shape, at::ScalarType type, const at::Tensor &x)
{
    if (out == Py_None) return at::empty(shape, x.options().dtype(type).requires_grad(false));
    const at::Tensor &t = device_tensor(out, type);
    int64_t n = 1;
    for (int64_t d : shape) n *= d;
    if (t.device() != x.device() || t.numel() != n) throw NotHere{};
    return t;
}
void *stream() { return (void *)c10::hip::getCurrentHIPStream().stream(); }

PyObject *finished(int rc, const at::Tensor &y)
{
    if (rc != RFQ_OK) {
        PyObject *r = PyObject_CallFunction(g_check, "i", rc);
        Py_XDECREF(r);
        if (r == nullptr) throw Raised{};
    }
    return THPVariable_Wrap(y);
}

// The library call without the interpreter's lock.
template <typename F> int unlocked(F &&f)
{
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

// Anything that C++ throws (no storage behind a wrapper, no memory left) is said again by the Python text.
template <typename F> PyObject *guarded(Py_ssize_t n, Py_ssize_t want, F &&f)
{
    if (n != want) {
        PyErr_Format(PyExc_TypeError, "%zd arguments, expected %zd", n, want);
        return nullptr;
    }
    if (at::impl::torch_function_mode_enabled() || c10::impl::TorchDispatchModeTLS::any_modes_set()) Py_RETURN_NONE;
    try {
        return f();
    } catch (const Raised &) {
        return nullptr;
    } catch (...) {
        if (PyErr_Occurred()) PyErr_Clear();
        Py_RETURN_NONE;
    }
}

// gemv(fmt, w, x, n, k, out)
PyObject *gemv(PyObject *, PyObject *const *a, Py_ssize_t na)
{
    return guarded(na, 6, [&]() -> PyObject * {
        const int fmt = whole(a[0]), n = whole(a[3]), k = whole(a[4]);
        const at::Tensor &w = device_tensor(a[1], at::kByte), &x = device_tensor(a[2], at::kFloat);
        const int m = rows_of(x, k);
        at::Tensor y = result(a[5], {m, n}, at::kFloat, x);
        const void *wp = w.data_ptr();
        const float *xp = (const float *)x.data_ptr();
        float *yp = (float *)y.data_ptr();
        const size_t bytes = (size_t)w.numel();
        void *s = stream();
        const int rc = unlocked([&] { return rfq_gemv(fmt, wp, bytes, xp, yp, m, n, k, s); });
        return finished(rc, x.dim() > 1 ? y : y.view({n}));
    });
}

// rms_norm_gemv(fmt, w, x, norm_weight, eps, n, k, scratch)
PyObject *rms_norm_gemv(PyObject *, PyObject *const *a, Py_ssize_t na)
{
    return guarded(na, 8, [&]() -> PyObject * {
        const int fmt = whole(a[0]), n = whole(a[5]), k = whole(a[6]);
        const float eps = real(a[4]);
        const at::Tensor &w = device_tensor(a[1], at::kByte), &x = device_tensor(a[2], at::kFloat), &nw = device_tensor(a[3], at::kFloat);
        const int m = rows_of(x, k);
        if (nw.numel() != k || a[7] != Py_True) throw NotHere{};
        at::Tensor y = at::empty({m, n}, x.options().requires_grad(false)), tmp = at::empty({m, k}, x.options().requires_grad(false));
        const void *wp = w.data_ptr();
        const float *xp = (const float *)x.data_ptr(), *np = (const float *)nw.data_ptr();
        float *yp = (float *)y.data_ptr(), *tp = (float *)tmp.data_ptr();
        const size_t bytes = (size_t)w.numel();
        void *s = stream();
        const int rc = unlocked([&] { return rfq_rms_norm_gemv(fmt, wp, bytes, xp, np, eps, yp, m, n, k, tp, s); });
        return finished(rc, x.dim() > 1 ? y : y.view({n}));
    });
}

// mlp_swiglu(fmt_gate_up, gate_w, up_w, fmt_down, down_w, x, norm_weight, eps, hidden, inter, scratch)
PyObject *mlp_swiglu(PyObject *, PyObject *const *a, Py_ssize_t na)
{
    return guarded(na, 11, [&]() -> PyObject * {
        const int fmt = whole(a[0]), fmt_down = whole(a[3]), hidden = whole(a[8]), inter = whole(a[9]);
        const float eps = real(a[7]);
        const at::Tensor &gate = device_tensor(a[1], at::kByte), &up = device_tensor(a[2], at::kByte), &down = device_tensor(a[4], at::kByte);
        const at::Tensor &x = device_tensor(a[5], at::kFloat);
        if (gate.numel() != up.numel()) throw NotHere{};
        const int m = rows_of(x, hidden);
        const float *np = nullptr;
        if (a[6] != Py_None) {
            const at::Tensor &nw = device_tensor(a[6], at::kFloat);
            if (nw.numel() != hidden) throw NotHere{};
            np = (const float *)nw.data_ptr();
        }
        at::Tensor tmp;
        if (a[10] == Py_None) {
            tmp = at::empty({(int64_t)rfq_mlp_scratch_bytes(m, hidden, inter)}, x.options().dtype(at::kByte).requires_grad(false));
        } else {
            tmp = device_tensor(a[10], at::kByte);
            if (tmp.device() != x.device()) throw NotHere{};
        }
        at::Tensor y = at::empty({m, hidden}, x.options().requires_grad(false));
        const void *gp = gate.data_ptr(), *upp = up.data_ptr(), *dp = down.data_ptr();
        const float *xp = (const float *)x.data_ptr();
        float *yp = (float *)y.data_ptr();
        void *tp = tmp.data_ptr(), *s = stream();
        const size_t bytes = (size_t)gate.numel(), down_bytes = (size_t)down.numel(), tmp_bytes = (size_t)tmp.numel();
        const int rc = unlocked([&] {
            return rfq_mlp_swiglu(fmt, gp, upp, bytes, fmt_down, dp, down_bytes, xp, np, eps, yp, m, hidden, inter, tp, tmp_bytes, s);
        });
        return finished(rc, x.dim() > 1 ? y : y.view({hidden}));
    });
}

// gemm_f16(fmt, w, a, n, k, f16, out_code, out): f16: the result's type, out_code: the library's
PyObject *gemm_f16(PyObject *, PyObject *const *a, Py_ssize_t na)
{
    return guarded(na, 8, [&]() -> PyObject * {
        const int fmt = whole(a[0]), n = whole(a[3]), k = whole(a[4]), code = whole(a[6]);
        const at::Tensor &w = device_tensor(a[1], at::kByte), &x = device_tensor(a[2], at::kHalf);
        if (x.dim() != 2) throw NotHere{};
        const int m = rows_of(x, k);
        at::Tensor y = result(a[7], {m, n}, a[5] == Py_True ? at::kHalf : at::kFloat, x);
        const void *wp = w.data_ptr(), *xp = x.data_ptr();
        void *yp = y.data_ptr(), *s = stream();
        const size_t bytes = (size_t)w.numel();
        const int rc = unlocked([&] { return rfq_gemm_f16(fmt, wp, bytes, xp, yp, code, m, n, k, s); });
        return finished(rc, y);
    });
}

// arrange(a) -> the arranged buffer
PyObject *arrange(PyObject *, PyObject *const *a, Py_ssize_t na)
{
    return guarded(na, 1, [&]() -> PyObject * {
        const at::Tensor &x = device_tensor(a[0], at::kHalf);
        if (x.dim() != 2 || x.size(0) > 0x7fffffff || x.size(1) > 0x7fffffff) throw NotHere{};
        const int m = (int)x.size(0), k = (int)x.size(1);
        const size_t bytes = rfq_gemm_f16_arranged_bytes(m, k);
        if (bytes == 0) throw NotHere{};
        at::Tensor y = at::empty({(int64_t)bytes}, x.options().dtype(at::kByte).requires_grad(false));
        const void *xp = x.data_ptr();
        void *yp = y.data_ptr(), *s = stream();
        const int rc = unlocked([&] { return rfq_gemm_f16_arrange(xp, m, k, yp, bytes, s); });
        return finished(rc, y);
    });
}

// gemm_f16_arranged(fmt, w, buf, m, n, k, f16, out_code, out)
PyObject *gemm_f16_arranged(PyObject *, PyObject *const *a, Py_ssize_t na)
{
    return guarded(na, 9, [&]() -> PyObject * {
        const int fmt = whole(a[0]), m = whole(a[3]), n = whole(a[4]), k = whole(a[5]), code = whole(a[7]);
        const at::Tensor &w = device_tensor(a[1], at::kByte), &b = device_tensor(a[2], at::kByte);
        at::Tensor y = result(a[8], {m, n}, a[6] == Py_True ? at::kHalf : at::kFloat, b);
        const void *wp = w.data_ptr(), *bp = b.data_ptr();
        void *yp = y.data_ptr(), *s = stream();
        const size_t bytes = (size_t)w.numel(), b_bytes = (size_t)b.numel();
        const int rc = unlocked([&] { return rfq_gemm_f16_arranged(fmt, wp, bytes, bp, b_bytes, yp, code, m, n, k, s); });
        return finished(rc, y);
    });
}

// dequant(fmt, packed, n_elems, out)
PyObject *dequant(PyObject *, PyObject *const *a, Py_ssize_t na)
{
    return guarded(na, 4, [&]() -> PyObject * {
        const int fmt = whole(a[0]);
        const at::Tensor &w = device_tensor(a[1], at::kByte);
        if (!PyLong_CheckExact(a[2])) throw NotHere{};
        int over = 0;
        const long long n = PyLong_AsLongLongAndOverflow(a[2], &over);
        if (over != 0 || n < 0) throw NotHere{};
        at::Tensor y = result(a[3], {(int64_t)n}, at::kFloat, w);
        const void *wp = w.data_ptr();
        float *yp = (float *)y.data_ptr();
        void *s = stream();
        const size_t bytes = (size_t)w.numel();
        const int rc = unlocked([&] { return rfq_dequant(fmt, wp, bytes, yp, (size_t)n, s); });
        return finished(rc, y);
    });
}

PyObject *set_check(PyObject *, PyObject *f)
{
    Py_INCREF(f);
    Py_XSETREF(g_check, f);
    Py_RETURN_NONE;
}

#define RFQ_FAST(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {RFQ_FAST(gemv), RFQ_FAST(rms_norm_gemv), RFQ_FAST(mlp_swiglu), RFQ_FAST(gemm_f16), RFQ_FAST(arrange),
                         RFQ_FAST(gemm_f16_arranged), RFQ_FAST(dequant), {"set_check", set_check, METH_O, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

} // namespace

// (the version whose C++ interface this was compiled over: nothing promises that another one's is the same)
PyMODINIT_FUNC PyInit__native()
{
    PyObject *m = PyModule_Create(&module);
    if (m != nullptr && PyModule_AddStringConstant(m, "torch_version", RFQ_TORCH_VERSION) < 0) Py_CLEAR(m);
    return m;
}
