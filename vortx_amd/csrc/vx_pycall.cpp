// vx_pycall.cpp — the Python binding's calls with torch tensors, as a CPython
// extension (vortx_amd/_pycall.<Python's tag>.so).
//
// Building the views of a call with ctypes structures took about 9 us of
// host time a call; reading the tensors' attributes through the C API instead
// takes 1 to 2. Calls whose kernel is shorter than that ran at the host's pace
// (a Q4_0 product at batch 1, 4096 x 4096: 11.4 us a call, now 5.6; a 64 x 64
// x 64 GEMM 13.0, now 7.0). These functions know only the plain case: exact
// torch.Tensor objects on the GPU of the expected element type, at most rank
// 4, streams by their cuda_stream attribute. For anything else (layout pairs,
// subclasses, wrong types, an exception on the way) they return None and the
// caller takes the ctypes path, which handles it or raises.
// Nothing is kept between calls.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <cstdint>
#include <initializer_list>

#include "vortx_hip.h"

namespace {

PyObject *g_qweight, *g_tensor, *g_f32, *g_raw_stream, *g_get_device;  // setup()
PyObject *s_dtype, *s_is_cuda, *s_shape, *s_stride, *s_data_ptr, *s_element_size, *s_cuda_stream, *s_data, *s_qtype, *s_rows,
    *s_cols, *s_row_stride, *s_is_contiguous, *s_nbytes;

struct Ref {  // owned reference
    PyObject* o;
    explicit Ref(PyObject* p) : o(p) {}
    ~Ref() { Py_XDECREF(o); }
    Ref(const Ref&) = delete;
    Ref& operator=(const Ref&) = delete;
};

bool as_u64(PyObject* o, uint64_t max, uint64_t* out) {
    if (!o || !PyLong_CheckExact(o)) return false;
    const unsigned long long v = PyLong_AsUnsignedLongLong(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) return false;
    *out = v;
    return v <= max;
}

bool attr_u64(PyObject* o, PyObject* name, uint64_t max, uint64_t* out) {
    Ref a(PyObject_GetAttr(o, name));
    return as_u64(a.o, max, out);
}

bool call_u64(PyObject* o, PyObject* name, uint64_t max, uint64_t* out) {
    Ref a(PyObject_CallMethodNoArgs(o, name));
    return as_u64(a.o, max, out);
}

bool is_gpu_tensor(PyObject* v) {
    if ((PyObject*)Py_TYPE(v) != g_tensor) return false;
    Ref c(PyObject_GetAttr(v, s_is_cuda));
    return c.o == Py_True;
}

// any4: any element type of four bytes, else float32
template <class View>
bool view_of(PyObject* v, bool any4, View* out) {
    if (!is_gpu_tensor(v)) return false;
    {
        Ref d(PyObject_GetAttr(v, s_dtype));
        uint64_t es = 0;
        if (d.o != g_f32 && !(any4 && d.o && call_u64(v, s_element_size, 4, &es) && es == 4)) return false;
    }
    Ref shape(PyObject_GetAttr(v, s_shape)), stride(PyObject_CallMethodNoArgs(v, s_stride));
    if (!shape.o || !stride.o || !PyTuple_Check(shape.o) || !PyTuple_Check(stride.o)) return false;
    const Py_ssize_t n = PyTuple_GET_SIZE(shape.o);
    if (n > 4 || PyTuple_GET_SIZE(stride.o) != n) return false;
    vx_layout& l = out->layout;
    for (int i = 0; i < 4; ++i) {
        uint64_t sz = 1, st = 1;
        if (i < n && (!as_u64(PyTuple_GET_ITEM(shape.o, i), UINT32_MAX, &sz) ||
                      !as_u64(PyTuple_GET_ITEM(stride.o, i), UINT32_MAX, &st)))
            return false;
        l.size[i] = (uint32_t)sz;
        l.stride[i] = (uint32_t)st;
    }
    l.rank = (uint32_t)n;
    l.offset = 0;  // in the pointer
    uint64_t p = 0;
    if (!call_u64(v, s_data_ptr, UINT64_MAX, &p) || !p) return false;  // (0: torch's for any empty view)
    out->base = (decltype(out->base))(uintptr_t)p;
    return true;
}

bool weight_of(PyObject* w, vx_qweight* out) {
    if ((PyObject*)Py_TYPE(w) != g_qweight) return false;
    Ref data(PyObject_GetAttr(w, s_data));
    uint64_t p = 0, q = 0, r = 0, c = 0, rs = 0;
    if (!data.o || !call_u64(data.o, s_data_ptr, UINT64_MAX, &p) || !attr_u64(w, s_qtype, UINT32_MAX, &q) ||
        !attr_u64(w, s_rows, UINT32_MAX, &r) || !attr_u64(w, s_cols, UINT32_MAX, &c) ||
        !attr_u64(w, s_row_stride, UINT64_MAX, &rs))
        return false;
    *out = vx_qweight{(const void*)(uintptr_t)p, (uint32_t)q, (uint32_t)r, (uint32_t)c, 0u, rs};
    return true;
}

// torch.cuda.current_stream().cuda_stream, or the attribute of the given one
bool stream_of(PyObject* s, vx_stream* out) {
    uint64_t v = 0;
    if (s == Py_None) {
        if (g_raw_stream == Py_None || g_get_device == Py_None) return false;
        Ref dev(PyObject_CallNoArgs(g_get_device));
        if (!dev.o) return false;
        Ref raw(PyObject_CallOneArg(g_raw_stream, dev.o));
        if (!as_u64(raw.o, UINT64_MAX, &v)) return false;
    } else if (!attr_u64(s, s_cuda_stream, UINT64_MAX, &v)) {
        return false;
    }
    *out = (vx_stream)(uintptr_t)v;
    return true;
}

void* addr(PyObject* o) {
    uint64_t v = 0;
    return as_u64(o, UINT64_MAX, &v) ? (void*)(uintptr_t)v : nullptr;
}

PyObject* other_path() {
    PyErr_Clear();
    Py_RETURN_NONE;
}

template <class F>
PyObject* run(F f) {
    int s;
    Py_BEGIN_ALLOW_THREADS
    s = f();
    Py_END_ALLOW_THREADS
    return PyLong_FromLong(s);
}

// setup(QWeight, torch.Tensor, torch.float32, raw stream of a device | None, current device | None)
PyObject* py_setup(PyObject*, PyObject* const* a, Py_ssize_t n) {
    PyObject** g[] = {&g_qweight, &g_tensor, &g_f32, &g_raw_stream, &g_get_device};
    if (n != 5) return PyErr_Format(PyExc_TypeError, "setup takes 5 arguments");
    for (int i = 0; i < 5; ++i) {
        Py_INCREF(a[i]);
        Py_XSETREF(*g[i], a[i]);
    }
    Py_RETURN_NONE;
}

// gemm(fn, ctx, stream, out, lhs, rhs[, alpha, beta, flags]): fn a vx_gemm_f32 or, with the options, vx_gemm_f32_ex
PyObject* py_gemm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 6 && n != 9) return other_path();
    void* fn = addr(a[0]);
    vx_ctx ctx = (vx_ctx)addr(a[1]);
    vx_stream st;
    vx_mview o;
    vx_cview l, r;
    if (!fn || PyErr_Occurred() || !view_of(a[3], false, &o) || !view_of(a[4], false, &l) || !view_of(a[5], false, &r) ||
        !stream_of(a[2], &st))
        return other_path();
    if (n == 6) {
        auto f = (int (*)(vx_ctx, vx_stream, const vx_mview*, const vx_cview*, const vx_cview*))fn;
        return run([&] { return f(ctx, st, &o, &l, &r); });
    }
    uint64_t flags = 0;
    const double al = PyFloat_AsDouble(a[6]), be = PyFloat_AsDouble(a[7]);
    if (PyErr_Occurred() || !as_u64(a[8], UINT32_MAX, &flags)) return other_path();
    const vx_gemm_opts opts{(float)al, (float)be, (uint32_t)flags, 0u};
    auto f = (int (*)(vx_ctx, vx_stream, const vx_mview*, const vx_cview*, const vx_cview*, const vx_gemm_opts*))fn;
    return run([&] { return f(ctx, st, &o, &l, &r, &opts); });
}

// gemv(vx_gemv_q_ex, vx_gemv_q_ws, ctx, stream, y, w, x, flags, workspace | None)
PyObject* py_gemv(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 9) return other_path();
    void *fex = addr(a[0]), *fws = addr(a[1]);
    vx_ctx ctx = (vx_ctx)addr(a[2]);
    vx_stream st;
    vx_mview y;
    vx_cview x;
    vx_qweight w;
    uint64_t flags = 0, wp = 0, wn = 0;
    if (!fex || !fws || PyErr_Occurred() || !view_of(a[4], false, &y) || !view_of(a[6], false, &x) || !weight_of(a[5], &w) ||
        !as_u64(a[7], UINT32_MAX, &flags) || !stream_of(a[3], &st))
        return other_path();
    if (a[8] == Py_None) {
        auto f = (int (*)(vx_ctx, vx_stream, const vx_mview*, const vx_qweight*, const vx_cview*, uint32_t))fex;
        return run([&] { return f(ctx, st, &y, &w, &x, (uint32_t)flags); });
    }
    if (!is_gpu_tensor(a[8])) return other_path();
    Ref c(PyObject_CallMethodNoArgs(a[8], s_is_contiguous));
    if (c.o != Py_True || !call_u64(a[8], s_data_ptr, UINT64_MAX, &wp) || !attr_u64(a[8], s_nbytes, UINT64_MAX, &wn))
        return other_path();
    auto f = (int (*)(vx_ctx, vx_stream, const vx_mview*, const vx_qweight*, const vx_cview*, uint32_t, void*, uint64_t))fws;
    return run([&] { return f(ctx, st, &y, &w, &x, (uint32_t)flags, (void*)(uintptr_t)wp, wn); });
}

// dequantize(fn, ctx, stream, out, w)
PyObject* py_dequantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 5) return other_path();
    auto f = (int (*)(vx_ctx, vx_stream, const vx_mview*, const vx_qweight*))addr(a[0]);
    vx_ctx ctx = (vx_ctx)addr(a[1]);
    vx_stream st;
    vx_mview o;
    vx_qweight w;
    if (!f || PyErr_Occurred() || !view_of(a[3], false, &o) || !weight_of(a[4], &w) || !stream_of(a[2], &st)) return other_path();
    return run([&] { return f(ctx, st, &o, &w); });
}

// quantize(fn, ctx, stream, w, x)
PyObject* py_quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 5) return other_path();
    auto f = (int (*)(vx_ctx, vx_stream, const vx_qweight*, const vx_cview*))addr(a[0]);
    vx_ctx ctx = (vx_ctx)addr(a[1]);
    vx_stream st;
    vx_cview x;
    vx_qweight w;
    if (!f || PyErr_Occurred() || !weight_of(a[3], &w) || !view_of(a[4], false, &x) || !stream_of(a[2], &st)) return other_path();
    return run([&] { return f(ctx, st, &w, &x); });
}

// contiguous(fn, ctx, stream, out, src)
PyObject* py_contiguous(PyObject*, PyObject* const* a, Py_ssize_t n) {
    if (n != 5) return other_path();
    auto f = (int (*)(vx_ctx, vx_stream, const vx_mview*, const vx_cview*, const uint32_t*))addr(a[0]);
    vx_ctx ctx = (vx_ctx)addr(a[1]);
    vx_stream st;
    vx_mview o;
    vx_cview v;
    if (!f || PyErr_Occurred() || !view_of(a[3], true, &o) || !view_of(a[4], true, &v) || !stream_of(a[2], &st)) return other_path();
    return run([&] { return f(ctx, st, &o, &v, nullptr); });
}

#define FAST(f) (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr
PyMethodDef methods[] = {{"setup", FAST(py_setup)},           {"gemm", FAST(py_gemm)},
                         {"gemv", FAST(py_gemv)},             {"dequantize", FAST(py_dequantize)},
                         {"quantize", FAST(py_quantize)},     {"contiguous", FAST(py_contiguous)},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_pycall", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__pycall(void) {
    struct {
        PyObject** s;
        const char* n;
    } names[] = {{&s_dtype, "dtype"},       {&s_is_cuda, "is_cuda"},           {&s_shape, "shape"},
                 {&s_stride, "stride"},     {&s_data_ptr, "data_ptr"},         {&s_element_size, "element_size"},
                 {&s_cuda_stream, "cuda_stream"}, {&s_data, "data"},           {&s_qtype, "qtype"},
                 {&s_rows, "rows"},         {&s_cols, "cols"},                 {&s_row_stride, "row_stride"},
                 {&s_is_contiguous, "is_contiguous"}, {&s_nbytes, "nbytes"}};
    for (auto& e : names)
        if (!(*e.s = PyUnicode_InternFromString(e.n))) return nullptr;
    for (PyObject** g : {&g_qweight, &g_tensor, &g_f32, &g_raw_stream, &g_get_device}) {  // nothing matches before setup()
        Py_INCREF(Py_None);
        *g = Py_None;
    }
    return PyModule_Create(&module);
}
