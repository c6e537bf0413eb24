// Native call path of the Python op interface (tileinfer_hip/backend.py): reads the tensors,
// checks them as backend.py does and calls the C ABI, without building ctypes structures.
//
// Every function returns the ti_status of the call, or -1 where it takes the arguments not to
// be plain ones (a tensor subclass, a CPU or non-contiguous tensor, a shape or type that does
// not fit): backend.py then runs its own checks, which raise, or make the call. So what is
// accepted and what is raised is defined there alone.
//
// Why: attention_inputs_ and paged_attention_ of a short step took 20.8 us a pair through
// Python checks and ctypes, whatever the GPU needed (its three kernels 8 to 12); here 9.3 us,
// and one float32 token (16 / 8 heads, 1024 positions) 23.8 -> 11.3 us.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "tileinfer_hip.h"

namespace {

decltype(&ti_attention) f_attention;
decltype(&ti_attention_inputs) f_inputs;
decltype(&ti_store_kv) f_store_kv;
decltype(&ti_rope) f_rope;
decltype(&ti_rmsnorm) f_rmsnorm;
PyObject *int8_pages, *n_layer_q, *n_layer_scale, *n_smooth, *n_half, *n_cos_sin;   // Int8Pages, attribute names

struct NotPlain {};   // leave the call to backend.py

// A plain GPU tensor of contiguous elements.
const at::Tensor &dev(PyObject *o) {
    if (!THPVariable_CheckExact(o)) throw NotPlain{};
    const at::Tensor &t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.layout() != at::kStrided || !t.is_contiguous()) throw NotPlain{};
    return t;
}
const at::Tensor *dev_or_none(PyObject *o) { return o == Py_None ? nullptr : &dev(o); }
void require(bool ok) {
    if (!ok) throw NotPlain{};
}
const int32_t *i32(const at::Tensor &t) {
    require(t.scalar_type() == at::kInt);
    return static_cast<const int32_t *>(t.data_ptr());
}
int dtype_of(const at::Tensor &t) {
    if (t.scalar_type() == at::kBFloat16) return TI_BF16;
    require(t.scalar_type() == at::kFloat);
    return TI_F32;
}
float number(PyObject *o) {
    require(PyFloat_CheckExact(o) || PyLong_CheckExact(o));
    const double x = PyFloat_AsDouble(o);
    require(!PyErr_Occurred());
    return (float)x;
}
long integer(PyObject *o) {
    require(PyLong_CheckExact(o));
    const long x = PyLong_AsLong(o);
    require(!PyErr_Occurred());
    return x;
}
void *stream_of(const at::Tensor &t) { return c10::hip::getCurrentHIPStream(t.device().index()).stream(); }

// An attribute held for the scope of a call.
struct Attr {
    PyObject *o;
    Attr(PyObject *of, PyObject *name) : o(PyObject_GetAttr(of, name)) { require(o != nullptr); }
    ~Attr() { Py_DECREF(o); }
    Attr(const Attr &) = delete;
};

// The layer's cache: dense pools [pages][H][P][D] of element type `like`, or an Int8Pages pair.
ti_kv_cache cache_of(PyObject *k, PyObject *v, at::ScalarType like) {
    ti_kv_cache c{};
    if ((PyObject *)Py_TYPE(k) == int8_pages || (PyObject *)Py_TYPE(v) == int8_pages) {
        require(Py_TYPE(k) == Py_TYPE(v));
        Attr lq(k, n_layer_q), lq2(v, n_layer_q), ls(k, n_layer_scale), sm(k, n_smooth), h0(k, n_half), h1(v, n_half);
        require(lq.o == lq2.o && integer(h0.o) == 0 && integer(h1.o) == 1);
        const at::Tensor &q = dev(lq.o);
        require(q.dim() == 5);
        c.kind = TI_KV_INT8;
        c.layer_q = static_cast<int8_t *>(q.data_ptr());
        c.layer_scale = static_cast<float *>(dev(ls.o).data_ptr());
        c.smooth = static_cast<const float *>(dev(sm.o).data_ptr());
        c.num_pages = (int32_t)q.size(1), c.kv_heads = (int32_t)q.size(2);
        c.page_size = (int32_t)q.size(3), c.head_dim = (int32_t)q.size(4);
        return c;
    }
    const at::Tensor &kt = dev(k), &vt = dev(v);
    require(kt.dim() == 4 && kt.sizes() == vt.sizes() && kt.scalar_type() == like && vt.scalar_type() == like);
    c.kind = TI_KV_DENSE;
    c.k_pages = kt.data_ptr();
    c.v_pages = vt.data_ptr();
    c.num_pages = (int32_t)kt.size(0), c.kv_heads = (int32_t)kt.size(1);
    c.page_size = (int32_t)kt.size(2), c.head_dim = (int32_t)kt.size(3);
    return c;
}

// Runs `body` (checks, then the call without the interpreter lock) and returns its status.
template <typename F>
PyObject *guarded(Py_ssize_t nargs, Py_ssize_t want, F &&body) {
    long status = -1;
    if (nargs == want && f_attention) {
        try {
            status = body();
        } catch (...) {
            status = -1;
        }
    }
    PyErr_Clear();
    return PyLong_FromLong(status);
}
template <typename F>
long unlocked(F &&call) {
    long status;
    Py_BEGIN_ALLOW_THREADS
    status = call();
    Py_END_ALLOW_THREADS
    return status;
}

// (out, workspace, q, k_pages, v_pages, block_tables, positions, scale, causal,
//  query_start_loc, max_query_len, path, one_sequence)
PyObject *py_attention(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 13, [&]() -> long {
        const at::Tensor &out = dev(a[0]), &q = dev(a[2]), &bt = dev(a[5]), &pos = dev(a[6]);
        const at::Tensor *ws = dev_or_none(a[1]), *qsl = dev_or_none(a[9]);
        require(q.dim() == 3 && out.sizes() == q.sizes() && out.scalar_type() == q.scalar_type());
        const ti_kv_cache c = cache_of(a[3], a[4], q.scalar_type());
        ti_attention_args g{};
        g.dtype = dtype_of(q);
        g.positions = i32(pos);
        g.block_tables = i32(bt);
        require(pos.numel() == q.size(0) && q.size(2) == c.head_dim && PyBool_Check(a[8]));
        const bool rows = bt.dim() == 2 && a[12] != Py_True;
        const int64_t B = rows ? bt.size(0) : 1;
        require(B > 0 && (!qsl || a[10] != Py_None));
        g.q_heads = (int32_t)q.size(1);
        g.num_seqs = (int32_t)B;
        g.max_query_len = (int32_t)(a[10] != Py_None ? integer(a[10]) : q.size(0) / B);
        g.total_tokens = (int32_t)q.size(0);
        g.block_table_stride = (int32_t)(rows ? bt.size(1) : bt.numel());
        g.q = q.data_ptr();
        g.out = out.data_ptr();
        g.query_start_loc = qsl ? i32(*qsl) : nullptr;
        g.scale = number(a[7]);
        g.causal = a[8] == Py_True;
        g.path = (int32_t)integer(a[11]);
        g.workspace = ws ? ws->data_ptr() : nullptr;
        g.workspace_bytes = ws ? (size_t)ws->nbytes() : 0;
        void *s = stream_of(q);
        return unlocked([&] { return f_attention(&g, &c, s); });
    });
}

// (q, k_pages, v_pages, qkv, q_norm, k_norm, table, positions, slots, eps)
PyObject *py_inputs(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 10, [&]() -> long {
        const Attr table(a[6], n_cos_sin);
        const at::Tensor &q = dev(a[0]), &qkv = dev(a[3]), &cs = dev(table.o), &pos = dev(a[7]), &slots = dev(a[8]);
        const at::Tensor *qn = dev_or_none(a[4]), *kn = dev_or_none(a[5]);
        require(q.dim() == 3 && !qn == !kn);
        const int64_t n = q.size(0), nq = q.size(1), D = q.size(2);
        const ti_kv_cache c = cache_of(a[1], a[2], q.scalar_type());
        require(qkv.scalar_type() == q.scalar_type() && qkv.numel() == n * (nq + 2 * (int64_t)c.kv_heads) * D && D == c.head_dim);
        require(cs.scalar_type() == q.scalar_type() && cs.dim() == 3 && cs.size(1) == 2 && cs.size(2) == D);
        require(pos.numel() == n && slots.numel() == n);
        const int dtype = dtype_of(q);
        const int32_t *p = i32(pos), *sl = i32(slots);
        const float eps = number(a[9]);
        void *s = stream_of(q), *qo = q.data_ptr();
        const void *x = qkv.data_ptr(), *w1 = qn ? qn->data_ptr() : nullptr, *w2 = kn ? kn->data_ptr() : nullptr, *t = cs.data_ptr();
        const int len = (int)cs.size(0);
        return unlocked([&] { return f_inputs(dtype, qo, &c, x, w1, w2, t, len, p, sl, (int)n, (int)nq, eps, s); });
    });
}

// (k_pages, v_pages, k, v, slots)
PyObject *py_store_kv(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 5, [&]() -> long {
        const at::Tensor &k = dev(a[2]), &v = dev(a[3]), &slots = dev(a[4]);
        require(k.dim() == 3 && k.sizes() == v.sizes() && k.scalar_type() == v.scalar_type());
        const ti_kv_cache c = cache_of(a[0], a[1], k.scalar_type());
        require(k.size(1) == c.kv_heads && k.size(2) == c.head_dim && slots.numel() == k.size(0));
        const int dtype = dtype_of(k);
        const int32_t *sl = i32(slots);
        void *s = stream_of(k);
        const void *kp = k.data_ptr(), *vp = v.data_ptr();
        const int n = (int)k.size(0);
        return unlocked([&] { return f_store_kv(dtype, &c, kp, vp, sl, n, s); });
    });
}

// (y, x, cos, sin, positions)
PyObject *py_rope(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 5, [&]() -> long {
        const at::Tensor &y = dev(a[0]), &x = dev(a[1]), &c = dev(a[2]), &s = dev(a[3]), &pos = dev(a[4]);
        const auto T = x.scalar_type();
        require(x.dim() == 3 && y.sizes() == x.sizes() && y.scalar_type() == T && c.scalar_type() == T && s.scalar_type() == T);
        require(c.dim() == 2 && c.sizes() == s.sizes() && c.size(1) == x.size(2) && pos.numel() == x.size(0));
        const int dtype = dtype_of(x);
        const int32_t *p = i32(pos);
        void *st = stream_of(x), *yp = y.data_ptr();
        const void *xp = x.data_ptr(), *cp = c.data_ptr(), *sp = s.data_ptr();
        const int len = (int)c.size(0), n = (int)x.size(0), H = (int)x.size(1), D = (int)x.size(2);
        return unlocked([&] { return f_rope(dtype, yp, xp, cp, sp, len, p, n, H, D, st); });
    });
}

// (y, x, w, eps)
PyObject *py_rmsnorm(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    return guarded(nargs, 4, [&]() -> long {
        const at::Tensor &y = dev(a[0]), &x = dev(a[1]), &w = dev(a[2]);
        require(x.dim() >= 1 && y.sizes() == x.sizes() && y.scalar_type() == x.scalar_type() && w.scalar_type() == x.scalar_type());
        const int64_t H = x.size(-1);
        require(H > 0 && w.dim() == 1 && w.size(0) == H);
        const int dtype = dtype_of(x);
        const float eps = number(a[3]);
        void *s = stream_of(x), *yp = y.data_ptr();
        const void *xp = x.data_ptr(), *wp = w.data_ptr();
        const int rows = (int)(x.numel() / H);
        return unlocked([&] { return f_rmsnorm(dtype, yp, xp, wp, rows, (int)H, eps, s); });
    });
}

// bind(Int8Pages, addresses of ti_attention, ti_attention_inputs, ti_store_kv, ti_rope, ti_rmsnorm)
PyObject *py_bind(PyObject *, PyObject *args) {
    PyObject *pages;
    unsigned long long f[5];
    if (!PyArg_ParseTuple(args, "OKKKKK", &pages, &f[0], &f[1], &f[2], &f[3], &f[4])) return nullptr;
    Py_INCREF(pages);
    Py_XDECREF(int8_pages);
    int8_pages = pages;
    f_attention = reinterpret_cast<decltype(f_attention)>(f[0]);
    f_inputs = reinterpret_cast<decltype(f_inputs)>(f[1]);
    f_store_kv = reinterpret_cast<decltype(f_store_kv)>(f[2]);
    f_rope = reinterpret_cast<decltype(f_rope)>(f[3]);
    f_rmsnorm = reinterpret_cast<decltype(f_rmsnorm)>(f[4]);
    Py_RETURN_NONE;
}

#define FAST(name, f) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {FAST("attention", py_attention), FAST("attention_inputs", py_inputs), FAST("store_kv", py_store_kv),
                         FAST("rope", py_rope), FAST("rmsnorm", py_rmsnorm), {"bind", py_bind, METH_VARARGS, nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__calls() {
    n_layer_q = PyUnicode_InternFromString("layer_q");
    n_layer_scale = PyUnicode_InternFromString("layer_scale");
    n_smooth = PyUnicode_InternFromString("smooth");
    n_half = PyUnicode_InternFromString("half");
    n_cos_sin = PyUnicode_InternFromString("cos_sin");
    PyObject *m = PyModule_Create(&module);
    // the torch and Python whose layouts this was compiled for; _lib.py compares
    if (m && PyModule_AddStringConstant(m, "built_for", BUILT_FOR) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
