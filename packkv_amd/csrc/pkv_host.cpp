// The host side of the calls that a decode loop repeats, in native code: the checks, the argument block and the result
// tensors of ops.attn_decode, AttnPlan's step, ops.window_append, ops.dense_view and the four matrix-vector ops.
//
// A decode step is two such calls around 12 us of GPU time, and in Python their checks and ctypes' conversions take 6 to
// 12 us each besides the launch.  Every function here serves the usual call and gives up on any other before it has done
// anything (it returns None): ops.py then goes on with the general code, which copies what has to be copied and
// words what has to be refused.  So nothing is refused here, and what is served meets every condition the general code checks.
// Host time in us a call, general code -> here: attn_decode 15.5 -> 7.8 (two launches in it), window_append 7.3 -> 3.2 (one), the
// cache's attend 8.8 -> 4.3, fused_kq with its wait 16.2 -> 11.5.  Whole passes of one tree without and with this file: a request of 509
// tokens and 24 steps in two layers 1562 -> 1089, a prompt of 3001 tokens and six steps that return the dense tensors 294 -> 192, the four
// matrix-vector ops over 65536 tokens 101 -> 86.  Without it, or with one that was built for another torch, the general code serves.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/packkv.h"

namespace {

struct Library {                   // libpackkv_hip.so, as _lib.py has loaded it
    decltype(&pkv_attn_decode) attn_decode = nullptr;
    decltype(&pkv_window_append) window_append = nullptr;
    decltype(&pkv_dense_view) dense_view = nullptr;
    decltype(&pkv_kq_mat_vec_mul) kq = nullptr;
    decltype(&pkv_wv_mat_vec_mul) wv = nullptr;
    decltype(&pkv_fused_kq) fused_kq = nullptr;
    decltype(&pkv_fused_wv) fused_wv = nullptr;
} lib;

// A plain torch.Tensor (a subclass, or a mode that wants to see the calls, gets the general code).
const at::Tensor *tensor(PyObject *o) { return o && THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }
bool modes() { return at::impl::torch_function_mode_enabled(); }

// The tensor's memory is addressable and lies on device `dev`.
bool there(const at::Tensor &t, int dev) { return t.is_cuda() && t.get_device() == dev && t.has_storage() && t.layout() == at::kStrided; }
bool dense(const at::Tensor &t, int dev) { return there(t, dev) && t.is_contiguous(); }
bool half(const at::Tensor &t) { return t.scalar_type() == at::kHalf || t.scalar_type() == at::kBFloat16; }
int code(const at::Tensor &t) { return t.scalar_type() == at::kHalf ? PKV_F16 : PKV_BF16; }
template <typename T> T *at_ptr(const at::Tensor &t) { return reinterpret_cast<T *>(t.data_ptr()); }

// The current device where `t` lies on it, else -1, which is no tensor's.  (HIP is not asked about a tensor on the host: there may
// be no GPU, and the general code has the words for that.)
int here(const at::Tensor *t) {
    if (!t || !t->is_cuda()) return -1;
    const int dev = c10::hip::current_device();
    return t->get_device() == dev ? dev : -1;
}
pkv_stream_t stream(int dev) { return (pkv_stream_t)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }

// An int argument (a plain Python int within 32 bits).
bool integer(PyObject *o, int *out) {
    if (!o || !PyLong_CheckExact(o)) return false;
    int over = 0;
    const long v = PyLong_AsLongAndOverflow(o, &over);
    if (over || v < INT_MIN || v > INT_MAX) return false;
    *out = (int)v;
    return true;
}

// The library may wait or allocate: other threads go on meanwhile.  `f` calls it and nothing else: no address is taken in there (a lazily
// cloned tensor gets its memory then, and may throw), no Python object touched.
template <typename F> int call(F &&f) {
    int rc;
    Py_BEGIN_ALLOW_THREADS
    rc = f();
    Py_END_ALLOW_THREADS
    return rc;
}

// K's and V's side of a compressed cache, dicts as ops.attn_decode takes them, into `a`.  `batch` 0: from the parameters.
struct Cache {
    int tokens = 0, heads = 0, batch = 0;
    const at::Tensor *like = nullptr;
};
bool cache_args(PyObject *k, PyObject *v, int dev, int batch, pkv_attn_args &a, Cache &c) {
    if (!PyDict_CheckExact(k) || !PyDict_CheckExact(v)) return false;
    const at::Tensor *t[2][4];
    static PyObject *const names[4] = {PyUnicode_InternFromString("stream"), PyUnicode_InternFromString("info"), PyUnicode_InternFromString("scale"),
                                       PyUnicode_InternFromString("zero")};
    static PyObject *const s_bits = PyUnicode_InternFromString("bits"), *const s_tokens = PyUnicode_InternFromString("tokens"),
                    *const s_heads = PyUnicode_InternFromString("heads");
    int bits[2], tokens[2];
    for (int i = 0; i < 2; i++) {
        PyObject *d = i ? v : k;
        for (int f = 0; f < 4; f++) {
            t[i][f] = tensor(PyDict_GetItem(d, names[f]));
            if (!t[i][f] || !dense(*t[i][f], dev)) return false;
        }
        if (t[i][2]->dim() != 2 || t[i][3]->dim() != 2 || t[i][3]->sizes() != t[i][2]->sizes()) return false;
        if (t[i][0]->scalar_type() != at::kByte || t[i][1]->scalar_type() != at::kUInt32) return false;
        if (!integer(PyDict_GetItem(d, s_bits), &bits[i])) return false;
        PyObject *n = PyDict_GetItem(d, s_tokens);
        if (!n) tokens[i] = (int)t[i][2]->size(1);
        else if (!integer(n, &tokens[i])) return false;
    }
    const at::Tensor &scale = *t[0][2];
    if (t[1][2]->sizes() != scale.sizes() || tokens[0] != tokens[1] || tokens[0] < 128 || tokens[0] > scale.size(1) || scale.size(1) > INT_MAX) return false;
    if (scale.size(0) < 1 || (batch && scale.size(0) != batch)) return false;
    c.batch = batch ? batch : (int)scale.size(0);
    c.tokens = tokens[0];
    const int64_t rows = tokens[0] / 64, k_blocks = t[0][1]->numel() / 2, v_blocks = t[1][1]->numel() / 2;
    PyObject *h = PyDict_GetItem(k, s_heads);
    if (!h) c.heads = (int)(k_blocks / rows / c.batch);
    else if (!integer(h, &c.heads)) return false;
    const int64_t blocks = rows * c.batch * c.heads;      // (V: half as many rows of twice the blocks)
    if (c.heads < 1 || k_blocks < blocks || v_blocks < blocks) return false;
    for (int i = 0; i < 2; i++)
        for (int f = 2; f < 4; f++)
            if (t[i][f]->scalar_type() != scale.scalar_type()) return false;
    c.like = &scale;
    a.k_stream = at_ptr<uint8_t>(*t[0][0]); a.k_info = at_ptr<uint32_t>(*t[0][1]); a.k_scale = at_ptr<void>(*t[0][2]); a.k_zero = at_ptr<void>(*t[0][3]);
    a.v_stream = at_ptr<uint8_t>(*t[1][0]); a.v_info = at_ptr<uint32_t>(*t[1][1]); a.v_scale = at_ptr<void>(*t[1][2]); a.v_zero = at_ptr<void>(*t[1][3]);
    a.k_bytes = (uint64_t)t[0][0]->numel();
    a.v_bytes = (uint64_t)t[1][0]->numel();
    a.k_bits = bits[0]; a.v_bits = bits[1];
    a.par_stride = (int)scale.size(1);
    return true;
}

// The 16-bit windows [batch, heads, cap, 128] and the rows in use (None: all).
bool window_args(const at::Tensor *k, const at::Tensor *v, PyObject *rows, int dev, const Cache &c, at::ScalarType type, pkv_attn_args &a) {
    if (!k || !v || !dense(*k, dev) || !dense(*v, dev) || k->dim() != 4 || v->sizes() != k->sizes() || k->scalar_type() != type || v->scalar_type() != type) return false;
    if (k->size(0) != c.batch || k->size(1) != c.heads || k->size(3) != 128 || k->size(2) > INT_MAX) return false;
    a.T_w = (int)k->size(2);
    if (rows != Py_None && !integer(rows, &a.T_w)) return false;
    if (a.T_w < 1 || a.T_w > k->size(2)) return false;
    a.win_stride = (int)k->size(2);
    a.k_win = at_ptr<void>(*k);
    a.v_win = at_ptr<void>(*v);
    return true;
}

PyObject *status(int rc) { return PyLong_FromLong(rc); }

// attn_decode(q, k, v, k_win, v_win, sm_scale, win_len) -> the result, a status that is not zero, or None
PyObject *attn_decode(PyObject *, PyObject *const *o, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *q = n == 7 && !modes() ? tensor(o[0]) : nullptr;
    const int dev = here(q);
    if (dev < 0 || !dense(*q, dev) || !half(*q) || q->dim() != 3 || q->size(2) != 128) Py_RETURN_NONE;
    pkv_attn_args a{};
    Cache c;
    c.batch = (int)q->size(0);
    if (q->size(0) < 1 || q->size(0) > INT_MAX || q->size(1) > INT_MAX) Py_RETURN_NONE;
    if (o[1] != Py_None) {
        if (!cache_args(o[1], o[2], dev, c.batch, a, c) || c.like->scalar_type() != q->scalar_type()) Py_RETURN_NONE;
        if ((reinterpret_cast<uintptr_t>(a.k_stream) | reinterpret_cast<uintptr_t>(a.v_stream)) % 16) Py_RETURN_NONE;
    } else if (o[2] != Py_None) {
        Py_RETURN_NONE;
    }
    if (o[3] != Py_None) {
        const at::Tensor *kw = tensor(o[3]);
        if (o[1] == Py_None && kw && kw->dim() == 4) c.heads = (int)kw->size(1);
        if (!window_args(kw, tensor(o[4]), o[6], dev, c, q->scalar_type(), a)) Py_RETURN_NONE;
    } else if (o[1] == Py_None || o[4] != Py_None) {
        Py_RETURN_NONE;
    }
    a.sm_scale = 0.08838834764831845f;                     // 128 ** -0.5
    if (o[5] != Py_None) {
        if (!PyFloat_CheckExact(o[5])) Py_RETURN_NONE;
        a.sm_scale = (float)PyFloat_AS_DOUBLE(o[5]);
    }
    at::Tensor out = at::empty(q->sizes(), q->options());
    a.q = at_ptr<void>(*q);
    a.out = at_ptr<void>(out);
    a.B = c.batch; a.Hq = (int)q->size(1); a.Hkv = c.heads; a.T_c = c.tokens;
    a.dtype = code(*q);
    const pkv_stream_t s = stream(dev);
    const int rc = call([&] { return lib.attn_decode(&a, nullptr, s); });
    return rc ? status(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// plan_step(address of the plan's arguments, its device, window rows, q) -> the result in q's shape, a status that is not zero, or
// None.  q [B, Hq, 128] or [B, Hq, 1, 128] like the plan's.
PyObject *plan_step(PyObject *, PyObject *const *o, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const at::Tensor *q = n == 4 && !modes() ? tensor(o[3]) : nullptr;
    int plan_dev = -1, rows = 0;
    const int dev = here(q);
    if (dev < 0 || !PyLong_CheckExact(o[0]) || !integer(o[1], &plan_dev) || !integer(o[2], &rows) || plan_dev != dev || !dense(*q, dev)) Py_RETURN_NONE;
    // (a copy: the plan's own q, out and rows stay what its owner has set, and keeps alive)
    pkv_attn_args a = *(const pkv_attn_args *)PyLong_AsVoidPtr(o[0]);
    const int64_t d = q->dim();
    if ((d != 3 && (d != 4 || q->size(2) != 1)) || q->size(0) != a.B || q->size(1) != a.Hq || q->size(d - 1) != 128 ||
        !half(*q) || code(*q) != a.dtype || a.flags || rows < 1 || rows > a.win_stride) Py_RETURN_NONE;
    at::Tensor out = at::empty(q->sizes(), q->options());
    a.q = at_ptr<void>(*q);
    a.out = at_ptr<void>(out);
    a.T_w = rows;
    const pkv_stream_t s = stream(dev);
    const int rc = call([&] { return lib.attn_decode(&a, nullptr, s); });
    return rc ? status(rc) : THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// window_append(k_new, v_new, cos, sin, k_win, v_win, win_pos) -> status or None
PyObject *window_append(PyObject *, PyObject *const *o, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 7 || modes()) Py_RETURN_NONE;
    const at::Tensor *k = tensor(o[0]), *v = tensor(o[1]), *kw = tensor(o[4]), *vw = tensor(o[5]);
    const int dev = here(k);
    int pos = 0;
    if (dev < 0 || !v || !kw || !vw || !there(*k, dev) || !there(*v, dev) || !dense(*kw, dev) || !dense(*vw, dev) || !integer(o[6], &pos)) Py_RETURN_NONE;
    const auto type = k->scalar_type();
    if (k->dim() != 4 || k->size(3) != 128 || v->sizes() != k->sizes() || !half(*k) || v->scalar_type() != type || k->strides() != v->strides() ||
        k->stride(3) != 1 || kw->dim() != 4 || vw->sizes() != kw->sizes() || kw->size(0) != k->size(0) || kw->size(1) != k->size(1) ||
        kw->size(3) != 128 || kw->scalar_type() != type || vw->scalar_type() != type) Py_RETURN_NONE;
    const int64_t B = k->size(0), H = k->size(1), rows = k->size(2), cap = kw->size(2);
    if (B > INT_MAX || H > INT_MAX || rows > INT_MAX || cap > INT_MAX) Py_RETURN_NONE;
    const void *cos_p = nullptr, *sin_p = nullptr;
    int64_t rot = 0;
    if (o[2] != Py_None) {
        const at::Tensor *cos = tensor(o[2]), *sin = tensor(o[3]);
        const int64_t shape[3] = {B, rows, 128};
        if (!cos || !sin || !there(*cos, dev) || !there(*sin, dev) || cos->sizes() != at::IntArrayRef(shape, 3) || sin->sizes() != cos->sizes() ||
            cos->scalar_type() != type || sin->scalar_type() != type || cos->strides() != sin->strides() || cos->stride(2) != 1 ||
            (rows > 1 && cos->stride(1) != 128)) Py_RETURN_NONE;
        cos_p = at_ptr<void>(*cos);
        sin_p = at_ptr<void>(*sin);
        rot = B > 1 ? cos->stride(0) : 0;
    }
    const void *const k_p = at_ptr<void>(*k), *const v_p = at_ptr<void>(*v);
    void *const kw_p = at_ptr<void>(*kw), *const vw_p = at_ptr<void>(*vw);
    const int64_t sb = k->stride(0), sh = k->stride(1), st = k->stride(2);
    const int dtype = code(*k);
    const pkv_stream_t s = stream(dev);
    return status(call([&] { return lib.window_append(k_p, v_p, cos_p, sin_p, dtype, (int)B, (int)H, (int)rows, sb, sh, st, rot, kw_p, vw_p, pos, (int)cap, s); }));
    END_HANDLE_TH_ERRORS
}

// dense_view(k, v, k_win, v_win, win_len) -> (K, V), a status that is not zero, or None
PyObject *dense_view(PyObject *, PyObject *const *o, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 5 || modes() || !PyDict_CheckExact(o[0])) Py_RETURN_NONE;
    const int dev = here(tensor(PyDict_GetItemString(o[0], "scale")));
    pkv_attn_args a{};
    Cache c;
    if (dev < 0 || !cache_args(o[0], o[1], dev, 0, a, c) || !half(*c.like)) Py_RETURN_NONE;
    if (o[2] != Py_None && !window_args(tensor(o[2]), tensor(o[3]), o[4], dev, c, c.like->scalar_type(), a)) Py_RETURN_NONE;
    a.B = c.batch; a.Hkv = c.heads; a.T_c = c.tokens;
    a.dtype = code(*c.like);
    at::Tensor k = at::empty({c.batch, c.heads, (int64_t)c.tokens + a.T_w, 128}, c.like->options()), v = at::empty_like(k);
    void *const k_p = at_ptr<void>(k), *const v_p = at_ptr<void>(v);
    const pkv_stream_t s = stream(dev);
    const int rc = call([&] { return lib.dense_view(&a, k_p, v_p, s); });
    if (rc) return status(rc);
    PyObject *both = PyTuple_New(2);
    if (!both) return nullptr;
    PyTuple_SET_ITEM(both, 0, THPVariable_Wrap(std::move(k)));
    PyTuple_SET_ITEM(both, 1, THPVariable_Wrap(std::move(v)));
    return both;
    END_HANDLE_TH_ERRORS
}

// A timed op: milliseconds, a status that is not zero, or None.
template <typename F> PyObject *timed(F &&f) {
    float ms = 0.f;
    const int rc = call([&] { return f(&ms); });
    return rc ? status(rc) : PyFloat_FromDouble((double)ms);
}

// mat_vec(is_k, stream, info, x, out, ctx_len, hidden_dim, ctx_blk, hid_blk, bits, interleaved)
PyObject *mat_vec(PyObject *, PyObject *const *o, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 11 || modes()) Py_RETURN_NONE;
    const bool is_k = o[0] == Py_True;
    const at::Tensor *stm = tensor(o[1]), *info = tensor(o[2]), *x = tensor(o[3]), *out = tensor(o[4]);
    const int dev = here(x);
    int i[5];
    for (int j = 0; j < 5; j++)
        if (!integer(o[5 + j], &i[j])) Py_RETURN_NONE;
    if (dev < 0 || !stm || !info || !out || !there(*stm, dev) || !there(*info, dev) || !there(*x, dev) || !there(*out, dev) || !half(*x) ||
        (!is_k && out->scalar_type() != at::kFloat) || (o[10] != Py_True && o[10] != Py_False)) Py_RETURN_NONE;
    const uint64_t bytes = (uint64_t)stm->numel() * (uint64_t)stm->element_size();
    const uint8_t *const stm_p = at_ptr<uint8_t>(*stm);
    const uint32_t *const info_p = at_ptr<uint32_t>(*info);
    const void *const x_p = at_ptr<void>(*x);
    void *const out_p = at_ptr<void>(*out);
    const int dtype = code(*x), interleaved = o[10] == Py_True;
    const pkv_stream_t s = stream(dev);
    if (is_k) return timed([&](float *ms) { return lib.kq(stm_p, bytes, info_p, x_p, out_p, i[0], i[1], i[2], i[3], i[4], dtype, interleaved, ms, s); });
    return timed([&](float *ms) { return lib.wv(stm_p, bytes, info_p, x_p, (float *)out_p, i[0], i[1], i[2], i[3], i[4], dtype, ms, s); });
    END_HANDLE_TH_ERRORS
}

// fused(is_k, out, x, zero, scale, t): ops.fused_kq(out, x = q, zero, scale, t) or ops.fused_wv(out, x = w, zero, scale, t = term1)
PyObject *fused(PyObject *, PyObject *const *o, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 6 || modes()) Py_RETURN_NONE;
    const bool is_k = o[0] == Py_True;
    const at::Tensor *out = tensor(o[1]), *x = tensor(o[2]), *zero = tensor(o[3]), *scale = tensor(o[4]), *t = tensor(o[5]);
    const int dev = here(x);
    if (dev < 0 || !out || !zero || !scale || !t || !dense(*out, dev) || !dense(*x, dev) || !dense(*zero, dev) || !dense(*scale, dev) || !dense(*t, dev) ||
        !half(*x)) Py_RETURN_NONE;
    if (out->dim() != 2 || x->dim() != 2 || t->dim() != 2 || zero->dim() != 1 || scale->dim() != 1) Py_RETURN_NONE;
    const int64_t M = x->size(0), K = x->size(1), T = t->size(1), columns = is_k ? T : K;
    if (t->size(0) != M || zero->size(0) != columns || scale->size(0) != columns || out->size(0) != M || out->size(1) != T ||
        (!is_k && t->scalar_type() != x->scalar_type()) || M > INT_MAX || K > INT_MAX || T > INT_MAX) Py_RETURN_NONE;
    void *const out_p = at_ptr<void>(*out);
    const void *const x_p = at_ptr<void>(*x), *const zero_p = at_ptr<void>(*zero), *const scale_p = at_ptr<void>(*scale), *const t_p = at_ptr<void>(*t);
    const int dtype = code(*x);
    const pkv_stream_t s = stream(dev);
    return timed([&](float *ms) { return (is_k ? lib.fused_kq : lib.fused_wv)(out_p, x_p, zero_p, scale_p, t_p, (int)M, (int)K, (int)T, dtype, ms, s); });
    END_HANDLE_TH_ERRORS
}

// bind(addresses of attn_decode, window_append, dense_view, kq, wv, fused_kq, fused_wv)
PyObject *bind(PyObject *, PyObject *const *o, Py_ssize_t n) {
    void *p[7];
    if (n != 7) {
        PyErr_SetString(PyExc_TypeError, "seven addresses");
        return nullptr;
    }
    for (int i = 0; i < 7; i++) {
        p[i] = PyLong_AsVoidPtr(o[i]);
        if (PyErr_Occurred()) return nullptr;
    }
    lib.attn_decode = (decltype(lib.attn_decode))p[0];
    lib.window_append = (decltype(lib.window_append))p[1];
    lib.dense_view = (decltype(lib.dense_view))p[2];
    lib.kq = (decltype(lib.kq))p[3];
    lib.wv = (decltype(lib.wv))p[4];
    lib.fused_kq = (decltype(lib.fused_kq))p[5];
    lib.fused_wv = (decltype(lib.fused_wv))p[6];
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
    {"bind", (PyCFunction)(void (*)(void))bind, METH_FASTCALL, nullptr},
    {"attn_decode", (PyCFunction)(void (*)(void))attn_decode, METH_FASTCALL, nullptr},
    {"plan_step", (PyCFunction)(void (*)(void))plan_step, METH_FASTCALL, nullptr},
    {"window_append", (PyCFunction)(void (*)(void))window_append, METH_FASTCALL, nullptr},
    {"dense_view", (PyCFunction)(void (*)(void))dense_view, METH_FASTCALL, nullptr},
    {"mat_vec", (PyCFunction)(void (*)(void))mat_vec, METH_FASTCALL, nullptr},
    {"fused", (PyCFunction)(void (*)(void))fused, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host(void) {
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch", PKV_TORCH_VERSION)) Py_CLEAR(m);
    return m;
}
