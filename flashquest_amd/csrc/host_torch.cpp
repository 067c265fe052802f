// Native host path of the per-layer operators: builds the C ABI's descriptors
// from the tensors, allocates the outputs and calls the library, in one C++
// call instead of Python and ctypes.
//
// Why: a serving program calls these once per layer and token, and a decode
// layer's kernels take about 20 us; the Python path took 31 us of host time for
// one (its three launches are 11 of them), 24 for a prefill and 10 for a
// quantiser.  Through here they take 15.6, 9.7 and 6, and an 8k-token layer in a
// loop 23.4 us instead of 29.7, which its kernels now bound.
//
// Every function answers None for whatever is not its plain case (tensor
// subclasses and transforms, other devices, layouts that need a copy, errors of
// any kind the library reports): the Python operators then go their general way,
// which copies, falls back or raises as it always has.  So this file holds no
// rule of its own: its checks are the Python path's conditions for passing the
// tensors through unchanged.
#include <Python.h>

#include <cmath>
#include <optional>

#include <ATen/TensorSubclassLikeUtils.h>
#include <ATen/ops/empty.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include "fq_hip.h"

namespace {

// The library's entries, as addresses from the loaded library (bind()).
struct Entries {
    decltype(&fq_workspace_bytes) ws_int4;
    decltype(&fq_turbo_workspace_bytes) ws_turbo;
    decltype(&fq_quest_decode_int4) decode4;
    decltype(&fq_quest_decode_int8) decode8;
    decltype(&fq_quest_decode_int4_tail) tail4;
    decltype(&fq_quest_decode_int8_tail) tail8;
    decltype(&fq_quest_decode_turbo) decode3;
    decltype(&fq_quest_fused_int4) fused4;
    decltype(&fq_quest_fused_int8) fused8;
    decltype(&fq_quest_fused_turbo) fused3;
    decltype(&fq_prefill_int4) prefill4;
    decltype(&fq_prefill_int8) prefill8;
    decltype(&fq_prefill_workspace_bytes) ws_prefill;
    decltype(&fq_quantize_k_int4) quant_k4;
    decltype(&fq_quantize_k_int8) quant_k8;
    decltype(&fq_quantize_v_int4) quant_v4;
    decltype(&fq_quantize_v_int8) quant_v8;
};
Entries g_fq{};

// An ordinary ROCm tensor (no subclass, transform or tracer), or null.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined() || !t.is_cuda() || t.layout() != at::kStrided || at::isTensorSubclassLike(t)) return nullptr;
    return &t;
}

int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kBFloat16: return FQ_BF16;
        case at::kHalf: return FQ_F16;
        case at::kFloat: return FQ_F32;
        default: return -1;
    }
}

// Unit inner stride, every other stride a multiple of `elems` elements, the data aligned to as many.
bool rows(const at::Tensor& t, int64_t elems = 1) {
    const auto st = t.strides();
    if (st.back() != 1) return false;
    for (size_t i = 0; i + 1 < st.size(); ++i)
        if (st[i] % elems) return false;
    return elems == 1 || (uintptr_t)t.data_ptr() % (elems * t.element_size()) == 0;
}

template <int N>
void strides(const at::Tensor& t, int64_t (&out)[N]) {
    const auto st = t.strides();
    const int lead = N - (int)st.size();
    for (int i = 0; i < N; ++i) out[i] = i < lead ? 0 : st[i - lead];
}

// t: K codes, K scale, K min, V codes, V scale, V min.
bool int_cache(const at::Tensor* const (&t)[6], int bits, int page, fq_int4_cache& c) {
    const int nd = (int)t[0]->dim();
    if (nd != 4 && nd != 5) return false;
    for (int i = 0; i < 6; ++i)
        if (t[i]->dim() != nd || t[i]->device() != t[0]->device()) return false;
    const int meta = dtype_code(*t[1]);
    if (meta != FQ_BF16 && meta != FQ_F16) return false;
    for (int i : {2, 4, 5})
        if (t[i]->scalar_type() != t[1]->scalar_type()) return false;
    if (t[0]->scalar_type() != at::kByte || t[3]->scalar_type() != at::kByte) return false;
    const int align = bits == 8 ? 8 : 4;
    if (!rows(*t[0], align) || !rows(*t[3], align) || !rows(*t[1], 8) || !rows(*t[2], 8) || !rows(*t[4]) || !rows(*t[5]))
        return false;
    c.k_packed = (const uint8_t*)t[0]->data_ptr(); strides(*t[0], c.k_strides);
    c.k_scale = t[1]->data_ptr(); strides(*t[1], c.ks_strides);
    c.k_mn = t[2]->data_ptr(); strides(*t[2], c.km_strides);
    c.v_packed = (const uint8_t*)t[3]->data_ptr(); strides(*t[3], c.v_strides);
    c.v_scale = t[4]->data_ptr(); strides(*t[4], c.vs_strides);
    c.v_mn = t[5]->data_ptr(); strides(*t[5], c.vm_strides);
    c.meta_dtype = meta;
    c.L = nd == 5 ? (int)t[0]->size(0) : 1;
    c.B = (int)t[0]->size(-4);
    c.H_kv = (int)t[0]->size(-3);
    c.S = (int)t[0]->size(-2);
    c.P = (int)t[1]->size(-2);
    c.D = (int)t[0]->size(-1) * (bits == 8 ? 1 : 2);
    c.page_size = page;
    c.v_groups = (int)t[4]->size(-1);
    return c.H_kv == t[1]->size(-3) && (bits == 4 || c.v_groups == 1);
}

// t: K MSB, K LSB, K scale, V MSB, V LSB, V scale; raw: the K page scale and min.
bool turbo_cache(const at::Tensor* const (&t)[6], const at::Tensor* const (&raw)[2], int page, fq_turbo_cache& c) {
    const int nd = (int)t[0]->dim();
    if (nd != 4 && nd != 5) return false;
    const int64_t D = t[0]->size(-1) * 8;
    for (int i = 0; i < 6; ++i) {
        if (t[i]->dim() != nd || t[i]->device() != t[0]->device() || !rows(*t[i])) return false;
        if (t[i]->size(-1) != (i % 3 == 0 ? D / 8 : i % 3 == 1 ? D / 4 : 1)) return false;
    }
    for (const at::Tensor* r : raw)
        if (r->dim() != nd || r->scalar_type() != at::kBFloat16 || r->strides().back() != 1) return false;
    c.k_msb = (const uint8_t*)t[0]->data_ptr(); strides(*t[0], c.kmsb_strides);
    c.k_lsb = (const uint8_t*)t[1]->data_ptr(); strides(*t[1], c.klsb_strides);
    c.k_scale = t[2]->data_ptr(); strides(*t[2], c.kst_strides);
    c.v_msb = (const uint8_t*)t[3]->data_ptr(); strides(*t[3], c.vmsb_strides);
    c.v_lsb = (const uint8_t*)t[4]->data_ptr(); strides(*t[4], c.vlsb_strides);
    c.v_scale = t[5]->data_ptr(); strides(*t[5], c.vst_strides);
    c.L = nd == 5 ? (int)t[0]->size(0) : 1;
    c.B = (int)t[0]->size(-4);
    c.H_kv = (int)t[0]->size(-3);
    c.S = (int)t[0]->size(-2);
    c.P = (int)raw[0]->size(-2);
    c.D = (int)D;
    c.page_size = page;
    return c.P <= (c.S + page - 1) / page;
}

// A partial-page tail (k, v same shape and dtype): 1 attended, 0 none, -1 not plain.
int tail_of(PyObject* k_obj, PyObject* v_obj, int nd, int64_t D, int64_t k_align, int64_t v_align, bool bf16_only,
            fq_tail& t) {
    if (k_obj == Py_None) return 0;
    const at::Tensor* k = plain(k_obj);
    const at::Tensor* v = plain(v_obj);
    if (!k || !v || k->dim() != nd || k->sizes() != v->sizes() || k->scalar_type() != v->scalar_type()) return -1;
    if (k->size(-2) == 0) return 0;
    if (k->size(-1) != D || !rows(*k, k_align) || !rows(*v, v_align)) return -1;
    t.dtype = dtype_code(*k);
    if (t.dtype < 0 || (bf16_only && t.dtype != FQ_BF16)) return -1;
    t.k = k->data_ptr(); strides(*k, t.k_strides);
    t.v = v->data_ptr(); strides(*v, t.v_strides);
    t.len = (int)k->size(-2);
    t.D = (int)D;
    return 1;
}

PyObject* none() { Py_RETURN_NONE; }

// decode(bits, Q, planes (6, or 8 with TurboQuant's raw metadata), retention rows, sinks, window, k_max or -1,
//        mode, page, sm_scale or None, return_lse, K_tail, V_tail, workspace, stream)
//   -> (O, lse or None), or None
// retention rows: (rows, layer stride), or a function of no arguments that gives them, called once everything else
// is known to be the plain case (it may copy to the device and launch), its errors raised.
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 15) return none();
    const int bits = (int)PyLong_AsLong(a[0]);
    const at::Tensor* Q = plain(a[1]);
    const Py_ssize_t np = PyTuple_Check(a[2]) ? PyTuple_GET_SIZE(a[2]) : 0;
    if (!Q || !Q->is_contiguous() || np != (bits == 3 ? 8 : 6)) return none();
    const at::Tensor* t[6];
    const at::Tensor* raw[2] = {nullptr, nullptr};
    for (Py_ssize_t i = 0; i < np; ++i) {
        const at::Tensor* x = plain(PyTuple_GET_ITEM(a[2], i));
        if (!x || x->device() != Q->device()) return none();
        (i < 6 ? t[i] : raw[i - 6]) = x;
    }
    const at::Tensor* ws = a[13] == Py_None ? nullptr : plain(a[13]);
    const int nd = (int)Q->dim();
    if (!ws || nd != t[0]->dim() || Q->size(-2) != 1) return none();
    const int sinks = (int)PyLong_AsLong(a[4]), window = (int)PyLong_AsLong(a[5]);
    int k_max = (int)PyLong_AsLong(a[6]);
    const int mode = (int)PyLong_AsLong(a[7]), page = (int)PyLong_AsLong(a[8]);
    const bool want_lse = a[10] == Py_True;

    fq_int4_cache c{};
    fq_turbo_cache tc{};
    if (bits == 3 ? !turbo_cache(t, raw, page, tc) : !int_cache(t, bits, page, c)) return none();
    const int L = bits == 3 ? tc.L : c.L, B = bits == 3 ? tc.B : c.B, Hkv = bits == 3 ? tc.H_kv : c.H_kv;
    const int D = bits == 3 ? tc.D : c.D, P = bits == 3 ? tc.P : c.P;
    const int Hq = (int)Q->size(-3);
    if (Q->size(-1) != D || Q->size(-4) != B || (nd == 5 && Q->size(0) != L) || Hkv < 1 || Hq % Hkv || Q->numel() == 0)
        return none();
    if (k_max > P) k_max = P;

    fq_query q{};
    q.q = q.out = Q->data_ptr();       // out: until O is there (the fused query below checks for one)
    q.q_dtype = q.out_dtype = dtype_code(*Q);
    if (q.q_dtype < 0) return none();
    // Q (..., H_q, 1, D) and O alike, contiguous: (l, b, h, d) strides
    q.q_strides[0] = nd == 5 ? (int64_t)B * Hq * D : 0;
    q.q_strides[1] = (int64_t)Hq * D;
    q.q_strides[2] = D;
    q.q_strides[3] = 1;
    for (int i = 0; i < 4; ++i) q.o_strides[i] = q.q_strides[i];
    q.H_q = Hq;
    q.sm_scale = a[9] == Py_None ? (float)(1.0 / std::sqrt((double)D)) : (float)PyFloat_AsDouble(a[9]);
    fq_tail tail{};
    const int has_tail = bits == 3 ? (a[11] == Py_None ? 0 : -1) : tail_of(a[11], a[12], nd, D, 1, 1, false, tail);
    if (PyErr_Occurred() || has_tail < 0) {
        PyErr_Clear();
        return none();
    }
    // more than 4 query heads per KV head: only where the library takes the step whole
    const int nrep = Hq / Hkv;
    if (nrep > 8) return none();
    if (nrep > 4 && D == 128 && page == 64) {
        if (nrep != 6 && nrep != 8) return none();
        const int whole = bits == 3 ? g_fq.fused3(&tc, &q)
                                    : (bits == 4 ? g_fq.fused4 : g_fq.fused8)(&c, &q, sinks, window, k_max, mode);
        if (whole != 1) return none();
    }
    const size_t need = bits == 3 ? g_fq.ws_turbo(&tc, Hq) : g_fq.ws_int4(&c, Hq);
    if (need > (size_t)ws->numel()) return none();
    const THPObjectPtr made(PyTuple_Check(a[3]) ? Py_NewRef(a[3]) : PyObject_CallNoArgs(a[3]));
    if (!made) return nullptr;
    const at::Tensor* ret =
        PyTuple_Check(made.get()) && PyTuple_GET_SIZE(made.get()) == 2 ? plain(PyTuple_GET_ITEM(made.get(), 0)) : nullptr;
    if (!ret) return none();
    q.retention_layer_stride = PyLong_AsLongLong(PyTuple_GET_ITEM(made.get(), 1));

    at::Tensor O = at::empty(Q->sizes(), Q->options()), lse;
    q.out = O.data_ptr();
    if (want_lse) {
        lse = at::empty(Q->sizes().slice(0, nd - 1), Q->options().dtype(at::kFloat));     // (..., H_q, 1)
        q.lse = (float*)lse.data_ptr();
        q.lse_strides[0] = nd == 5 ? (int64_t)B * Hq : 0;
        q.lse_strides[1] = Hq;
        q.lse_strides[2] = 1;
    }
    const float* r = (const float*)ret->data_ptr();
    void* w = ws->data_ptr();
    const size_t wn = (size_t)ws->numel();
    fq_stream_t st = (fq_stream_t)PyLong_AsVoidPtr(a[14]);
    int64_t s0[5], s1[5];
    if (bits == 3) {
        strides(*raw[0], s0);
        strides(*raw[1], s1);
    }
    int status;
    Py_BEGIN_ALLOW_THREADS
    if (bits == 3)
        status = g_fq.decode3(&tc, raw[0]->data_ptr(), s0, raw[1]->data_ptr(), s1, &q, r, sinks, window, k_max, mode,
                              nullptr, w, wn, st);
    else if (has_tail)
        status = (bits == 4 ? g_fq.tail4 : g_fq.tail8)(&c, &q, &tail, r, sinks, window, k_max, mode, w, wn, st);
    else
        status = (bits == 4 ? g_fq.decode4 : g_fq.decode8)(&c, &q, r, sinks, window, k_max, mode, nullptr, nullptr, w,
                                                           wn, st);
    Py_END_ALLOW_THREADS
    if (status != FQ_OK) return none();
    PyObject* lo = want_lse ? THPVariable_Wrap(std::move(lse)) : Py_NewRef(Py_None);
    return Py_BuildValue("(NN)", THPVariable_Wrap(std::move(O)), lo);
    END_HANDLE_TH_ERRORS
}

// prefill(bits, q, planes, K_tail, V_tail, page, causal_offset, sm_scale or None, stream) -> out, or None
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 9) return none();
    const int bits = (int)PyLong_AsLong(a[0]);
    const at::Tensor* Q = plain(a[1]);
    if (!Q || Q->dim() != 4 || Q->scalar_type() != at::kBFloat16 || !rows(*Q, 8) || !PyTuple_Check(a[2]) ||
        PyTuple_GET_SIZE(a[2]) != 6)
        return none();
    const at::Tensor* t[6];
    for (int i = 0; i < 6; ++i) {
        t[i] = plain(PyTuple_GET_ITEM(a[2], i));
        if (!t[i] || t[i]->device() != Q->device() || t[i]->dim() != 4) return none();
    }
    fq_int4_cache c{};
    if (!rows(*t[0], bits == 8 ? 16 : 8) || !int_cache(t, bits, (int)PyLong_AsLong(a[5]), c)) return none();
    const int64_t D = Q->size(3);
    if (c.B != Q->size(0) || c.D != D) return none();
    fq_tail tail{};
    if (tail_of(a[3], a[4], 4, D, 8, 4, true, tail) < 0) return none();
    fq_prefill p{};
    p.q = Q->data_ptr(); strides(*Q, p.q_strides);
    p.H_q = (int)Q->size(1);
    p.S_q = (int)Q->size(2);
    p.causal_offset = (int)PyLong_AsLong(a[6]);
    p.sm_scale = a[7] == Py_None ? 0.f : (float)PyFloat_AsDouble(a[7]);
    p.D = (int)D;
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return none();
    }
    at::Tensor out = at::empty(Q->sizes(), Q->options()), ws;
    p.out = out.data_ptr(); strides(out, p.o_strides);
    const size_t bytes = g_fq.ws_prefill(&c, &tail, &p, bits);
    if (bytes) ws = at::empty({(int64_t)bytes}, Q->options().dtype(at::kByte));
    void* w = bytes ? ws.data_ptr() : nullptr;
    fq_stream_t st = (fq_stream_t)PyLong_AsVoidPtr(a[8]);
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = (bits == 4 ? g_fq.prefill4 : g_fq.prefill8)(&c, &tail, &p, w, bytes, st);
    Py_END_ALLOW_THREADS
    if (status != FQ_OK) return none();
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// quantize(which (0: K, 1: V), bits, X, page or V group, metadata dtype code, stream) -> (codes, scale, min), or None
PyObject* quantize(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 6) return none();
    const bool v = PyLong_AsLong(a[0]) != 0;
    const int bits = (int)PyLong_AsLong(a[1]), meta = (int)PyLong_AsLong(a[4]);
    const int64_t unit = PyLong_AsLongLong(a[3]);
    const at::Tensor* X = plain(a[2]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        return none();
    }
    if (!X || X->dim() != 4 || unit < 1 || (meta != FQ_BF16 && meta != FQ_F16)) return none();
    const int in = dtype_code(*X);
    const int64_t B = X->size(0), H = X->size(1), S = X->size(2), D = X->size(3);
    if (in < 0 || D % 2 || (v && D % unit)) return none();
    const auto mt = X->options().dtype(meta == FQ_BF16 ? at::kBFloat16 : at::kHalf);
    at::Tensor codes = at::empty({B, H, S, bits == 8 ? D : D / 2}, X->options().dtype(at::kByte));
    at::Tensor scale = v ? at::empty({B, H, S, D / unit}, mt) : at::empty({B, H, (S + unit - 1) / unit, D}, mt);
    at::Tensor mn = at::empty(scale.sizes(), mt);
    int64_t xs[4], cs[4], ss[4], ms[4];
    strides(*X, xs); strides(codes, cs); strides(scale, ss); strides(mn, ms);
    const void* x = X->data_ptr();
    uint8_t* cp = (uint8_t*)codes.data_ptr();
    void* sp = scale.data_ptr();
    void* mp = mn.data_ptr();
    fq_stream_t st = (fq_stream_t)PyLong_AsVoidPtr(a[5]);
    const int b = (int)B, h = (int)H, s = (int)S, d = (int)D, u = (int)unit;
    int status;
    Py_BEGIN_ALLOW_THREADS
    if (!v) status = (bits == 4 ? g_fq.quant_k4 : g_fq.quant_k8)(x, in, xs, b, h, s, d, u, cp, cs, sp, ss, mp, ms, meta, st);
    else if (bits == 4) status = g_fq.quant_v4(x, in, xs, b, h, s, d, u, cp, cs, sp, ss, mp, ms, meta, st);
    else status = g_fq.quant_v8(x, in, xs, b, h, s, d, cp, cs, sp, ss, mp, ms, meta, st);
    Py_END_ALLOW_THREADS
    if (status != FQ_OK) return none();
    return Py_BuildValue("(NNN)", THPVariable_Wrap(std::move(codes)), THPVariable_Wrap(std::move(scale)),
                         THPVariable_Wrap(std::move(mn)));
    END_HANDLE_TH_ERRORS
}

// bind({entry name: address}): the library's entries; raises KeyError for a missing one.
PyObject* bind(PyObject*, PyObject* table) {
    auto get = [&](const char* name) -> void* {
        PyObject* v = PyMapping_GetItemString(table, name);
        if (!v) return nullptr;
        void* p = PyLong_AsVoidPtr(v);
        Py_DECREF(v);
        return p;
    };
    Entries e{};
#define FQ_BIND(field, name)                                                       \
    if (!(e.field = (decltype(e.field))get(#name))) {                              \
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, #name " is NULL"); \
        return nullptr;                                                            \
    }
    FQ_BIND(ws_int4, fq_workspace_bytes)
    FQ_BIND(ws_turbo, fq_turbo_workspace_bytes)
    FQ_BIND(decode4, fq_quest_decode_int4)
    FQ_BIND(decode8, fq_quest_decode_int8)
    FQ_BIND(tail4, fq_quest_decode_int4_tail)
    FQ_BIND(tail8, fq_quest_decode_int8_tail)
    FQ_BIND(decode3, fq_quest_decode_turbo)
    FQ_BIND(fused4, fq_quest_fused_int4)
    FQ_BIND(fused8, fq_quest_fused_int8)
    FQ_BIND(fused3, fq_quest_fused_turbo)
    FQ_BIND(prefill4, fq_prefill_int4)
    FQ_BIND(prefill8, fq_prefill_int8)
    FQ_BIND(ws_prefill, fq_prefill_workspace_bytes)
    FQ_BIND(quant_k4, fq_quantize_k_int4)
    FQ_BIND(quant_k8, fq_quantize_k_int8)
    FQ_BIND(quant_v4, fq_quantize_v_int4)
    FQ_BIND(quant_v8, fq_quantize_v_int8)
#undef FQ_BIND
    g_fq = e;
    Py_RETURN_NONE;
}

PyMethodDef g_methods[] = {
    {"bind", bind, METH_O, "Take the library's entry addresses."},
    {"decode", (PyCFunction)(void (*)(void))decode, METH_FASTCALL, "One decode step, or None."},
    {"prefill", (PyCFunction)(void (*)(void))prefill, METH_FASTCALL, "One prefill, or None."},
    {"quantize", (PyCFunction)(void (*)(void))quantize, METH_FASTCALL, "One quantiser call, or None."},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_fq_host", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fq_host(void) { return PyModule_Create(&g_module); }
