// host.cpp - the Python entry points' way to the C ABI in native code
// (_sqahost.so). A decode step's node took 12 us of host time per call in Python
// (a ctypes descriptor per tensor at 1.5 to 2.2 us each, the ctypes call and the
// stream lookup), more than its kernels take on the GPU at short contexts; the
// same call takes about 1 us here beside its launches.
//
// Each function takes the tensors of one entry point, with the output and the
// workspace given, and the current stream. It checks what the Python wrapper
// checks and returns the library's status; anything it does not take as it is (a
// tensor subclass, another rank or type, a stream argument, an int that is not
// an int) it answers with None before any work, and the wrapper takes its general
// path, which raises what it always raised. Nothing is kept between calls.
#include <Python.h>

#include <cmath>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../include/sqattn.h"
#include "call.hpp"

namespace {

using sqa_py::answer;
using sqa_py::General;
using sqa_py::without_gil;

const at::Tensor &tensor(PyObject *o) {
    if (!THPVariable_CheckExact(o)) throw General();
    return THPVariable_Unpack(o);
}

int64_t integer(PyObject *o) {
    if (!PyLong_CheckExact(o)) throw General();
    int over = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &over);
    if (over) throw General();
    return v;
}

double real(PyObject *o);

// the softmax scale, or head dim ** -0.5 for None
float scale_of(PyObject *o, const at::Tensor &q) {
    return (float)(o == Py_None ? std::pow((double)q.size(2), -0.5) : real(o));
}

double real(PyObject *o) {
    if (!PyFloat_CheckExact(o)) throw General();
    return PyFloat_AS_DOUBLE(o);
}

void need(bool ok) {
    if (!ok) throw General();
}

sqa_tensor make(int type, const at::Tensor &t, int64_t ne0, int64_t ne1, int64_t ne2, int64_t nb0, int64_t nb1,
                int64_t nb2, int64_t nb3) {
    sqa_tensor d{};
    d.type = type;
    d.ne[0] = ne0, d.ne[1] = ne1, d.ne[2] = ne2, d.ne[3] = 1;
    d.nb[0] = (uint64_t)nb0, d.nb[1] = (uint64_t)nb1, d.nb[2] = (uint64_t)nb2, d.nb[3] = (uint64_t)nb3;
    d.data = t.data_ptr();
    return d;
}

// (n0, n1) rows of 4-byte values, the row stride as it is
sqa_tensor rows2(const at::Tensor &t, int64_t n0, int64_t n1) {
    const int64_t s = t.stride(0) * 4;
    return make(SQA_TYPE_F32, t, n0, n1, 1, 4, s, s * n1, s * n1);
}

sqa_tensor cache_rows(const at::Tensor &c, int64_t ne0) {
    need(c.dim() >= 1 && c.size(0) > 0);
    const int64_t rows = c.size(0), rb = c.numel() / rows;
    need(rb == ne0 / SQA_QK4_0 * SQA_Q4_0_BLOCK_BYTES);
    return make(SQA_TYPE_Q4_0, c, ne0, rows, 1, SQA_Q4_0_BLOCK_BYTES, rb, rb * rows, rb * rows);
}

sqa_tensor index(const at::Tensor &t, int type, int64_t nb0) {
    need(t.dim() >= 1);
    const int64_t n = t.size(0);
    return make(type, t, n, 1, 1, nb0, nb0 * n, nb0 * n, nb0 * n);
}

sqa_tensor q_view(const at::Tensor &q) {  // (n_q, H, D) -> [D, n_q, H]
    need(q.dim() == 3);
    return make(SQA_TYPE_F32, q, q.size(2), q.size(0), q.size(1), 4, q.stride(0) * 4, q.stride(1) * 4,
                q.stride(1) * 4 * q.size(1));
}

sqa_tensor cache_view(const at::Tensor &c, int64_t n_kv) {  // (rows, Hkv, bytes) -> [D, n_kv, Hkv]
    need(c.dim() == 3 && c.scalar_type() == at::kByte && c.is_contiguous() && n_kv <= c.size(0));
    const int64_t Hkv = c.size(1), rb = c.size(2);
    return make(SQA_TYPE_Q4_0, c, rb / SQA_Q4_0_BLOCK_BYTES * SQA_QK4_0, n_kv, Hkv, SQA_Q4_0_BLOCK_BYTES, Hkv * rb, rb,
                rb * Hkv);
}

sqa_tensor out_view(const at::Tensor &o) {  // (n_q, H, D) -> [D, H, n_q]
    need(o.dim() == 3 && o.is_contiguous());
    const int64_t n_q = o.size(0), H = o.size(1), D = o.size(2);
    return make(SQA_TYPE_F32, o, D, H, n_q, 4, D * 4, H * D * 4, H * D * 4 * n_q);
}

sqa_tensor mask_view(const at::Tensor &m) {
    need(m.dim() == 2 && m.scalar_type() == at::kHalf && m.stride(1) == 1);
    const int64_t s = m.stride(0) * 2;
    return make(SQA_TYPE_F16, m, m.size(1), m.size(0), 1, 2, s, s * m.size(0), s * m.size(0));
}

void *stream() { return c10::hip::getCurrentHIPStream().stream(); }

// q, k_cache, v_cache, n_kv, mask, scale, max_bias, softcap, out, workspace
PyObject *fa(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return answer([&]() -> int {
        need(n == 10);
        const at::Tensor &q = tensor(a[0]), &ws = tensor(a[9]);
        const int64_t n_kv = integer(a[3]);
        const sqa_tensor tq = q_view(q), tk = cache_view(tensor(a[1]), n_kv), tv = cache_view(tensor(a[2]), n_kv),
                         to = out_view(tensor(a[8]));
        sqa_tensor tm;
        const bool mask = a[4] != Py_None;
        if (mask) tm = mask_view(tensor(a[4]));
        const float scale = scale_of(a[5], q), bias = (float)real(a[6]), cap = (float)real(a[7]);
        void *wp = ws.data_ptr(), *st = stream();
        const size_t wb = (size_t)ws.numel();
        return without_gil([&] {
            return sqa_flash_attn_ext(&tq, &tk, &tv, mask ? &tm : nullptr, scale, bias, cap, &to, wp, wb, st);
        });
    });
}

// q, k_cache, v_cache, n_kv, q_pos0, gate, scale, out, workspace
PyObject *fa_causal(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return answer([&]() -> int {
        need(n == 9);
        const at::Tensor &q = tensor(a[0]), &ws = tensor(a[8]);
        const int64_t n_kv = integer(a[3]), pos0 = integer(a[4]);
        const sqa_tensor tq = q_view(q), tk = cache_view(tensor(a[1]), n_kv), tv = cache_view(tensor(a[2]), n_kv),
                         to = out_view(tensor(a[7]));
        sqa_tensor tg;
        const bool gate = a[5] != Py_None;
        if (gate) {
            const at::Tensor &t = tensor(a[5]);
            need(t.dim() >= 2);
            tg = make(SQA_TYPE_F32, t, q.size(2), q.size(1), q.size(0), 4, t.stride(1) * 4, t.stride(0) * 4,
                      t.stride(0) * 4 * q.size(0));
        }
        const float scale = scale_of(a[6], q);
        void *wp = ws.data_ptr(), *st = stream();
        const size_t wb = (size_t)ws.numel();
        return without_gil([&] {
            return sqa_flash_attn_ext_causal(&tq, &tk, &tv, pos0, gate ? &tg : nullptr, scale, &to, wp, wb, st);
        });
    });
}

// mask, step_start
PyObject *fill_mask(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return answer([&]() -> int {
        need(n == 2);
        const sqa_tensor tm = mask_view(tensor(a[0]));
        const int64_t start = integer(a[1]);
        void *st = stream();
        return without_gil([&] { return sqa_fill_causal_mask(&tm, start, st); });
    });
}

// cache, src, idx
PyObject *set_rows(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return answer([&]() -> int {
        need(n == 3);
        const at::Tensor &src = tensor(a[1]), &idx = tensor(a[2]);
        need(src.dim() == 2 && idx.dim() >= 1);
        const int64_t ne0 = src.size(1);
        const sqa_tensor td = cache_rows(tensor(a[0]), ne0), ts = rows2(src, ne0, src.size(0)),
                         ti = index(idx, SQA_TYPE_I64, idx.stride(0) * 8);
        void *st = stream();
        return without_gil([&] { return sqa_set_rows_q4_0(&td, &ts, &ti, st); });
    });
}

// cache or out, src, norm_w, eps, pos, rope, idx (None: F32 output)
PyObject *rope_norm(PyObject *, PyObject *const *a, Py_ssize_t n) {
    Py_buffer view{};
    PyObject *r = answer([&]() -> int {
        need(n == 7);
        const at::Tensor &dst = tensor(a[0]), &src = tensor(a[1]), &pos = tensor(a[4]);
        need(src.dim() == 3);
        const int64_t n_tok = src.size(0), n_head = src.size(1), D = src.size(2);
        const sqa_tensor ts = make(SQA_TYPE_F32, src, D, n_head, n_tok, 4, src.stride(1) * 4, src.stride(0) * 4,
                                   src.stride(0) * 4 * n_tok),
                         tp = index(pos, SQA_TYPE_I32, 4);
        sqa_tensor tw;
        const bool norm = a[2] != Py_None;
        if (norm) tw = make(SQA_TYPE_F32, tensor(a[2]), D, 1, 1, 4, 4 * D, 4 * D, 4 * D);
        const float eps = (float)real(a[3]);
        need(PyObject_GetBuffer(a[5], &view, PyBUF_SIMPLE) == 0 && view.len == (Py_ssize_t)sizeof(sqa_rope));
        const sqa_rope *rope = (const sqa_rope *)view.buf;
        void *st = stream();
        if (a[6] == Py_None) {
            const sqa_tensor to = make(SQA_TYPE_F32, dst, D, n_head, n_tok, 4, D * 4, n_head * D * 4, n_head * D * 4 * n_tok);
            return without_gil([&] { return sqa_rope_norm_f32(&to, &ts, norm ? &tw : nullptr, eps, &tp, rope, st); });
        }
        const at::Tensor &idx = tensor(a[6]);
        need(idx.dim() >= 1);
        const sqa_tensor td = cache_rows(dst, n_head * D), ti = index(idx, SQA_TYPE_I64, idx.stride(0) * 8);
        return without_gil([&] {
            return sqa_rope_norm_set_rows_q4_0(&td, &ts, norm ? &tw : nullptr, eps, &tp, rope, &ti, st);
        });
    });
    if (view.obj) PyBuffer_Release(&view);
    return r;
}

// w, x, gate, out, workspace
PyObject *out_proj(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return answer([&]() -> int {
        need(n == 5);
        const at::Tensor &w = tensor(a[0]), &x = tensor(a[1]), &o = tensor(a[3]), &ws = tensor(a[4]);
        need(x.dim() == 2 && w.dim() >= 1 && o.dim() >= 1);
        const int64_t M = x.size(0), K = x.size(1), N = w.size(0), wn = w.stride(0);
        const sqa_tensor tw = make(SQA_TYPE_Q4_K, w, K, N, 1, 144, wn, wn * N, wn * N), tx = rows2(x, K, M),
                         to = rows2(o, N, M);
        sqa_tensor tg;
        const bool gate = a[2] != Py_None;
        if (gate) {
            need(tensor(a[2]).dim() >= 1);
            tg = rows2(tensor(a[2]), K, M);
        }
        void *wp = ws.data_ptr(), *st = stream();
        const size_t wb = (size_t)ws.numel();
        return without_gil([&] { return sqa_out_proj(&tw, &tx, gate ? &tg : nullptr, &to, wp, wb, st); });
    });
}

// handle, slot, k_cur, v_cur, idx
PyObject *append(PyObject *, PyObject *const *a, Py_ssize_t n) {
    return answer([&]() -> int {
        need(n == 5);
        sqa_kv_cache *kv = (sqa_kv_cache *)(uintptr_t)integer(a[0]);
        const int64_t slot = integer(a[1]);
        need(slot == (int64_t)(int32_t)slot);
        const at::Tensor &k = tensor(a[2]), &v = tensor(a[3]);
        need(k.dim() == 2 && v.dim() >= 1);
        const int64_t n_tok = k.size(0), ne0 = k.size(1);
        const sqa_tensor tk = rows2(k, ne0, n_tok), tv = rows2(v, ne0, n_tok),
                         ti = make(SQA_TYPE_I64, tensor(a[4]), n_tok, 1, 1, 8, 8 * n_tok, 8 * n_tok, 8 * n_tok);
        void *st = stream();
        return without_gil([&] { return sqa_kv_cache_append(kv, (int32_t)slot, &tk, &tv, &ti, st); });
    });
}

PyMethodDef methods[] = {
#define SQA_FN(f) {#f, (PyCFunction)(void (*)(void))f, METH_FASTCALL, nullptr}
    SQA_FN(fa),        SQA_FN(fa_causal), SQA_FN(fill_mask), SQA_FN(set_rows),
    SQA_FN(rope_norm), SQA_FN(out_proj),  SQA_FN(append),    {nullptr, nullptr, 0, nullptr},
#undef SQA_FN
};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sqahost", nullptr, -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__sqahost() { return PyModule_Create(&module); }
