// The per-call host path of the operators that a generated token runs through: argument checks, output and workspace tensors, the
// stream and the library call in one native function each.
//
// Bound: a decode launch lasts 5 - 13 us, so the host has to be through a call in less.  The same steps written in Python (checks
// 1.4 us, two tensors 2.8, stream and device 2.5, the ctypes call 3.8 of which 3.6 are the launch itself) came to 13.2 us a call; here
// 5.6 us (Q4_K 5120x5120, one row, back to back: 14.1 -> 5.8 us a call; a MiniMax-M2 layer's token 121 -> 55 us).
//
// Every function serves the plain case only - exact torch tensors on the current device, everything contiguous and of the expected
// types and sizes - and returns None for anything else without having done anything: the Python wrapper (hip_kernel.py) then runs its own
// checks, which state each error, and its own call.  A library status other than success raises RuntimeError with the wrapper's text.
// The interpreter lock is released while the library enqueues its kernels: everything that may throw (pointers, stream) is taken before.
#include <Python.h>

#include <ATen/core/Tensor.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <vector>

#include "../../include/pllm_hip.h"

namespace {

using at::Tensor;

// a borrowed plain tensor, or nullptr
const Tensor* tensor(PyObject* o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }
// a strided tensor that owns memory, all of it in order (the wrapper tensors of vmap, jvp and grad look like plain tensors and own none: the
// Python path states the error)
bool dense(const Tensor* t) { return t && t->layout() == at::kStrided && t->has_storage() && t->is_contiguous(); }
bool plain(const Tensor* t) { return dense(t) && t->is_cuda(); }
bool plain(const Tensor* t, at::ScalarType st) { return plain(t) && t->scalar_type() == st; }
bool here(const Tensor* t) { return t->get_device() == c10::hip::current_device(); }

int code_of(at::ScalarType st) { return st == at::kFloat ? PLLM_F32 : (st == at::kHalf ? PLLM_F16 : (st == at::kBFloat16 ? PLLM_BF16 : -1)); }
bool dtype_arg(PyObject* o, at::ScalarType& out) {
    if (!THPDtype_Check(o)) return false;
    out = reinterpret_cast<THPDtype*>(o)->scalar_type;
    return code_of(out) >= 0;
}
bool int_arg(PyObject* o, int64_t& v) {
    if (!PyLong_CheckExact(o)) return false;
    int overflow = 0;
    v = PyLong_AsLongLongAndOverflow(o, &overflow);
    return overflow == 0;
}
bool float_arg(PyObject* o, float& v) {
    if (!PyFloat_CheckExact(o)) return false;
    v = static_cast<float>(PyFloat_AS_DOUBLE(o));
    return true;
}
// the codebook tensor that a type asks for (hip_kernel.py: _check_grid); the table-free types take anything
bool grid_ok(PyObject* o, int64_t type_id) {
    if (type_id != PLLM_TYPE_IQ2_XXS && type_id != PLLM_TYPE_IQ1_M && type_id != PLLM_TYPE_IQ2_XS && type_id != PLLM_TYPE_IQ3_XXS) return true;
    const Tensor* g = tensor(o);
    if (!plain(g, at::kChar)) return false;
    if (type_id == PLLM_TYPE_IQ2_XXS) return g->numel() == 256 * 128 * 8;
    if (type_id == PLLM_TYPE_IQ1_M) return g->numel() == 2048 * 8;
    return g->numel() >= 512 * 128 * 8 + 256 * 128 * 8;
}

void* stream_of(const Tensor& t) { return c10::hip::getCurrentHIPStream(t.get_device()).stream(); }
Tensor like_rows(const Tensor& x, int64_t n, at::ScalarType st) {         // x's leading shape, n columns
    c10::SmallVector<int64_t, 5> shape(x.sizes().begin(), x.sizes().end());
    shape.back() = n;
    return at::empty(shape, x.options().dtype(st));
}
Tensor workspace(const Tensor& x, size_t bytes) { return at::empty({static_cast<int64_t>(std::max<size_t>(bytes, 1))}, x.options().dtype(at::kByte)); }

// a library call without the interpreter lock; its arguments are formed, and may throw, while the lock is still held
template <typename T> struct AsDeclared { using type = T; };
template <typename... P> int unlocked(int (*call)(P...), typename AsDeclared<P>::type... args) {
    struct Released {
        PyThreadState* state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
    } released;
    return call(args...);
}

PyObject* failed(PyObject* name, int status) {
    return PyErr_Format(PyExc_RuntimeError, "%S: %s (status %d)", name, pllm_status_string(status), status);
}

struct Dense {
    const Tensor *x = nullptr, *blocks = nullptr;
    int64_t k = 0, type_id = 0, rows = 0, n = 0, bpr = 0;
    int x_code = -1;
};
// x [M, K] or [B, S, K] against raw blocks [N, K / 256, block bytes]
bool dense_args(PyObject* x, PyObject* blocks, PyObject* row_elems, PyObject* type_id, PyObject* grid, Dense& d) {
    d.x = tensor(x);
    d.blocks = tensor(blocks);
    if (!plain(d.x) || !plain(d.blocks, at::kByte) || !int_arg(row_elems, d.k) || !int_arg(type_id, d.type_id) || !here(d.x)) return false;
    if ((d.x->dim() != 2 && d.x->dim() != 3) || d.blocks->dim() != 3 || d.k <= 0 || d.type_id < 0 || d.type_id > PLLM_TYPE_Q6_K) return false;
    d.n = d.blocks->size(0);
    d.bpr = d.blocks->size(1);
    d.x_code = code_of(d.x->scalar_type());
    if (d.x_code < 0 || d.x->size(-1) != d.k || d.bpr * 256 < d.k || d.blocks->size(2) != pllm_gguf_block_bytes(static_cast<int>(d.type_id))) return false;
    d.rows = d.x->numel() / d.k;
    return d.rows > 0 && d.n > 0 && grid_ok(grid, d.type_id);
}

// (name, x, blocks, row_elems, type_id, grid, out_dtype) -> y
PyObject* quant_gemm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Dense d;
    at::ScalarType out;
    if (nargs != 7 || !dense_args(a[1], a[2], a[3], a[4], a[5], d) || !dtype_arg(a[6], out)) Py_RETURN_NONE;
    const int type_id = static_cast<int>(d.type_id);
    Tensor y = like_rows(*d.x, d.n, out);
    const size_t bytes = pllm_gguf_quant_gemm_workspace_bytes(type_id, d.rows, d.k, d.n, d.bpr);
    Tensor ws = workspace(*d.x, bytes);
    const int st = unlocked(pllm_gguf_quant_gemm, d.x->const_data_ptr(), d.x_code, static_cast<const uint8_t*>(d.blocks->const_data_ptr()), type_id,
                            y.data_ptr(), code_of(out), d.rows, d.k, d.n, d.bpr, ws.data_ptr(), bytes, stream_of(*d.x));
    return st == PLLM_OK ? THPVariable_Wrap(std::move(y)) : failed(a[0], st);
    END_HANDLE_TH_ERRORS
}

// (name, x, blocks, row_elems, type_id, grid, y) -> True; None also where the library has no such launch
PyObject* quant_gemm_accumulate(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    Dense d;
    if (nargs != 7 || !dense_args(a[1], a[2], a[3], a[4], a[5], d)) Py_RETURN_NONE;
    const Tensor* y = tensor(a[6]);
    if (!plain(y) || code_of(y->scalar_type()) < 0 || y->get_device() != d.x->get_device() || y->dim() != d.x->dim() || y->size(-1) != d.n ||
        !std::equal(y->sizes().begin(), y->sizes().end() - 1, d.x->sizes().begin()))
        Py_RETURN_NONE;
    const int type_id = static_cast<int>(d.type_id);
    const size_t bytes = pllm_gguf_quant_gemm_workspace_bytes(type_id, d.rows, d.k, d.n, d.bpr);
    Tensor ws = workspace(*d.x, bytes);
    const int st = unlocked(pllm_gguf_quant_gemm_accumulate, d.x->const_data_ptr(), d.x_code, static_cast<const uint8_t*>(d.blocks->const_data_ptr()), type_id,
                            y->data_ptr(), code_of(y->scalar_type()), d.rows, d.k, d.n, d.bpr, ws.data_ptr(), bytes, stream_of(*d.x));
    if (st == PLLM_ERR_UNSUPPORTED) Py_RETURN_NONE;
    if (st != PLLM_OK) return failed(a[0], st);
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// (name, x, [blocks], row_elems, type_id, grid, norm_weight or None, eps, round_fp16, out_dtype) -> [y]; None also where the library has no
// such launch
PyObject* quant_gemm_multi(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    at::ScalarType out;
    float eps;
    if (nargs != 10 || !PyList_CheckExact(a[2]) || !float_arg(a[7], eps) || !PyBool_Check(a[8]) || !dtype_arg(a[9], out)) Py_RETURN_NONE;
    const Py_ssize_t count = PyList_GET_SIZE(a[2]);
    if (count < 1 || count > 4) Py_RETURN_NONE;
    Dense d[4];
    const uint8_t* blocks[4];
    int64_t heights[4];
    for (Py_ssize_t i = 0; i < count; ++i) {
        if (!dense_args(a[1], PyList_GET_ITEM(a[2], i), a[3], a[4], a[5], d[i]) || d[i].bpr != d[0].bpr) Py_RETURN_NONE;
        blocks[i] = static_cast<const uint8_t*>(d[i].blocks->const_data_ptr());
        heights[i] = d[i].n;
    }
    const float* norm = nullptr;
    if (a[6] != Py_None) {
        const Tensor* w = tensor(a[6]);
        if (!plain(w, at::kFloat) || w->dim() != 1 || w->size(0) != d[0].k) Py_RETURN_NONE;
        norm = w->const_data_ptr<float>();
    }
    Tensor y[4];
    void* ys[4];
    for (Py_ssize_t i = 0; i < count; ++i) {
        y[i] = like_rows(*d[0].x, d[i].n, out);
        ys[i] = y[i].data_ptr();
    }
    const size_t bytes = pllm_gguf_quant_gemm_multi_workspace_bytes(static_cast<int>(d[0].type_id), static_cast<int>(count), heights, d[0].rows, d[0].bpr);
    Tensor ws = workspace(*d[0].x, bytes);
    const int st = unlocked(pllm_gguf_quant_gemm_multi, d[0].x->const_data_ptr(), d[0].x_code, norm, eps, a[8] == Py_True, static_cast<int>(count), blocks,
                            heights, static_cast<int>(d[0].type_id), ys, code_of(out), d[0].rows, d[0].k, d[0].bpr, ws.data_ptr(), bytes, stream_of(*d[0].x));
    if (st == PLLM_ERR_UNSUPPORTED) Py_RETURN_NONE;
    if (st != PLLM_OK) return failed(a[0], st);
    PyObject* list = PyList_New(count);
    for (Py_ssize_t i = 0; list && i < count; ++i) PyList_SET_ITEM(list, i, THPVariable_Wrap(std::move(y[i])));
    return list;
    END_HANDLE_TH_ERRORS
}

// (name, x, blocks, row_elems, out_dtype) -> y
PyObject* q8_0_gemm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    at::ScalarType out;
    int64_t k;
    if (nargs != 5) Py_RETURN_NONE;
    const Tensor *x = tensor(a[1]), *b = tensor(a[2]);
    if (!plain(x) || !plain(b, at::kByte) || !int_arg(a[3], k) || !dtype_arg(a[4], out) || !here(x)) Py_RETURN_NONE;
    const int x_code = code_of(x->scalar_type());
    if (x_code < 0 || (x->dim() != 2 && x->dim() != 3) || b->dim() != 3 || b->size(2) != 34 || k <= 0 || x->size(-1) != k || b->size(1) * 32 < k) Py_RETURN_NONE;
    const int64_t rows = x->numel() / k, n = b->size(0), bpr = b->size(1);
    if (rows == 0 || n == 0) Py_RETURN_NONE;
    Tensor y = like_rows(*x, n, out);
    const size_t bytes = pllm_q8_0_gemm_workspace_bytes(rows, k, n, bpr);
    Tensor ws = workspace(*x, bytes);
    const int st = unlocked(pllm_q8_0_gemm, x->const_data_ptr(), x_code, static_cast<const uint8_t*>(b->const_data_ptr()), y.data_ptr(), code_of(out), rows, k,
                            n, bpr, ws.data_ptr(), bytes, stream_of(*x));
    return st == PLLM_OK ? THPVariable_Wrap(std::move(y)) : failed(a[0], st);
    END_HANDLE_TH_ERRORS
}

bool fp8_bytes(const Tensor* w) { return plain(w) && (w->scalar_type() == at::kFloat8_e4m3fn || w->scalar_type() == at::kByte); }
bool fp8_scales(const Tensor* s, int64_t n, int64_t k) {
    return plain(s, at::kFloat) && s->dim() == 2 && s->size(0) == (n + 127) / 128 && s->size(1) == (k + 127) / 128;
}

// (name, x, weight, scale, out_dtype) -> y
PyObject* fp8_block_gemm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    at::ScalarType out;
    if (nargs != 5) Py_RETURN_NONE;
    const Tensor *x = tensor(a[1]), *w = tensor(a[2]), *s = tensor(a[3]);
    if (!plain(x) || !fp8_bytes(w) || !dtype_arg(a[4], out) || !here(x) || w->dim() != 2 || x->dim() < 1) Py_RETURN_NONE;
    const int x_code = code_of(x->scalar_type());
    const int64_t n = w->size(0), k = w->size(1);
    if (x_code < 0 || k <= 0 || n <= 0 || x->size(-1) != k || !fp8_scales(s, n, k) || x->numel() == 0) Py_RETURN_NONE;
    const int64_t rows = x->numel() / k;
    Tensor y = like_rows(*x, n, out), ws;
    const size_t bytes = pllm_fp8_block_gemm_workspace_bytes(rows, k, n);
    if (bytes) ws = workspace(*x, bytes);
    const int st = unlocked(pllm_fp8_block_gemm, x->const_data_ptr(), x_code, static_cast<const uint8_t*>(w->const_data_ptr()), s->const_data_ptr<float>(),
                            y.data_ptr(), code_of(out), rows, k, n, bytes ? ws.data_ptr() : nullptr, bytes, stream_of(*x));
    return st == PLLM_OK ? THPVariable_Wrap(std::move(y)) : failed(a[0], st);
    END_HANDLE_TH_ERRORS
}

// (name, q, k_new, v_new, keys, values, pos, q_norm_weight or None, k_norm_weight or None, eps, cos_row or None, sin_row or None, rope_dim) -> out
PyObject* attention_decode(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 13) Py_RETURN_NONE;
    int64_t pos, rope;
    float eps;
    const Tensor *q = tensor(a[1]), *kn = tensor(a[2]), *vn = tensor(a[3]), *ks = tensor(a[4]), *vs = tensor(a[5]);
    if (!plain(q) || !here(q) || (q->scalar_type() != at::kHalf && q->scalar_type() != at::kBFloat16)) Py_RETURN_NONE;
    const at::ScalarType st16 = q->scalar_type();
    if (!plain(kn, st16) || !plain(vn, st16) || !plain(ks, st16) || !plain(vs, st16) || !int_arg(a[6], pos) || !float_arg(a[9], eps) || !int_arg(a[12], rope)) Py_RETURN_NONE;
    if (q->dim() != 2 || kn->dim() != 2 || vn->dim() != 2 || ks->dim() != 4 || vs->sizes() != ks->sizes()) Py_RETURN_NONE;
    const int64_t batch = q->size(0), kv_heads = ks->size(1), capacity = ks->size(2), dim = ks->size(3);
    if (batch <= 0 || dim <= 0 || pos < 0 || pos >= capacity || ks->size(0) < batch || q->size(1) % dim || kn->size(0) != batch || kn->size(1) != kv_heads * dim ||
        vn->sizes() != kn->sizes())
        Py_RETURN_NONE;
    const int64_t heads = q->size(1) / dim;
    auto row = [&](PyObject* o, int64_t width, const float*& p) {
        p = nullptr;
        if (o == Py_None) return true;
        const Tensor* t = tensor(o);
        if (!plain(t, at::kFloat) || t->numel() != width) return false;
        p = t->const_data_ptr<float>();
        return true;
    };
    const float *qw, *kw, *cos_row = nullptr, *sin_row = nullptr;
    if (!row(a[7], heads * dim, qw) || !row(a[8], kv_heads * dim, kw)) Py_RETURN_NONE;
    if (rope != 0 && (!row(a[10], dim, cos_row) || !row(a[11], dim, sin_row) || !cos_row || !sin_row)) Py_RETURN_NONE;
    Tensor out = at::empty(q->sizes(), q->options());
    const size_t bytes = pllm_attention_decode_workspace_bytes(batch, heads, pos);
    Tensor ws = workspace(*q, bytes);
    const int st = unlocked(pllm_attention_decode, q->const_data_ptr(), kn->const_data_ptr(), vn->const_data_ptr(), code_of(st16), qw, kw, eps, cos_row, sin_row,
                            rope, ks->data_ptr(), vs->data_ptr(), ks->stride(0), ks->stride(1), batch, heads, kv_heads, dim, pos, out.data_ptr(), ws.data_ptr(),
                            bytes, stream_of(*q));
    return st == PLLM_OK ? THPVariable_Wrap(std::move(out)) : failed(a[0], st);
    END_HANDLE_TH_ERRORS
}

// (name, x, norm_weight, eps, gate_weight, gate_bias or None, top_k, softmax, out_dtype) -> (indices, weights, normalized rows); None also where
// the library has no such launch
PyObject* route_rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    at::ScalarType out;
    float eps;
    int64_t top_k;
    if (nargs != 9) Py_RETURN_NONE;
    const Tensor *x = tensor(a[1]), *nw = tensor(a[2]), *gw = tensor(a[4]);
    if (!plain(x) || !here(x) || !plain(nw, at::kFloat) || !plain(gw, at::kFloat) || !float_arg(a[3], eps) || !int_arg(a[6], top_k) || !PyBool_Check(a[7]) ||
        !dtype_arg(a[8], out))
        Py_RETURN_NONE;
    const int x_code = code_of(x->scalar_type());
    if (x_code < 0 || x->dim() != 2 || gw->dim() != 2 || x->size(1) != gw->size(1) || nw->numel() != x->size(1)) Py_RETURN_NONE;
    const int64_t t = x->size(0), e = gw->size(0), dim = x->size(1);
    if (t < 1 || t > 4 || dim < 1 || top_k < 1 || top_k > e) Py_RETURN_NONE;
    const float* bias = nullptr;
    if (a[5] != Py_None) {
        const Tensor* b = tensor(a[5]);
        if (!plain(b, at::kFloat) || b->numel() != e) Py_RETURN_NONE;
        bias = b->const_data_ptr<float>();
    }
    Tensor indices = at::empty({t, top_k}, x->options().dtype(at::kLong)), weights = at::empty({t, top_k}, x->options().dtype(at::kFloat));
    Tensor logits = at::empty({t, e}, x->options().dtype(at::kFloat)), normed = at::empty({t, dim}, x->options().dtype(out));
    const int st = unlocked(pllm_moe_route_rmsnorm, x->const_data_ptr(), x_code, nw->const_data_ptr<float>(), eps, normed.data_ptr(), code_of(out), t, dim,
                            gw->const_data_ptr<float>(), bias, e, top_k, a[7] == Py_True, logits.data_ptr<float>(), indices.data_ptr<int64_t>(),
                            weights.data_ptr<float>(), stream_of(*x));
    if (st == PLLM_ERR_UNSUPPORTED) Py_RETURN_NONE;
    if (st != PLLM_OK) return failed(a[0], st);
    PyObject* r = PyTuple_New(3);
    if (!r) return nullptr;
    PyTuple_SET_ITEM(r, 0, THPVariable_Wrap(std::move(indices)));
    PyTuple_SET_ITEM(r, 1, THPVariable_Wrap(std::move(weights)));
    PyTuple_SET_ITEM(r, 2, THPVariable_Wrap(std::move(normed)));
    return r;
    END_HANDLE_TH_ERRORS
}

int type_of_block_bytes(int64_t bytes) {
    for (int t = 0; t <= PLLM_TYPE_Q6_K; ++t)
        if (pllm_gguf_block_bytes(t) == bytes) return t;
    return -1;
}

// (name, x [1, D], route_slots, route_weights, w1, w3, w2, swiglu_limit, y or None) -> the routed experts' sum as float32 [1, D] (y None), or True
// with the sum added into y; None also where the library has no launch that adds
PyObject* moe_single_token(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    float limit;
    if (nargs != 9) Py_RETURN_NONE;
    const Tensor *x = tensor(a[1]), *slots = tensor(a[2]), *rw = tensor(a[3]), *w1 = tensor(a[4]), *w3 = tensor(a[5]), *w2 = tensor(a[6]);
    if (!plain(x) || !here(x) || !plain(slots, at::kLong) || !plain(rw, at::kFloat) || !plain(w1, at::kByte) || !plain(w3, at::kByte) || !plain(w2, at::kByte) ||
        !float_arg(a[7], limit))
        Py_RETURN_NONE;
    const int x_code = code_of(x->scalar_type());
    if (x_code < 0 || x->dim() != 2 || x->size(0) != 1 || slots->dim() != 1 || rw->dim() != 1 || slots->size(0) != rw->size(0) || slots->size(0) < 1 || w1->dim() != 4 ||
        w3->dim() != 4 || w2->dim() != 4 || w1->sizes() != w3->sizes() || w1->size(0) != w2->size(0))
        Py_RETURN_NONE;
    const int64_t dim = x->size(1), inter = w1->size(1), routes = rw->size(0), experts = w1->size(0);
    const int t13 = type_of_block_bytes(w1->size(3)), t2 = type_of_block_bytes(w2->size(3));
    if (t13 < 0 || t2 < 0 || dim < 1 || inter < 1 || w1->size(2) * 256 < dim || w2->size(1) != dim || w2->size(2) * 256 < inter) Py_RETURN_NONE;
    const uint8_t *p1 = static_cast<const uint8_t*>(w1->const_data_ptr()), *p3 = static_cast<const uint8_t*>(w3->const_data_ptr()),
                  *p2 = static_cast<const uint8_t*>(w2->const_data_ptr());
    Tensor out;
    const Tensor* y = nullptr;
    if (a[8] != Py_None) {
        y = tensor(a[8]);
        if (!plain(y) || y->numel() != dim || code_of(y->scalar_type()) < 0) Py_RETURN_NONE;
    } else {
        out = at::empty({1, dim}, x->options().dtype(at::kFloat));
    }
    const size_t bytes = pllm_gguf_moe_workspace_bytes(1, routes, dim, inter);
    Tensor ws = workspace(*x, bytes);
    const int st =
        y ? unlocked(pllm_gguf_moe_single_token_accumulate, x->const_data_ptr(), x_code, dim, inter, slots->const_data_ptr<int64_t>(), rw->const_data_ptr<float>(), routes, p1, p3,
                     t13, p2, t2, limit, y->data_ptr(), code_of(y->scalar_type()), ws.data_ptr(), bytes, stream_of(*x))
          : unlocked(pllm_gguf_moe_forward, x->const_data_ptr(), x_code, 1, dim, inter, nullptr, slots->const_data_ptr<int64_t>(), nullptr, experts, rw->const_data_ptr<float>(),
                     routes, p1, p3, t13, p2, t2, limit, out.data_ptr<float>(), ws.data_ptr(), bytes, stream_of(*x));
    if (y && st == PLLM_ERR_UNSUPPORTED) Py_RETURN_NONE;
    if (st != PLLM_OK) return failed(a[0], st);
    if (y) Py_RETURN_TRUE;
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// (tensor) -> whether the functions above may read its memory as it lies (the device aside)
PyObject* dense_tensor(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    return PyBool_FromLong(nargs == 1 && dense(tensor(a[0])));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
#define PLLM_FN(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(name)), METH_FASTCALL, nullptr}
    PLLM_FN(quant_gemm), PLLM_FN(quant_gemm_accumulate), PLLM_FN(quant_gemm_multi), PLLM_FN(q8_0_gemm), PLLM_FN(fp8_block_gemm),
    PLLM_FN(attention_decode), PLLM_FN(route_rmsnorm), PLLM_FN(moe_single_token), PLLM_FN(dense_tensor),
#undef PLLM_FN
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_bindings", "Native host path of the per-token operators.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__bindings() { return PyModule_Create(&module_def); }
