// The operator calls of ops.py in native code: argument checks, the argument structs of the C ABI, output allocation and the
// call itself. In Python one call cost 20 to 25 us of host time (attribute access on tensors, ctypes structs), more than the
// GPU takes for a block of the U-Net's deeper levels; here it is 3 to 8, most of it the launches.
//
// Every function returns None, having launched nothing, when a call is not plainly valid (wrong shape, dtype, device, layout, an
// argument of another type): the Python implementation then runs, whose checks word the error. So all checks of a call come
// before its first launch, and what is taken here must be what the Python code takes (tests/test_native_calls_gpu.py makes the
// same calls both ways). The library's own refusals (return value -1) are raised here.
//
// The library is not linked but bound to at import (bind): the ctypes layer and this module use the same loaded copy.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <ATen/ops/empty_like.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstring>
#include <initializer_list>
#include <string>

#include "mi_attention.h"

namespace {

using at::Tensor;

struct Lib {
    decltype(&mi_last_error) last_error;
    decltype(&mi_sdpa_forward) sdpa;
    decltype(&mi_sdpa_split_scratch_bytes) sdpa_split_bytes;
    decltype(&mi_rope_apply) rope;
    decltype(&mi_headnorm_rope) headnorm_rope;
    decltype(&mi_linear_forward) linear;
    decltype(&mi_linear_forward_n) linear_n;
    decltype(&mi_linear_geglu_forward) geglu;
    decltype(&mi_add_inplace) add_inplace;
    decltype(&mi_rms_norm_forward) rms_norm;
    decltype(&mi_rms_norm_pair_forward) rms_norm_pair;
    decltype(&mi_attn_block_scratch_bytes) block_scratch_bytes;
    decltype(&mi_flash_attention_qkvo_forward) qkvo;
    decltype(&mi_flash_attention_q_with_kv_cached_forward) kv_cached;
    decltype(&mi_linear_attn_workspace_bytes) la_workspace_bytes;
    decltype(&mi_linear_attn_scratch_bytes) la_scratch_bytes;
    decltype(&mi_linear_attn_relu_forward) linear_attn;
} L;
bool bound = false;

// ── reading arguments: a call that is not plainly valid throws Decline and becomes None ──
struct Decline {};
struct PyError {};   // a Python exception is set
void need(bool ok) { if (!ok) throw Decline{}; }

bool none(PyObject* o) { return o == Py_None; }
// the tensor behind `o`, on the current GPU
const Tensor& tensor(PyObject* o) {
    need(THPVariable_Check(o));
    const Tensor& t = THPVariable_Unpack(o);
    need(t.is_cuda() && t.get_device() == c10::hip::current_device());
    return t;
}
long integer(PyObject* o) {
    need(PyLong_Check(o));
    const long v = PyLong_AsLong(o);
    if (v == -1 && PyErr_Occurred()) { PyErr_Clear(); throw Decline{}; }
    return v;
}
int int32(PyObject* o) {
    const long v = integer(o);
    need(v >= -0x7fffffffL && v <= 0x7fffffffL);
    return static_cast<int>(v);
}
bool truth(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) { PyErr_Clear(); throw Decline{}; }
    return v != 0;
}
double number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) { PyErr_Clear(); throw Decline{}; }
    return v;
}

int dtype_code(const Tensor& t) {
    if (t.scalar_type() == at::kBFloat16) return MI_DTYPE_BF16;
    need(t.scalar_type() == at::kHalf);
    return MI_DTYPE_F16;
}
void* current_stream() { return c10::hip::getCurrentHIPStream().stream(); }
// The launches of one call, in order up to the first that is refused, without the interpreter lock: a launch waits where its
// queue is full, and loads its kernel the first time. What they read and write is held by the caller's arguments and by the
// Tensors of the calling function; the library's error message is one per thread.
template <typename... F> void run(const char* op, F... launch) {
    int rc = 0;
    Py_BEGIN_ALLOW_THREADS
    (void)((rc = launch(), rc == 0) && ...);
    Py_END_ALLOW_THREADS
    if (rc == 0) return;
    PyErr_Format(PyExc_RuntimeError, "%s: %s", op, L.last_error());
    throw PyError{};
}
const char* name_of(PyObject* op) {
    const char* s = PyUnicode_Check(op) ? PyUnicode_AsUTF8(op) : nullptr;
    if (!s) { PyErr_Clear(); throw Decline{}; }
    return s;
}
const float* f32(const Tensor& t) { return static_cast<const float*>(t.data_ptr()); }
int rows32(int64_t n) { need(n >= 0 && n <= 0x7fffffff); return static_cast<int>(n); }

// (rows, cols) or (batch, rows, cols), contiguous along columns
struct Mat { int64_t b, rows, cols, rs, bs; };
Mat as3(const Tensor& t) {
    if (t.dim() == 2) {
        need(t.stride(1) == 1);
        return {1, t.size(0), t.size(1), t.stride(0), t.stride(0) * t.size(0)};
    }
    need(t.dim() == 3 && t.stride(2) == 1);
    return {t.size(0), t.size(1), t.size(2), t.stride(1), t.stride(0)};
}

// The result of a wrapped function as a Python value; Decline -> None.
template <typename F> PyObject* guarded(F f) {
    try {
        need(bound);
        return f();
    } catch (const Decline&) {
        Py_RETURN_NONE;
    } catch (const PyError&) {
        return nullptr;
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    }
}
#define NATIVE(name, n_args) PyObject* name(PyObject*, PyObject* const* a, Py_ssize_t n) { if (n != n_args) Py_RETURN_NONE; return guarded([&]() -> PyObject* {
#define NATIVE_END }); }
PyObject* given(PyObject* o, const Tensor& t) {   // the caller's own tensor object where there is one
    if (!none(o)) { Py_INCREF(o); return o; }
    return THPVariable_Wrap(t);
}

// ── linear layers ──
const void* bias_ptr(PyObject* o, at::ScalarType dt, int64_t n) {
    if (none(o)) return nullptr;
    const Tensor& t = tensor(o);
    need(t.scalar_type() == dt && t.numel() == n && t.is_contiguous());
    return t.data_ptr();
}
// a weight of the activation dtype, or INT8 with FP32 scales per row; returns the scales
const float* weight(PyObject* w, PyObject* scales, at::ScalarType dt, int64_t rows = -1, int64_t cols = -1) {
    const Tensor& t = tensor(w);
    need(t.dim() == 2 && t.is_contiguous() && (rows < 0 || t.size(0) == rows) && (cols < 0 || t.size(1) == cols));
    if (none(scales)) { need(t.scalar_type() == dt); return nullptr; }
    need(t.scalar_type() == at::kChar);
    const Tensor& s = tensor(scales);
    need(s.scalar_type() == at::kFloat && s.numel() == t.size(0) && s.is_contiguous());
    return f32(s);
}
// `out` given: contiguous, `cols` wide, `numel` values; else allocated with x's leading sizes
Tensor output(PyObject* out, const Tensor& x, int64_t cols) {
    need(x.dim() >= 1 && x.size(-1) > 0);   // (no row count for rows without values)
    const int64_t numel = x.numel() / x.size(-1) * cols;
    if (none(out)) {
        auto sizes = x.sizes().vec();
        sizes.back() = cols;
        return at::empty(sizes, x.options());
    }
    const Tensor& y = tensor(out);
    need(y.dim() >= 1 && y.scalar_type() == x.scalar_type() && y.is_contiguous() && y.size(-1) == cols && y.numel() == numel);
    return y;
}
mi_linear_args linear_args(PyObject* W, PyObject* bias, const Tensor& x, const Tensor& y, PyObject* scales, int64_t n_out) {
    const Tensor& w = tensor(W);
    mi_linear_args p;
    std::memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.dtype = dtype_code(x);
    p.w_scales = weight(W, scales, x.scalar_type());
    p.x = x.data_ptr(); p.w = w.data_ptr(); p.y = y.data_ptr();
    p.bias = bias_ptr(bias, x.scalar_type(), w.size(0));
    p.rows = rows32(x.numel() / x.size(-1)); p.in_features = rows32(w.size(1)); p.out_features = rows32(n_out);
    p.stream = current_stream();
    return p;
}
const Tensor& activations(PyObject* o, PyObject* W) {
    const Tensor& x = tensor(o);
    const Tensor& w = tensor(W);
    need(x.dim() >= 1 && x.is_contiguous() && w.dim() == 2 && x.size(-1) == w.size(1) && w.size(1) > 0);
    return x;
}

// W, bias, X, Y, W_scales, op
NATIVE(linear, 6)
    const Tensor& x = activations(a[2], a[0]);
    const int64_t n_out = tensor(a[0]).size(0);
    const Tensor y = output(a[3], x, n_out);
    const mi_linear_args p = linear_args(a[0], a[1], x, y, a[4], n_out);
    run(name_of(a[5]), [&] { return L.linear(&p); });
    return given(a[3], y);
NATIVE_END

// X, W, b, Y, W_scales, op
NATIVE(geglu, 6)
    const Tensor& x = activations(a[0], a[1]);
    const int64_t two_n = tensor(a[1]).size(0);
    need(two_n % 2 == 0);
    const Tensor y = output(a[3], x, two_n / 2);
    const mi_linear_args p = linear_args(a[1], a[2], x, y, a[4], two_n / 2);
    run(name_of(a[5]), [&] { return L.geglu(&p); });
    return given(a[3], y);
NATIVE_END

// Y, X
NATIVE(add_inplace, 2)
    const Tensor &y = tensor(a[0]), &x = tensor(a[1]);
    need(y.sizes() == x.sizes() && y.scalar_type() == x.scalar_type() && y.is_contiguous() && x.is_contiguous());
    void* const py = y.data_ptr();
    const void* const px = x.data_ptr();
    const int64_t numel = y.numel();
    const int dt = dtype_code(y);
    void* const stream = current_stream();
    run("add_inplace_vec", [&] { return L.add_inplace(py, px, numel, dt, stream); });
    return given(a[0], y);
NATIVE_END

// X, gain, eps, out
NATIVE(rms_norm, 4)
    const Tensor &x = tensor(a[0]), &g = tensor(a[1]);
    need(x.dim() == 2 && x.stride(1) == 1 && g.scalar_type() == x.scalar_type() && g.numel() == x.size(1) && g.is_contiguous());
    const Tensor y = none(a[3]) ? at::empty_like(x) : tensor(a[3]);
    need(y.sizes() == x.sizes() && y.scalar_type() == x.scalar_type() && y.stride(1) == 1);
    const void *const px = x.data_ptr(), *const pg = g.data_ptr();
    void* const py = y.data_ptr();
    const int rows = rows32(x.size(0)), cols = rows32(x.size(1)), dt = dtype_code(x);
    const int64_t x_rs = x.stride(0), y_rs = y.stride(0);
    const float eps = static_cast<float>(number(a[2]));
    void* const stream = current_stream();
    run("rms_norm_rows", [&] { return L.rms_norm(px, pg, py, rows, cols, x_rs, y_rs, eps, dt, stream); });
    return given(a[3], y);
NATIVE_END

// ── RoPE ──
const float* table(PyObject* o, int64_t rows, int64_t half) {
    const Tensor& t = tensor(o);
    need(t.scalar_type() == at::kFloat && t.dim() == 2 && t.size(0) == rows && t.size(1) == half && t.is_contiguous());
    return f32(t);
}

// X, cos, sin, head_dim, num_heads, out, per_head, split_half, op
NATIVE(rope, 9)
    const Tensor& x = tensor(a[0]);
    const int hd = int32(a[3]), heads = int32(a[4]);
    need(hd > 0 && heads > 0 && x.dim() == 2 && x.stride(1) == 1 && x.size(1) == static_cast<int64_t>(hd) * heads);
    const Tensor y = none(a[5]) ? at::empty_like(x) : tensor(a[5]);
    need(y.sizes() == x.sizes() && y.scalar_type() == x.scalar_type() && y.stride(1) == 1);
    mi_rope_args p;
    std::memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.dtype = dtype_code(x);
    p.per_head = truth(a[6]);
    p.split_half = truth(a[7]);
    const int64_t trows = p.per_head ? x.size(0) * heads : x.size(0);
    p.x = x.data_ptr(); p.out = y.data_ptr(); p.cos = table(a[1], trows, hd / 2); p.sin = table(a[2], trows, hd / 2);
    p.rows = rows32(x.size(0)); p.num_heads = heads; p.head_dim = hd;
    p.x_row_stride = x.stride(0); p.out_row_stride = y.stride(0);
    p.stream = current_stream();
    run(name_of(a[8]), [&] { return L.rope(&p); });
    return given(a[5], y);
NATIVE_END

// X, gain, eps, cos, sin, head_dim, num_heads, out, cache_out, split_half
NATIVE(headnorm_rope, 10)
    const Tensor &x = tensor(a[0]), &g = tensor(a[1]);
    const int hd = int32(a[5]), heads = int32(a[6]);
    need(x.dim() == 2 && x.stride(1) == 1 && x.size(1) == static_cast<int64_t>(hd) * heads);
    need(g.scalar_type() == x.scalar_type() && g.numel() == hd && g.is_contiguous());
    const Tensor y = none(a[7]) ? at::empty_like(x) : tensor(a[7]);
    need(y.sizes() == x.sizes() && y.scalar_type() == x.scalar_type() && y.stride(1) == 1);
    mi_headnorm_rope_args p;
    std::memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.dtype = dtype_code(x);
    p.x = x.data_ptr(); p.out = y.data_ptr(); p.gain = g.data_ptr();
    need(none(a[3]) == none(a[4]));
    if (!none(a[3])) { p.cos = table(a[3], x.size(0), hd / 2); p.sin = table(a[4], x.size(0), hd / 2); }
    p.eps = static_cast<float>(number(a[2]));
    p.split_half = truth(a[9]);
    p.rows = rows32(x.size(0)); p.num_heads = heads; p.head_dim = hd;
    p.x_row_stride = x.stride(0); p.out_row_stride = y.stride(0);
    if (!none(a[8])) {
        const Tensor& c = tensor(a[8]);
        need(c.dim() == 2 && c.scalar_type() == x.scalar_type() && c.size(1) == x.size(1) && c.stride(1) == 1 && c.size(0) <= x.size(0));
        p.out2 = c.data_ptr(); p.out2_rows = rows32(c.size(0)); p.out2_row_stride = c.stride(0);
    }
    p.stream = current_stream();
    run("headnorm_rope", [&] { return L.headnorm_rope(&p); });
    return given(a[7], y);
NATIVE_END

// ── softmax attention ──
PyObject *s_mode, *s_q_offset, *s_window, *s_seg_q_end, *s_seg_k_end, *s_seg_causal;   // interned attribute names of SdpaMask
struct Attr {
    PyObject* o;
    Attr(PyObject* from, PyObject* name) : o(PyObject_GetAttr(from, name)) { if (!o) { PyErr_Clear(); throw Decline{}; } }
    ~Attr() { Py_DECREF(o); }
};
void set_mask(mi_sdpa_args& p, PyObject* mask) {
    if (none(mask)) return;
    p.mask_mode = int32(Attr(mask, s_mode).o);
    p.q_offset = int32(Attr(mask, s_q_offset).o);
    p.window = int32(Attr(mask, s_window).o);
    if (p.mask_mode != MI_MASK_BLOCK_CAUSAL) return;
    const Attr qe(mask, s_seg_q_end), ke(mask, s_seg_k_end), ca(mask, s_seg_causal);
    need(PyList_Check(qe.o) && PyList_Check(ke.o) && PyList_Check(ca.o));
    const Py_ssize_t n = PyList_GET_SIZE(qe.o);
    need(n >= 1 && n <= MI_MAX_SEGMENTS && PyList_GET_SIZE(ke.o) == n && PyList_GET_SIZE(ca.o) == n);
    p.n_segments = static_cast<int>(n);
    for (Py_ssize_t i = 0; i < n; ++i) {
        p.seg_q_end[i] = int32(PyList_GET_ITEM(qe.o, i));
        p.seg_k_end[i] = int32(PyList_GET_ITEM(ke.o, i));
        p.seg_causal[i] = truth(PyList_GET_ITEM(ca.o, i));
    }
}
PyObject* lend_scratch = nullptr;   // ops._own_split_scratch(device index, bytes) -> tensor of the calling thread

struct Attention {   // one call; q, k, v and the output are always there
    mi_sdpa_args p;
    Tensor out, scratch;
    int64_t B, Lk;
    Attention(const Tensor& q, const Tensor& k, const Tensor& v, long heads, long kv_heads, PyObject* out_obj) {
        std::memset(&p, 0, sizeof(p));
        p.struct_size = sizeof(p);
        p.dtype = dtype_code(q);
        need(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type());
        const Mat mq = as3(q), mk = as3(k), mv = as3(v);
        need(heads > 0 && mq.cols % heads == 0);
        const int64_t hd = mq.cols / heads, hkv = kv_heads > 0 ? kv_heads : heads;
        need(heads % hkv == 0 && mk.b == mq.b && mv.b == mq.b && mk.cols == hkv * hd && mv.cols == hkv * hd && mv.rows == mk.rows);
        out = none(out_obj) ? at::empty_like(q) : tensor(out_obj);
        need(out.sizes() == q.sizes() && out.scalar_type() == q.scalar_type());
        const Mat mo = as3(out);
        p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr(); p.o = out.data_ptr();
        p.batch = rows32(mq.b); p.num_heads = rows32(heads); p.head_dim = rows32(hd); p.num_kv_heads = rows32(hkv);
        p.q_len = rows32(mq.rows); p.kv_len = rows32(mk.rows);
        p.q_row_stride = mq.rs; p.q_batch_stride = mq.bs; p.k_row_stride = mk.rs; p.k_batch_stride = mk.bs;
        p.v_row_stride = mv.rs; p.v_batch_stride = mv.bs; p.o_row_stride = mo.rs; p.o_batch_stride = mo.bs;
        B = mq.b; Lk = mk.rows;
        p.prefix_k_scale = p.prefix_v_scale = 1.f;
        p.stream = current_stream();
    }
    void rope(PyObject* cos, PyObject* sin, bool on_q) {
        const int64_t rows = on_q ? p.q_len : p.kv_len;
        const float *c = table(cos, rows, p.head_dim / 2), *s = table(sin, rows, p.head_dim / 2);
        if (on_q) { p.rope_cos_q = c; p.rope_sin_q = s; } else { p.rope_cos_k = c; p.rope_sin_k = s; }
    }
    void rope_scratch(const Tensor& t, const Tensor& q, const Tensor& k) {
        need(p.rope_cos_k != nullptr && t.scalar_type() == q.scalar_type() && t.is_contiguous() && t.numel() >= k.numel());
        p.rope_k_scratch = t.data_ptr();
    }
    void key_mask(PyObject* o) {
        const Tensor& m = tensor(o);
        need(m.scalar_type() == at::kFloat && m.is_contiguous());
        const int64_t keys = p.prefix_len + Lk;
        if (m.numel() == keys) p.key_mask_batch_stride = 0;
        else { need(m.numel() == B * keys); p.key_mask_batch_stride = keys; }
        p.key_mask = f32(m);
    }
    // split_scratch: None = the scratch of ops.py for this device and stream, False = none, a tensor = that
    void lend(PyObject* split_scratch) {
        if (split_scratch == Py_False) return;
        const size_t bytes = L.sdpa_split_bytes(&p);
        if (bytes == 0) return;
        PyObject* own = nullptr;
        if (none(split_scratch)) {
            own = PyObject_CallFunction(lend_scratch, "in", static_cast<int>(out.get_device()), static_cast<Py_ssize_t>(bytes));
            if (!own) throw PyError{};
        }
        try { scratch = tensor(own ? own : split_scratch); } catch (...) { Py_XDECREF(own); throw; }
        Py_XDECREF(own);
        need(scratch.is_contiguous());
        p.split_scratch = scratch.data_ptr();
        p.split_scratch_bytes = scratch.numel() * scratch.element_size();
    }
};

// q, k, v, num_heads, out, num_kv_heads, k_prefix, v_prefix, scale, mask, kv_valid_len, key_mask, rope_q, rope_k, rope_k_scratch,
// rope_split_half, split_scratch, op
NATIVE(sdpa, 18)
    const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    Attention c(q, k, v, integer(a[3]), integer(a[5]), a[4]);
    mi_sdpa_args& p = c.p;
    need(none(a[6]) == none(a[7]));
    if (!none(a[6])) {
        const Tensor &kp = tensor(a[6]), &vp = tensor(a[7]);
        need(kp.scalar_type() == q.scalar_type() && vp.scalar_type() == q.scalar_type());
        const Mat mk = as3(kp), mv = as3(vp);
        const int64_t cols = static_cast<int64_t>(p.num_kv_heads) * p.head_dim;
        need(mk.b == c.B && mv.b == c.B && mk.cols == cols && mv.cols == cols && mv.rows == mk.rows);
        p.k_prefix = kp.data_ptr(); p.v_prefix = vp.data_ptr(); p.prefix_len = rows32(mk.rows);
        p.kp_row_stride = mk.rs; p.kp_batch_stride = mk.bs; p.vp_row_stride = mv.rs; p.vp_batch_stride = mv.bs;
    }
    if (!none(a[8])) p.scale = static_cast<float>(number(a[8]));
    set_mask(p, a[9]);
    if (!none(a[10])) {
        const Tensor& t = tensor(a[10]);
        need(t.scalar_type() == at::kInt && t.numel() == c.B && t.is_contiguous());
        p.kv_valid_len = static_cast<const int32_t*>(t.data_ptr());
    }
    if (!none(a[11])) c.key_mask(a[11]);
    for (int i = 12; i <= 13; ++i)
        if (!none(a[i])) {
            need(PyTuple_Check(a[i]) && PyTuple_GET_SIZE(a[i]) == 2);
            c.rope(PyTuple_GET_ITEM(a[i], 0), PyTuple_GET_ITEM(a[i], 1), i == 12);
        }
    p.rope_split_half = truth(a[15]);
    if (!none(a[14])) c.rope_scratch(tensor(a[14]), q, k);
    c.lend(a[16]);
    run(name_of(a[17]), [&] { return L.sdpa(&p); });
    return given(a[4], c.out);
NATIVE_END

// Q, K, V, cos, sin, head_dim, num_heads, out, Kr, split_half
NATIVE(joint, 10)
    const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    const long hd = integer(a[5]), heads = integer(a[6]);
    need(q.dim() == 2 && q.size(1) == hd * heads && k.sizes() == q.sizes() && v.sizes() == q.sizes());
    Attention c(q, k, v, heads, 0, a[7]);
    c.rope(a[3], a[4], true);
    c.rope(a[3], a[4], false);
    c.p.rope_split_half = truth(a[9]);
    if (!none(a[8])) {
        const Tensor& kr = tensor(a[8]);
        need(kr.sizes() == k.sizes() && kr.scalar_type() == k.scalar_type());
        c.rope_scratch(kr, q, k);
    }
    c.lend(Py_None);
    run("joint_attention", [&] { return L.sdpa(&c.p); });
    return given(a[7], c.out);
NATIVE_END

// ── attention with its projections ──
// X, Ctx, K, V, Wq, bq, Wk, bk, Wv, bv, Wo, bo, d_mask, num_heads, causal, out, scratch, Wq_scales, Wk_scales, Wv_scales, Wo_scales, op
NATIVE(attn_block, 22)
    const Tensor &x = tensor(a[0]), &wq = tensor(a[4]), &wo = tensor(a[10]);
    need(x.is_contiguous() && wq.dim() == 2 && wo.dim() == 2);
    const at::ScalarType dt = x.scalar_type();
    const Mat mx = as3(x);
    const int64_t inner = wq.size(0), c_out = wo.size(0);
    mi_attn_block_args p;
    std::memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.dtype = dtype_code(x);
    p.wq_scales = weight(a[4], a[17], dt, -1, mx.cols);
    p.wo_scales = weight(a[10], a[20], dt, -1, inner);
    p.x = x.data_ptr(); p.wq = wq.data_ptr(); p.wo = wo.data_ptr();
    p.bq = bias_ptr(a[5], dt, inner); p.bo = bias_ptr(a[11], dt, c_out);
    int64_t lk = mx.rows;
    const bool cached = !none(a[2]);
    if (cached) {
        const Tensor &k = tensor(a[2]), &v = tensor(a[3]);
        const Mat mk = as3(k);
        need(mk.b == mx.b && mk.cols == inner && v.sizes() == k.sizes() && k.scalar_type() == dt && v.scalar_type() == dt && k.is_contiguous() && v.is_contiguous());
        lk = mk.rows;
        p.k = const_cast<void*>(static_cast<const void*>(k.data_ptr())); p.v = v.data_ptr();
    } else {
        int64_t cc = mx.cols;
        if (!none(a[1])) {
            const Tensor& ctx = tensor(a[1]);
            const Mat mc = as3(ctx);
            need(mc.b == mx.b && ctx.scalar_type() == dt && ctx.is_contiguous());
            cc = mc.cols; lk = mc.rows;
            p.ctx = ctx.data_ptr();
        }
        p.wk_scales = weight(a[6], a[18], dt, inner, cc);
        p.wv_scales = weight(a[8], a[19], dt, inner, cc);
        p.wk = tensor(a[6]).data_ptr(); p.wv = tensor(a[8]).data_ptr();
        p.bk = bias_ptr(a[7], dt, inner); p.bv = bias_ptr(a[9], dt, inner);
        p.ctx_channels = rows32(cc);
    }
    p.batch = rows32(mx.b); p.q_len = rows32(mx.rows); p.kv_len = rows32(lk);
    p.channels = rows32(mx.cols); p.inner = rows32(inner); p.out_channels = rows32(c_out);
    p.num_heads = int32(a[13]);
    p.causal = truth(a[14]);
    if (!none(a[12])) {
        const Tensor& m = tensor(a[12]);
        need(m.scalar_type() == at::kFloat && m.is_contiguous() && (m.numel() == lk || m.numel() == mx.b * lk));
        p.key_mask = f32(m);
        p.key_mask_batch_stride = m.numel() == mx.b * lk && mx.b > 1 ? lk : 0;
    }
    const Tensor out = output(a[15], x, c_out);
    p.out = out.data_ptr();
    const Tensor scratch = none(a[16]) ? at::empty({static_cast<int64_t>(L.block_scratch_bytes(&p))}, x.options().dtype(at::kByte)) : tensor(a[16]);
    need(scratch.is_contiguous());
    p.scratch = scratch.data_ptr(); p.scratch_bytes = scratch.numel() * scratch.element_size();
    p.stream = current_stream();
    run(name_of(a[21]), [&] { return (cached ? L.kv_cached : L.qkvo)(&p); });
    return given(a[15], out);
NATIVE_END

// X, Wq, Wk, Wv, Wo, bq, bk, bv, bo, d_mask, num_heads, qh, kh, vh, yc, out -> (out, qh, kh, vh, yc)
NATIVE(mha, 16)
    const Tensor& x = activations(a[0], a[1]);
    need(x.dim() == 2);
    const int64_t inner = tensor(a[1]).size(0);
    const long heads = integer(a[10]);
    need(heads > 0 && inner % heads == 0);
    mi_linear_args p[3];
    Tensor qkv[3];
    for (int i = 0; i < 3; ++i) {
        activations(a[0], a[1 + i]);
        need(tensor(a[1 + i]).size(0) == inner);
        qkv[i] = output(a[11 + i], x, inner);
        need(qkv[i].dim() == 2);
        p[i] = linear_args(a[1 + i], a[5 + i], x, qkv[i], Py_None, inner);
    }
    Attention c(qkv[0], qkv[1], qkv[2], heads, 0, a[14]);
    if (!none(a[9])) {
        need(tensor(a[9]).numel() == x.size(0));
        c.key_mask(a[9]);
    }
    const int64_t n_out = tensor(a[4]).size(0);
    need(c.out.is_contiguous() && tensor(a[4]).dim() == 2 && tensor(a[4]).size(1) == inner);
    const Tensor y = output(a[15], c.out, n_out);
    const mi_linear_args po = linear_args(a[4], a[8], c.out, y, Py_None, n_out);
    c.lend(Py_None);
    run("mha_forward", [&] { return L.linear_n(p, 3); }, [&] { return L.sdpa(&c.p); }, [&] { return L.linear(&po); });
    PyObject* parts[5] = {given(a[15], y), given(a[11], qkv[0]), given(a[12], qkv[1]), given(a[13], qkv[2]), given(a[14], c.out)};
    PyObject* t = PyTuple_New(5);
    for (int i = 0; i < 5; ++i) PyTuple_SET_ITEM(t, i, parts[i]);
    return t;
NATIVE_END

// ── ReLU linear attention ──
void linear_attn_args(mi_linear_attn_args& p, const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, int heads, float eps, const Tensor& ws, bool accumulate) {
    std::memset(&p, 0, sizeof(p));
    p.struct_size = sizeof(p);
    p.dtype = dtype_code(q);
    need(k.scalar_type() == q.scalar_type() && v.scalar_type() == q.scalar_type() && k.sizes() == q.sizes() && v.sizes() == q.sizes());
    need(o.sizes() == q.sizes() && o.scalar_type() == q.scalar_type());
    const Mat mq = as3(q), mk = as3(k), mv = as3(v), mo = as3(o);
    need(heads > 0 && mq.cols % heads == 0);
    p.q = q.data_ptr(); p.k = k.data_ptr(); p.v = v.data_ptr(); p.o = o.data_ptr();
    p.batch = rows32(mq.b); p.num_heads = heads; p.head_dim = rows32(mq.cols / heads); p.n_tokens = rows32(mq.rows);
    p.q_row_stride = mq.rs; p.q_batch_stride = mq.bs; p.k_row_stride = mk.rs; p.k_batch_stride = mk.bs;
    p.v_row_stride = mv.rs; p.v_batch_stride = mv.bs; p.o_row_stride = mo.rs; p.o_batch_stride = mo.bs;
    p.eps = eps;
    p.accumulate_state = accumulate;
    need(ws.scalar_type() == at::kFloat && ws.is_contiguous() &&
         static_cast<size_t>(ws.numel()) * 4 >= L.la_workspace_bytes(p.batch, p.num_heads, p.head_dim));
    p.workspace = ws.data_ptr(); p.workspace_bytes = ws.numel() * 4;
    p.stream = current_stream();
}

// Q, K, V, num_heads, out, eps, workspace, accumulate_state, scratch, form
NATIVE(linear_attn, 10)
    const Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]);
    const int heads = int32(a[3]);
    need((q.dim() == 2 || q.dim() == 3) && heads > 0 && q.size(-1) % heads == 0);
    const bool accumulate = truth(a[7]);
    need(!(accumulate && none(a[6])));
    const int B = q.dim() == 3 ? rows32(q.size(0)) : 1, hd = rows32(q.size(-1) / heads);
    const auto f32_opts = q.options().dtype(at::kFloat);
    const Tensor out = none(a[4]) ? at::empty_like(q) : tensor(a[4]);
    const Tensor ws = none(a[6]) ? at::empty({static_cast<int64_t>(L.la_workspace_bytes(B, heads, hd) / 4)}, f32_opts) : tensor(a[6]);
    mi_linear_attn_args p;
    linear_attn_args(p, q, k, v, out, heads, static_cast<float>(number(a[5])), ws, accumulate);
    Tensor sc;
    if (a[8] != Py_False) {
        sc = none(a[8]) ? at::empty({static_cast<int64_t>(L.la_scratch_bytes(B, heads, hd) / 4)}, f32_opts) : tensor(a[8]);
        need(sc.scalar_type() == at::kFloat && sc.is_contiguous());
        if (sc.numel() > 0) { p.scratch = sc.data_ptr(); p.scratch_bytes = sc.numel() * 4; }
    }
    p.form = int32(a[9]);
    run("linear_attention_relu_forward", [&] { return L.linear_attn(&p); });
    return given(a[4], out);
NATIVE_END

// x_mod, Wq, Wk, Wv, Wo, bo, num_heads, nq, nk, rms_eps, attn_eps, state (None, or the tensor that captures it), out
NATIVE(sana, 13)
    const Tensor& x = activations(a[0], a[1]);
    const int heads = int32(a[6]);
    need(x.dim() == 2 && heads > 0 && x.size(1) % heads == 0 && x.size(0) > 0);
    const int64_t d = x.size(1), hd = d / heads;
    for (int i = 1; i <= 4; ++i) { const Tensor& w = tensor(a[i]); need(w.dim() == 2 && w.size(1) == d && (i == 4 || w.size(0) == d)); }
    need(none(a[7]) == none(a[8]));
    // q, k, v and the attention output, the partial states and (unless it is captured) the state, in two allocations
    const int64_t n = x.size(0);
    const Tensor qkvo = at::empty({4, n, d}, x.options());
    const int64_t state = heads * (hd * hd + hd), scratch = L.la_scratch_bytes(1, heads, rows32(hd)) / 4;
    const Tensor f = at::empty({(state + scratch + 7) / 4 * 4}, x.options().dtype(at::kFloat));
    const Tensor q = qkvo.select(0, 0), k = qkvo.select(0, 1), v = qkvo.select(0, 2), attn = qkvo.select(0, 3);
    mi_linear_args p[3] = {linear_args(a[1], Py_None, x, q, Py_None, d), linear_args(a[2], Py_None, x, k, Py_None, d), linear_args(a[3], Py_None, x, v, Py_None, d)};
    const int dt = dtype_code(x);
    const void *gq = nullptr, *gk = nullptr;
    if (!none(a[7])) {
        gq = bias_ptr(a[7], x.scalar_type(), d);
        gk = bias_ptr(a[8], x.scalar_type(), d);
    }
    if (!none(a[11])) { const Tensor& s = tensor(a[11]); need(s.scalar_type() == at::kFloat && s.is_contiguous() && s.numel() == state); }
    const Tensor ws = none(a[11]) ? f.narrow(0, (scratch + 3) / 4 * 4, state) : tensor(a[11]);
    mi_linear_attn_args la;
    linear_attn_args(la, q, k, v, attn, heads, static_cast<float>(number(a[10])), ws, false);
    la.scratch = f.data_ptr(); la.scratch_bytes = scratch * 4;
    const int64_t n_out = tensor(a[4]).size(0);
    const Tensor y = output(a[12], x, n_out);
    const mi_linear_args po = linear_args(a[4], a[5], attn, y, Py_None, n_out);
    void *const pq = q.data_ptr(), *const pk = k.data_ptr(), *const stream = current_stream();
    const float rms_eps = static_cast<float>(number(a[9]));
    const int rows = rows32(n), cols = rows32(d);
    auto norms = [&] { return gq ? L.rms_norm_pair(pq, gq, pq, pk, gk, pk, rows, cols, 0, 0, rms_eps, dt, stream) : 0; };
    run("sana_self_attention", [&] { return L.linear_n(p, 3); }, norms, [&] { return L.linear_attn(&la); }, [&] { return L.linear(&po); });
    return given(a[12], y);
NATIVE_END

// ── module ──
PyObject* bind(PyObject*, PyObject* args) {
    const char* path;
    PyObject* lend;
    if (!PyArg_ParseTuple(args, "sO", &path, &lend)) return nullptr;
    void* h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!h) return PyErr_Format(PyExc_RuntimeError, "%s", dlerror());
    bool ok = true;
    auto get = [&](auto& f, const char* name) {
        f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(dlsym(h, name));
        ok = ok && f != nullptr;
    };
    get(L.last_error, "mi_last_error"); get(L.sdpa, "mi_sdpa_forward"); get(L.sdpa_split_bytes, "mi_sdpa_split_scratch_bytes");
    get(L.rope, "mi_rope_apply"); get(L.headnorm_rope, "mi_headnorm_rope"); get(L.linear, "mi_linear_forward"); get(L.linear_n, "mi_linear_forward_n");
    get(L.geglu, "mi_linear_geglu_forward"); get(L.add_inplace, "mi_add_inplace"); get(L.rms_norm, "mi_rms_norm_forward");
    get(L.rms_norm_pair, "mi_rms_norm_pair_forward"); get(L.block_scratch_bytes, "mi_attn_block_scratch_bytes");
    get(L.qkvo, "mi_flash_attention_qkvo_forward"); get(L.kv_cached, "mi_flash_attention_q_with_kv_cached_forward");
    get(L.la_workspace_bytes, "mi_linear_attn_workspace_bytes"); get(L.la_scratch_bytes, "mi_linear_attn_scratch_bytes");
    get(L.linear_attn, "mi_linear_attn_relu_forward");
    if (!ok) return PyErr_Format(PyExc_RuntimeError, "%s does not export every function of mi_attention.h: build the library again", path);
    Py_INCREF(lend);
    Py_XSETREF(lend_scratch, lend);
    bound = true;
    Py_RETURN_NONE;
}

#define FAST(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"bind", bind, METH_VARARGS, nullptr}, FAST(linear), FAST(geglu), FAST(add_inplace), FAST(rms_norm), FAST(rope), FAST(headnorm_rope),
                         FAST(sdpa), FAST(joint), FAST(attn_block), FAST(mha), FAST(linear_attn), FAST(sana), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", "Native host path of brodiffusion_amd.ops.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) {
    s_mode = PyUnicode_InternFromString("mode"); s_q_offset = PyUnicode_InternFromString("q_offset"); s_window = PyUnicode_InternFromString("window");
    s_seg_q_end = PyUnicode_InternFromString("seg_q_end"); s_seg_k_end = PyUnicode_InternFromString("seg_k_end");
    s_seg_causal = PyUnicode_InternFromString("seg_causal");
    return PyModule_Create(&module);
}
