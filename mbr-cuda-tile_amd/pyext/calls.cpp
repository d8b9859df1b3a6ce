// Native half of the Python binding: the calls a model makes hundreds of times per chunk, from
// torch tensors straight to the C-ABI of libmbrt.so.  Each function checks what its Python
// wrapper (mbrt/__init__.py) documents, reads pointers, sizes and dtypes from the tensors,
// and enqueues on the given stream handle, or on torch's current stream for None.
//
// What it is for: a small kernel runs for 2-4 us, while a call through ctypes took 8.3 us of host
// time (attribute lookups, a ctypes object per argument, a Structure filled element by
// element), so that a chunk's loops of small calls ran at the host's pace.  From here a call
// takes 3.9 us, most of it the launch: the 60 per-band slices and norms of a chunk, 121
// calls, 1009 -> 475 us; the 40 calls of a one-minute song's overlap-add 335 -> 242 us.
//
// Like ctypes' calls, the library is entered without the interpreter lock.
#include <torch/csrc/Dtype.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <c10/hip/HIPStream.h>

#include <vector>

#include "../../include/mbrt.h"

namespace {

PyObject* g_error = nullptr;  // mbrt.MbrtError(function, status, message)

[[noreturn]] void raise(PyObject* type, const char* msg) {
    PyErr_SetString(type, msg);
    throw python_error();
}

const at::Tensor& tensor(PyObject* o) {
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, "mbrt: expected a torch.Tensor");
    return THPVariable_Unpack(o);
}

// An optional tensor argument: undefined for None.
at::Tensor tensor_or_none(PyObject* o) { return o == Py_None ? at::Tensor() : tensor(o); }

int dtype_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case at::kFloat: return MBRT_F32;
        case at::kHalf: return MBRT_F16;
        case at::kBFloat16: return MBRT_BF16;
        case at::kLong: return MBRT_I64;
        case at::kInt: return MBRT_I32;
        default: break;
    }
    const std::string msg = std::string("mbrt: unsupported dtype torch.") + torch::getTHPDtype(t.scalar_type())->name;
    raise(PyExc_TypeError, msg.c_str());
}
int dtype_or(const at::Tensor& t, int none) { return t.defined() ? dtype_code(t) : none; }

void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }

void contig(std::initializer_list<const at::Tensor*> ts) {
    for (const at::Tensor* t : ts)
        if (t->defined() && !t->is_contiguous()) raise(PyExc_ValueError, "mbrt: expected a contiguous tensor");
}

int64_t integer(PyObject* o) {
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw python_error();
    return v;
}
double number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return v;
}
int truth(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw python_error();
    return v;
}

int64_t floor_div(int64_t a, int64_t b) {
    if (b == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    return a / b;
}

mbrt_stream_t stream(PyObject* o) {
    if (o == Py_None) return c10::hip::getCurrentHIPStream().stream();
    return reinterpret_cast<mbrt_stream_t>(static_cast<uintptr_t>(integer(o)));
}

template <class F>
PyObject* call(const char* name, F f) {
    int status;
    Py_BEGIN_ALLOW_THREADS
    status = f();
    Py_END_ALLOW_THREADS
    if (status != MBRT_OK) {
        PyObject* e = PyObject_CallFunction(g_error, "sis", name, status, mbrt_last_error());
        if (e != nullptr) {
            PyErr_SetObject(g_error, e);
            Py_DECREF(e);
        }
        throw python_error();
    }
    Py_RETURN_NONE;
}

void count(Py_ssize_t n, Py_ssize_t want) {
    if (n != want) raise(PyExc_TypeError, "mbrt: wrong number of arguments to a native call");
}

void check_dims(const at::Tensor& t) {
    if (t.dim() > MBRT_MAX_DIMS) raise(PyExc_IndexError, "invalid index");
}

#define MBRT_PY(fname) PyObject* fname(PyObject*, PyObject* const* a, Py_ssize_t n)

// fill(t, value, stream)
MBRT_PY(fill) {
    HANDLE_TH_ERRORS
    count(n, 3);
    const at::Tensor& t = tensor(a[0]);
    contig({&t});
    const int dt = dtype_code(t);
    void* p = ptr(t);
    const double v = number(a[1]);
    const int64_t ne = t.numel();
    const mbrt_stream_t st = stream(a[2]);
    return call("mbrt_fill", [&] { return mbrt_fill(p, dt, ne, v, st); });
    END_HANDLE_TH_ERRORS
}

// strided_copy(src, dst, stream)
MBRT_PY(strided_copy) {
    HANDLE_TH_ERRORS
    count(n, 3);
    const at::Tensor &src = tensor(a[0]), &dst = tensor(a[1]);
    contig({&dst});
    if (src.sizes() != dst.sizes()) raise(PyExc_ValueError, "strided_copy: shape mismatch");
    check_dims(src);
    mbrt_strided_meta m{};
    m.ndim = (int32_t)src.dim();
    for (int64_t d = 0; d < src.dim(); ++d) {
        m.dst_shape[d] = src.size(d);
        m.src_strides[d] = src.stride(d);
    }
    const int dt = dtype_code(src);
    void *sp = ptr(src), *dp = ptr(dst);
    const mbrt_stream_t st = stream(a[2]);
    return call("mbrt_strided_copy", [&] { return mbrt_strided_copy(sp, dp, dt, &m, st); });
    END_HANDLE_TH_ERRORS
}

// pad(src, out, before (sequence), value, reflect, stream)
MBRT_PY(pad) {
    HANDLE_TH_ERRORS
    count(n, 6);
    const at::Tensor &src = tensor(a[0]), &out = tensor(a[1]);
    contig({&src, &out});
    check_dims(src);
    mbrt_pad_meta m{};
    m.ndim = (int32_t)src.dim();
    for (int64_t d = 0; d < src.dim(); ++d) {
        m.src_shape[d] = src.size(d);
        m.dst_shape[d] = out.size(d);
        PyObject* b = PySequence_GetItem(a[2], d);
        if (b == nullptr) throw python_error();
        const int64_t v = PyLong_AsLongLong(b);
        Py_DECREF(b);
        if (v == -1 && PyErr_Occurred()) throw python_error();
        m.pad_before[d] = v;
    }
    const int dt = dtype_code(src);
    void *sp = ptr(src), *op = ptr(out);
    const mbrt_stream_t st = stream(a[5]);
    if (truth(a[4])) return call("mbrt_pad_reflect", [&] { return mbrt_pad_reflect(sp, op, dt, &m, st); });
    const float value = (float)number(a[3]);
    return call("mbrt_pad_const", [&] { return mbrt_pad_const(sp, op, dt, &m, value, st); });
    END_HANDLE_TH_ERRORS
}

// cat(srcs (sequence), dim, out, stream)
MBRT_PY(cat) {
    HANDLE_TH_ERRORS
    count(n, 4);
    const at::Tensor& out = tensor(a[2]);
    contig({&out});
    THPObjectPtr seq(PySequence_Fast(a[0], "mbrt.cat: expected a sequence of tensors"));
    if (!seq) throw python_error();
    const Py_ssize_t ns = PySequence_Fast_GET_SIZE(seq.get());
    PyObject** items = PySequence_Fast_ITEMS(seq.get());
    for (Py_ssize_t i = 0; i < ns; ++i) contig({&tensor(items[i])});
    if (out.dim() == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    int64_t dim = integer(a[1]) % out.dim();
    if (dim < 0) dim += out.dim();
    int64_t outer = 1, inner = 1, off = 0;
    for (int64_t d = 0; d < dim; ++d) outer *= out.size(d);
    for (int64_t d = dim + 1; d < out.dim(); ++d) inner *= out.size(d);
    std::vector<mbrt_cat_src> srcs((size_t)ns);
    for (Py_ssize_t i = 0; i < ns; ++i) {
        const at::Tensor& s = tensor(items[i]);
        srcs[i] = mbrt_cat_src{ptr(s), s.size(dim), off};
        off += s.size(dim);
    }
    void* op = ptr(out);
    const int64_t total = out.size(dim), bytes = inner * (int64_t)out.element_size();
    const mbrt_stream_t st = stream(a[3]);
    return call("mbrt_cat", [&] { return mbrt_cat(op, srcs.data(), (int)ns, outer, total, bytes, st); });
    END_HANDLE_TH_ERRORS
}

// rms_norm(x, gamma, out, scale, eps, stream)
MBRT_PY(rms_norm) {
    HANDLE_TH_ERRORS
    count(n, 6);
    const at::Tensor &x = tensor(a[0]), &g = tensor(a[1]), &out = tensor(a[2]);
    contig({&x, &g, &out});
    const int64_t dim = x.size(-1);
    const int xd = dtype_code(x), gd = dtype_code(g), od = dtype_code(out);
    const int64_t rows = floor_div(x.numel(), dim);
    void *xp = ptr(x), *gp = ptr(g), *op = ptr(out);
    const float scale = (float)number(a[3]), eps = (float)number(a[4]);
    const mbrt_stream_t st = stream(a[5]);
    return call("mbrt_rms_norm", [&] { return mbrt_rms_norm(xp, xd, gp, gd, op, od, rows, dim, scale, eps, st); });
    END_HANDLE_TH_ERRORS
}

// residual_add_rms_norm(residual, update, gamma, sum_out | None, normed, scale, eps, stream)
MBRT_PY(residual_add_rms_norm) {
    HANDLE_TH_ERRORS
    count(n, 8);
    const at::Tensor &r = tensor(a[0]), &u = tensor(a[1]), &g = tensor(a[2]), &out = tensor(a[4]);
    const at::Tensor sum = tensor_or_none(a[3]);
    contig({&r, &u, &g, &sum, &out});
    const int64_t dim = r.size(-1);
    const int rd = dtype_code(r), gd = dtype_code(g), od = dtype_code(out), sd = dtype_or(sum, rd);
    const int64_t rows = floor_div(r.numel(), dim);
    void *rp = ptr(r), *up = ptr(u), *gp = ptr(g), *sp = ptr(sum), *op = ptr(out);
    const float scale = (float)number(a[5]), eps = (float)number(a[6]);
    const mbrt_stream_t st = stream(a[7]);
    return call("mbrt_residual_add_rms_norm", [&] {
        return mbrt_residual_add_rms_norm(rp, up, rd, gp, gd, sp, sd, op, od, rows, dim, scale, eps, st);
    });
    END_HANDLE_TH_ERRORS
}

// bias_act(x, bias | None, out, act, stream)
MBRT_PY(bias_act) {
    HANDLE_TH_ERRORS
    count(n, 5);
    const at::Tensor &x = tensor(a[0]), &out = tensor(a[2]);
    const at::Tensor bias = tensor_or_none(a[1]);
    contig({&x, &bias, &out});
    const int64_t cols = x.size(-1);
    const int xd = dtype_code(x), bd = dtype_or(bias, MBRT_F32), od = dtype_code(out);
    const int64_t rows = floor_div(x.numel(), cols);
    void *xp = ptr(x), *bp = ptr(bias), *op = ptr(out);
    const int act = (int)integer(a[3]);
    const mbrt_stream_t st = stream(a[4]);
    return call("mbrt_bias_act", [&] { return mbrt_bias_act(xp, xd, bp, bd, op, od, rows, cols, act, st); });
    END_HANDLE_TH_ERRORS
}

// glu(x, out, stream)
MBRT_PY(glu) {
    HANDLE_TH_ERRORS
    count(n, 3);
    const at::Tensor &x = tensor(a[0]), &out = tensor(a[1]);
    contig({&x, &out});
    const int64_t full = x.size(-1);
    if (full % 2 != 0) raise(PyExc_ValueError, "glu_last_dim: last dimension must be even");
    const int xd = dtype_code(x), od = dtype_code(out);
    const int64_t rows = floor_div(x.numel(), full);
    void *xp = ptr(x), *op = ptr(out);
    const mbrt_stream_t st = stream(a[2]);
    return call("mbrt_glu_last_dim", [&] { return mbrt_glu_last_dim(xp, xd, op, od, rows, full / 2, st); });
    END_HANDLE_TH_ERRORS
}

// gate_merge(attn, gate, out, layout, gate_is_logit, stream)
MBRT_PY(gate_merge) {
    HANDLE_TH_ERRORS
    count(n, 6);
    const at::Tensor &at_ = tensor(a[0]), &g = tensor(a[1]), &out = tensor(a[2]);
    contig({&at_, &g, &out});
    const int layout = (int)integer(a[3]);
    if (at_.dim() != 4) raise(PyExc_ValueError, "gate_merge: expected a 4-d attention output");
    const bool bhnd = layout == MBRT_LAYOUT_BHND;
    const int64_t B = at_.size(0), H = at_.size(bhnd ? 1 : 2), N = at_.size(bhnd ? 2 : 1), D = at_.size(3);
    const int ad = dtype_code(at_), gd = dtype_code(g), od = dtype_code(out), logit = truth(a[4]);
    void *ap = ptr(at_), *gp = ptr(g), *op = ptr(out);
    const mbrt_stream_t st = stream(a[5]);
    return call("mbrt_sigmoid_gate_merge", [&] {
        return mbrt_sigmoid_gate_merge(ap, ad, gp, gd, logit, op, od, B, H, N, D, layout, st);
    });
    END_HANDLE_TH_ERRORS
}

// softmax(x, out, scale, stream)
MBRT_PY(softmax) {
    HANDLE_TH_ERRORS
    count(n, 4);
    const at::Tensor &x = tensor(a[0]), &out = tensor(a[1]);
    contig({&x, &out});
    const int64_t cols = x.size(-1);
    const int xd = dtype_code(x), od = dtype_code(out);
    const int64_t rows = floor_div(x.numel(), cols);
    void *xp = ptr(x), *op = ptr(out);
    const float scale = (float)number(a[2]);
    const mbrt_stream_t st = stream(a[3]);
    return call("mbrt_softmax_rows", [&] { return mbrt_softmax_rows(xp, xd, op, od, rows, cols, scale, st); });
    END_HANDLE_TH_ERRORS
}

// split_qkv_rotary(qkv, cos, sin, q, k, v, heads, stream)
MBRT_PY(split_qkv_rotary) {
    HANDLE_TH_ERRORS
    count(n, 8);
    const at::Tensor &qkv = tensor(a[0]), &c = tensor(a[1]), &s = tensor(a[2]), &q = tensor(a[3]), &k = tensor(a[4]),
                     &v = tensor(a[5]);
    contig({&qkv, &c, &s, &q, &k, &v});
    if (qkv.dim() != 3) raise(PyExc_ValueError, "split_qkv_rotary: expected qkv [B, N, 3 H D]");
    const int64_t heads = integer(a[6]), B = qkv.size(0), N = qkv.size(1), D = floor_div(qkv.size(2), 3 * heads);
    const int64_t out_n = q.size(2);
    const int id = dtype_code(qkv), td = dtype_code(c), od = dtype_code(q);
    void *ip = ptr(qkv), *cp = ptr(c), *sp = ptr(s), *qp = ptr(q), *kp = ptr(k), *vp = ptr(v);
    const mbrt_stream_t st = stream(a[7]);
    return call("mbrt_split_qkv_heads_rotary", [&] {
        return mbrt_split_qkv_heads_rotary(ip, id, cp, sp, td, qp, kp, vp, od, B, N, heads, D, out_n, st);
    });
    END_HANDLE_TH_ERRORS
}

// attention_ex(q, k, v, (B, H, n_q, n_k, D), (six strides), cos | None, sin | None, gate | None, gate_is_logit,
//              out, scale, p_precision, stream)
MBRT_PY(attention_ex) {
    HANDLE_TH_ERRORS
    count(n, 13);
    const at::Tensor &q = tensor(a[0]), &k = tensor(a[1]), &v = tensor(a[2]), &out = tensor(a[9]);
    const at::Tensor c = tensor_or_none(a[5]), s = tensor_or_none(a[6]), g = tensor_or_none(a[7]);
    int64_t z[11];
    for (int i = 0; i < 5; ++i) z[i] = integer(PyTuple_GET_ITEM(a[3], i));
    for (int i = 0; i < 6; ++i) z[5 + i] = integer(PyTuple_GET_ITEM(a[4], i));
    const int dt = dtype_code(q), td = dtype_or(c, MBRT_F32), gd = dtype_or(g, MBRT_F32), od = dtype_code(out);
    const int logit = truth(a[8]), pm = (int)integer(a[11]);
    void *qp = ptr(q), *kp = ptr(k), *vp = ptr(v), *cp = ptr(c), *sp = ptr(s), *gp = ptr(g), *op = ptr(out);
    const float scale = (float)number(a[10]);
    const mbrt_stream_t st = stream(a[12]);
    return call("mbrt_attention_ex", [&] {
        return mbrt_attention_ex(qp, kp, vp, dt, z[0], z[1], z[2], z[3], z[4], z[5], z[6], z[7], z[8], z[9], z[10], cp,
                                 sp, td, gp, gd, logit, op, od, scale, pm, st);
    });
    END_HANDLE_TH_ERRORS
}

// stft(x [B, L], window, hop, center, normalized, out, n_fft, win_length, stream)
MBRT_PY(stft) {
    HANDLE_TH_ERRORS
    count(n, 9);
    const at::Tensor &x = tensor(a[0]), &w = tensor(a[1]), &out = tensor(a[5]);
    contig({&x, &w, &out});
    const int64_t hop = integer(a[2]), n_fft = integer(a[6]), win = integer(a[7]);
    const int center = truth(a[3]), normalized = truth(a[4]);
    const int64_t B = x.size(0), L = x.size(1), wn = w.numel();
    const float *xp = static_cast<const float*>(ptr(x)), *wp = static_cast<const float*>(ptr(w));
    float* op = static_cast<float*>(ptr(out));
    const mbrt_stream_t st = stream(a[8]);
    return call("mbrt_stft", [&] { return mbrt_stft(xp, wp, op, B, L, n_fft, hop, win, wn, center, normalized, st); });
    END_HANDLE_TH_ERRORS
}

// istft(spec, window, hop, center, normalized, length, out, workspace, n_fft, win_length, stream)
MBRT_PY(istft) {
    HANDLE_TH_ERRORS
    count(n, 11);
    const at::Tensor &s = tensor(a[0]), &w = tensor(a[1]), &out = tensor(a[6]), &ws = tensor(a[7]);
    contig({&s, &w, &out});
    if (s.dim() != 4) raise(PyExc_ValueError, "istft: expected a spectrum [B, F, T, 2]");
    const int64_t hop = integer(a[2]), length = integer(a[5]), n_fft = integer(a[8]), win = integer(a[9]);
    const int center = truth(a[3]), normalized = truth(a[4]), dt = dtype_code(s);
    const int64_t B = s.size(0), F = s.size(1), T = s.size(2), wn = w.numel();
    const int64_t bytes = ws.numel() * (int64_t)ws.element_size();
    void *sp = ptr(s), *wsp = ptr(ws);
    const float* wp = static_cast<const float*>(ptr(w));
    float* op = static_cast<float*>(ptr(out));
    const mbrt_stream_t st = stream(a[10]);
    return call("mbrt_istft", [&] {
        return mbrt_istft(sp, dt, wp, op, B, F, T, n_fft, hop, win, wn, center, normalized, length, wsp, bytes, st);
    });
    END_HANDLE_TH_ERRORS
}

// chunk_accumulate(dest, weight_sum, src, window, offset, stream)
MBRT_PY(chunk_accumulate) {
    HANDLE_TH_ERRORS
    count(n, 6);
    const at::Tensor &d = tensor(a[0]), &ws = tensor(a[1]), &s = tensor(a[2]), &w = tensor(a[3]);
    contig({&d, &ws, &s, &w});
    const int64_t len = s.size(-1), L = d.size(-1), off = integer(a[4]);
    const int64_t channels = s.numel() / (len > 1 ? len : 1);
    float *dp = static_cast<float*>(ptr(d)), *wsp = static_cast<float*>(ptr(ws));
    const float *sp = static_cast<const float*>(ptr(s)), *wp = static_cast<const float*>(ptr(w));
    const mbrt_stream_t st = stream(a[5]);
    return call("mbrt_chunk_accumulate",
                [&] { return mbrt_chunk_accumulate(dp, wsp, sp, wp, channels, len, L, off, st); });
    END_HANDLE_TH_ERRORS
}

// init(MbrtError)
MBRT_PY(init) {
    HANDLE_TH_ERRORS
    count(n, 1);
    Py_INCREF(a[0]);
    Py_XDECREF(g_error);
    g_error = a[0];
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define MBRT_DEF(fname) {#fname, (PyCFunction)(void (*)(void))fname, METH_FASTCALL, nullptr}
PyMethodDef kMethods[] = {
    MBRT_DEF(init), MBRT_DEF(fill), MBRT_DEF(strided_copy), MBRT_DEF(pad), MBRT_DEF(cat), MBRT_DEF(rms_norm),
    MBRT_DEF(residual_add_rms_norm), MBRT_DEF(bias_act), MBRT_DEF(glu), MBRT_DEF(gate_merge), MBRT_DEF(softmax),
    MBRT_DEF(split_qkv_rotary), MBRT_DEF(attention_ex), MBRT_DEF(stft), MBRT_DEF(istft), MBRT_DEF(chunk_accumulate),
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef kModule = {PyModuleDef_HEAD_INIT, "_mbrt_calls", nullptr, -1, kMethods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__mbrt_calls(void) { return PyModule_Create(&kModule); }
