// Host path of the quantised linear layers in eager mode: what Linear.forward does between the model's call and the
// kernels -- argument checks, the memory of the result and of the int8 rows, the launches -- without the Python
// interpreter.  A layer of a few hundred tokens runs for 5 to 20 microseconds on the GPU, less than the two dozen Python
// calls and two ctypes calls of the general path take (77 x 3072 x 3072: 31 us a forward that way, 11 us this way).
//
//   bind(path)                  the kernels' library
//   linear(...)                 one layer: Linear.forward with its optional prologue, gate and residual
//   fanout(...)                 several layers that read the same tokens, quantised once
//   vector_fanout(...)          several small-batch layers that read the same rows, in one launch
//
// Every function takes the cases it can decide on cheaply and returns None for all others (tensors of other types,
// devices or layouts, operands that need a cast or a copy, errors): the caller then goes the general way in Python, which
// also words the errors.  Nothing is kept between calls.
//
// Everything that belongs to Python (arguments, the tensors' sizes and pointers) is read first; the allocations and the
// launches then run without the interpreter's lock, as behind ctypes and torch's own operators: a full hardware queue or an
// allocator that has to give memory back makes this thread wait, not the others.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/autocast_mode.h>
#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include "../../../include/i8f.h"
#include "../quant_lora_entry.hpp"
#include "../w8a16_rotated.hpp"

namespace {

// ---- the kernels' library -----------------------------------------------------------------
#define I8F_ENTRY_POINTS(X)                                                                                              \
    X(i8f_quant_rowwise) X(i8f_quant_rowwise_prologue) X(i8f_quant_rowwise_norm_modulate) X(i8f_quant_rowwise_rms_norm)  \
    X(i8f_quant_rowwise_concat_gelu) X(i8f_rotate128) X(i8f_linear_w8a8_gated) X(i8f_linear_w8a8_grouped) X(i8f_linear_w8a16_small_m) \
    X(i8f_linear_w8a16_small_m_grouped) X(i8f_internal_w8a16_rotated) X(i8f_linear_w8a8_lora) X(i8f_internal_quant_lora)
struct Library {
#define X(name) decltype(&::name) name = nullptr;
    I8F_ENTRY_POINTS(X)
#undef X
    bool bound = false;
} lib;

PyObject *bind(PyObject *, PyObject *arg) {
    const char *path = PyUnicode_AsUTF8(arg);
    if (!path) return nullptr;
    void *h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!h) return PyErr_Format(PyExc_RuntimeError, "cannot load %s: %s", path, dlerror());
#define X(name)                                                                                                    \
    if (!(lib.name = (decltype(lib.name))dlsym(h, #name)))                                                         \
        return PyErr_Format(PyExc_RuntimeError, "%s has no %s: build it again", path, #name);
    I8F_ENTRY_POINTS(X)
#undef X
    lib.bound = true;
    Py_RETURN_NONE;
}

// ---- arguments -----------------------------------------------------------------------------
int code_of(at::ScalarType t) {
    return t == at::kBFloat16 ? I8F_BF16 : t == at::kHalf ? I8F_F16 : t == at::kFloat ? I8F_F32 : -1;
}

// A plain torch.Tensor or Parameter (subclasses -- fake and wrapped tensors among them -- are the general path's).
const at::Tensor *tensor(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

bool aligned16(const at::Tensor &t) { return (uintptr_t)t.const_data_ptr() % 16 == 0; }

// The rows of t, all but its last dimension flattened, if they are a matrix of contiguous rows at one stride.
bool rows_of(const at::Tensor &t, int64_t &M, int64_t &K, int64_t &ld) {
    const int64_t d = t.dim();
    if (d < 1) return false;
    const auto sizes = t.sizes(), strides = t.strides();
    K = sizes[d - 1], M = 1, ld = K;
    if (K < 1 || (K > 1 && strides[d - 1] != 1)) return false;
    int64_t expect = -1;  // stride that the next outer dimension has to have
    for (int64_t i = d - 2; i >= 0; --i) {
        if (sizes[i] == 1) continue;
        if (sizes[i] == 0) return false;
        if (expect < 0) ld = strides[i];
        else if (strides[i] != expect) return false;
        expect = strides[i] * sizes[i];
        M *= sizes[i];
    }
    return ld >= K;
}

// A vector per leading index of x, shared by its tokens: [K], or [..., 1, K] with x's leading dimensions.
// K: the last dimension of what it is applied to (x itself or the layer's output).
bool broadcasts_over_tokens(const at::Tensor &x, int64_t K, const at::Tensor &v) {
    if (v.scalar_type() != x.scalar_type() || v.device() != x.device() || !v.is_contiguous() || x.dim() < 2) return false;
    if (v.dim() == 1) return v.size(0) == K;
    if (v.dim() != x.dim() || v.size(-1) != K || v.size(-2) != 1) return false;
    for (int64_t i = 0; i < x.dim() - 2; ++i)
        if (v.size(i) != x.size(i)) return false;
    return true;
}

// Weight, scale and bias of a layer as the kernels take them.
struct Layer {
    const int8_t *w = nullptr;
    const float *ws = nullptr;
    float ws_host = 0.0f;
    int mode = I8F_SCALE_TENSOR, bias_code = I8F_BF16;
    const void *bias = nullptr;
    int64_t N = 0, K = 0;
};

bool layer_of(PyObject *weight, PyObject *scale, PyObject *bias, bool per_row, const at::Device &dev, Layer &l) {
    const at::Tensor *w = tensor(weight);
    if (!w || w->scalar_type() != at::kChar || w->dim() != 2 || w->device() != dev || !w->is_contiguous()) return false;
    l.w = (const int8_t *)w->const_data_ptr(), l.N = w->size(0), l.K = w->size(1);
    if (l.N < 1) return false;
    if (PyFloat_Check(scale)) {
        if (per_row) return false;
        l.ws_host = (float)PyFloat_AS_DOUBLE(scale);
    } else {
        const at::Tensor *s = tensor(scale);
        if (!s || s->scalar_type() != at::kFloat || s->device() != dev || !s->is_contiguous() || s->numel() < 1) return false;
        if (per_row && s->numel() != l.N) return false;
        l.ws = (const float *)s->const_data_ptr();
        l.mode = per_row && s->numel() != 1 ? I8F_SCALE_ROW : I8F_SCALE_TENSOR;  // (one scale: element 0 counts)
    }
    if (bias != Py_None) {
        const at::Tensor *b = tensor(bias);
        if (!b || b->device() != dev || !b->is_contiguous() || b->numel() != l.N || (l.bias_code = code_of(b->scalar_type())) < 0) return false;
        l.bias = b->const_data_ptr();
    }
    return true;
}

at::Tensor empty(at::IntArrayRef size, at::ScalarType t, const at::Device &dev) {
    return at::detail::empty_cuda(size, t, dev, std::nullopt);
}

// The size of a layer's output on x's tokens: x's leading dimensions and N columns.
using Size = c10::SmallVector<int64_t, 6>;
Size output_size(const at::Tensor &x, int64_t N) {
    Size size(x.sizes().begin(), x.sizes().end());
    size.back() = N;
    return size;
}

// The interpreter's lock is released while one of these lives.  (Taking it again ends the thread where the interpreter has
// been shut down meanwhile, by an unwinding that has to be let out of here.)
struct WithoutGil {
    PyThreadState *state = PyEval_SaveThread();
    ~WithoutGil() noexcept(false) { PyEval_RestoreThread(state); }
};

struct Stream {
    void *handle;
    bool ok;
    explicit Stream(const at::Device &dev) : handle(nullptr), ok(dev.is_cuda() && dev.index() == c10::hip::current_device()) {
        if (ok) handle = (void *)c10::hip::getCurrentHIPStream(dev.index()).stream();
    }
};

struct Owned {  // a new reference
    PyObject *p = nullptr;
    ~Owned() { Py_XDECREF(p); }
};

// ---- 16 rows or fewer: W8A16 ----------------------------------------------------------------
PyObject *small_m(const at::Tensor &x, int64_t M, int64_t K, int64_t ld, const Layer &l, bool rotate, void *stream) {
    const at::ScalarType type = x.scalar_type();
    const at::Device dev = x.device();
    const int dt = code_of(type);
    const void *xp = x.const_data_ptr();
    const Size size = output_size(x, l.N);
    at::Tensor rotated, y;
    bool done = false;
    {
        const WithoutGil released;
        y = empty(size, type, dev);
        void *out = y.data_ptr();
        done = rotate && !lib.i8f_internal_w8a16_rotated(xp, dt, M, K, ld, l.w, l.ws, l.ws_host, l.mode, l.bias, l.bias_code, out, l.N, stream);
        bool ready = true;
        if (rotate && !done) {
            rotated = empty({M, K}, type, dev);
            ready = !lib.i8f_rotate128(xp, dt, M, K, ld, rotated.data_ptr(), stream);
            xp = rotated.const_data_ptr(), ld = K;
        }
        if (ready && !done) done = !lib.i8f_linear_w8a16_small_m(xp, dt, M, K, ld, l.w, l.ws, l.ws_host, l.mode, l.bias, l.bias_code, out, l.N, stream);
    }
    if (!done) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
}

// ---- a dynamic LoRA on the layer ---------------------------------------------------------------
// Its first product by the launch that quantises x, the second inside the GEMM.  Two launches: with the BLAS library's call
// between them and the interpreter's part of it all, the host took 63 us a layer and the GPU waited for it below 2000 rows.
//
// linear_lora(x, weight, scale, bias, per_row, order, lora_A, lora_B, lora_alpha): a layer of more than 16 rows with the factors
// of a dynamic LoRA, no rotation, nothing in front and nothing behind.
PyObject *linear_lora(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 9) return PyErr_Format(PyExc_TypeError, "linear_lora takes 9 arguments, got %zd", n);
    const at::Tensor *xt = tensor(a[0]), *A = tensor(a[6]), *B = tensor(a[7]);
    if (!lib.bound || !xt || !A || !B || A->dim() != 2 || !xt->is_cuda()) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int64_t R = A->size(0);  // (the GEMM's LoRA epilogue takes ranks in steps of 16 up to 64)
    int64_t M, K, ld;
    if (R % 16 || R < 16 || R > 64 || !rows_of(x, M, K, ld)) Py_RETURN_NONE;
    // (every 16 rows read the factor once more: 16384 rows are as many as were measured.  There a 3072 x 3072 layer of rank 16 takes
    // 160 us where the quantiser, the BLAS library's product and the GEMM take 174, of rank 64 178 and 181, 4096 x 4096 277 either way)
    if (M > 16384 || K % 128 || K > (R > 32 ? 4096 : 6144) || ld % 8) Py_RETURN_NONE;
    Layer l;
    const at::ScalarType type = x.scalar_type();
    if ((type != at::kBFloat16 && type != at::kHalf) || !layer_of(a[1], a[2], a[3], a[4] == Py_True, x.device(), l)) Py_RETURN_NONE;
    for (const at::Tensor *f : {A, B})
        if (f->scalar_type() != type || f->device() != x.device() || f->dim() != 2 || !f->is_contiguous() || !aligned16(*f)) Py_RETURN_NONE;
    if (A->size(1) != K || B->size(0) != l.N || B->size(1) != R) Py_RETURN_NONE;
    if (K != l.K || l.N % 8 || !aligned16(x) || (uintptr_t)l.w % 16 || (l.mode == I8F_SCALE_ROW && (uintptr_t)l.ws % 16) || (uintptr_t)l.bias % 16 ||
        l.N * K >= (1ll << 31))
        Py_RETURN_NONE;
    if (at::autocast::is_autocast_enabled(at::kCUDA)) Py_RETURN_NONE;  // (the product's type is then the context's)
    float alpha = 0.0f;
    const bool has_alpha = a[8] != Py_None;
    if (has_alpha) {
        if (!PyFloat_CheckExact(a[8]) && !PyLong_CheckExact(a[8])) Py_RETURN_NONE;
        alpha = (float)PyFloat_AsDouble(a[8]);
        if (PyErr_Occurred()) return nullptr;
    }
    const Stream st(x.device());
    if (!st.ok) Py_RETURN_NONE;
    const int order = (int)PyLong_AsLong(a[5]);
    const at::Device dev = x.device();
    const Size size = output_size(x, l.N);
    const int dt = code_of(type);
    const void *xp = x.const_data_ptr(), *ap = A->const_data_ptr(), *bp = B->const_data_ptr();
    at::Tensor scratch, y;
    int rc;
    {
        const WithoutGil released;
        const int64_t q_bytes = (M * K + 255) / 256 * 256, t_bytes = (2 * M * R + 255) / 256 * 256;
        scratch = empty({q_bytes + t_bytes + 4 * M}, at::kByte, dev);
        int8_t *q = (int8_t *)scratch.data_ptr();
        void *t = q + q_bytes;
        float *qs = (float *)(q + q_bytes + t_bytes);
        y = empty(size, type, dev);
        rc = lib.i8f_internal_quant_lora(xp, dt, M, K, ld, ap, R, q, qs, t, st.handle);
        if (!rc)
            rc = lib.i8f_linear_w8a8_lora(q, qs, l.w, l.ws, l.ws_host, l.mode, l.bias, l.bias_code, t, bp, R, has_alpha, alpha, y.data_ptr(), dt, M,
                                          l.N, K, order, st.handle);
    }
    if (rc) Py_RETURN_NONE;
    return THPVariable_Wrap(std::move(y));
}

constexpr int MAX_FANOUT = 8;

PyObject *list_of(at::Tensor *y, Py_ssize_t count) {
    PyObject *out = PyList_New(count);
    if (!out) return nullptr;
    for (Py_ssize_t i = 0; i < count; ++i) {
        PyObject *o = THPVariable_Wrap(std::move(y[i]));
        if (!o) {
            Py_DECREF(out);
            return nullptr;
        }
        PyList_SET_ITEM(out, i, o);
    }
    return out;
}

// The W8A8 form of linear and fanout, whose arguments these are; a gate or a residual for one layer only.
PyObject *w8a8(PyObject *const *a, const at::Tensor &x, int64_t M, int64_t K, int64_t ld, const Layer *l, int count, const Stream &st) {
    const int dt = code_of(x.scalar_type()), order = (int)PyLong_AsLong(a[7]), kind = (int)PyLong_AsLong(a[8]);
    const bool rotate = a[5] == Py_True, fused_add = a[13] == Py_True, gated = a[14] != Py_None, with_residual = a[15] != Py_None;
    if (count != 1 && (gated || with_residual)) Py_RETURN_NONE;

    // the operation in front of the layer and its operands
    const at::Tensor *s = nullptr, *t = nullptr, *w = nullptr;
    int64_t V = 1, Kall = K, Kb = 0, ldb = 0;
    float eps = 0.0f;
    if (kind == I8F_PRO_NORM_MODULATE || kind == I8F_PRO_RMS_NORM) {
        eps = (float)PyFloat_AsDouble(a[11]);
        if (PyErr_Occurred()) return nullptr;
    }
    if (kind == I8F_PRO_MODULATE || kind == I8F_PRO_NORM_MODULATE || kind == I8F_PRO_RMS_NORM) {
        s = a[9] == Py_None ? nullptr : tensor(a[9]), t = a[10] == Py_None ? nullptr : tensor(a[10]);
        if ((a[9] != Py_None && !s) || (a[10] != Py_None && !t) || (kind != I8F_PRO_RMS_NORM && !(s && t))) Py_RETURN_NONE;
        for (const at::Tensor *v : {s, t}) {
            if (!v) continue;
            if (!broadcasts_over_tokens(x, K, *v) || !aligned16(*v)) Py_RETURN_NONE;
            V = v->numel() / K;
        }
        if (s && t && s->sizes() != t->sizes()) Py_RETURN_NONE;
        if (V < 1 || M % V) Py_RETURN_NONE;
        if (kind != I8F_PRO_MODULATE && (K > 16384 || K % 16 || (M > 1 && ld % 8) || !aligned16(x))) Py_RETURN_NONE;
        if (kind == I8F_PRO_RMS_NORM && a[12] != Py_None) {
            w = tensor(a[12]);
            if (!w || w->scalar_type() != x.scalar_type() || w->dim() != 1 || w->size(0) != K || w->device() != x.device() || !w->is_contiguous() ||
                !aligned16(*w))
                Py_RETURN_NONE;
        }
    } else if (kind == I8F_PRO_CONCAT_GELU) {
        s = tensor(a[9]);
        int64_t Mb;
        if (!s || s->scalar_type() != x.scalar_type() || s->device() != x.device() || s->dim() != x.dim() || !rows_of(*s, Mb, Kb, ldb)) Py_RETURN_NONE;
        for (int64_t i = 0; i + 1 < x.dim(); ++i)
            if (s->size(i) != x.size(i)) Py_RETURN_NONE;
        Kall = K + Kb;
        if (K % 16 || Kb % 16 || Kall > 16384 || (M > 1 && (ld % 8 || ldb % 8)) || !aligned16(x) || !aligned16(*s) || (rotate && Kb % 128)) Py_RETURN_NONE;
    } else if (kind == I8F_PRO_SILU_GATE) {
        s = tensor(a[9]);
        if (!s || s->scalar_type() != x.scalar_type() || s->device() != x.device() || s->sizes() != x.sizes() || !s->is_contiguous()) Py_RETURN_NONE;
    } else if (kind != I8F_PRO_NONE && kind != I8F_PRO_GELU_TANH && kind != I8F_PRO_GELU_ERF) {
        Py_RETURN_NONE;
    }
    for (int i = 0; i < count; ++i)
        if (l[i].K != Kall) Py_RETURN_NONE;

    // what follows the layer
    const at::Tensor *gate = nullptr, *res = nullptr, *work = nullptr;
    int64_t gate_rows = 1;
    if (gated) {
        gate = tensor(a[14]);
        if (!gate || !broadcasts_over_tokens(x, l[0].N, *gate)) Py_RETURN_NONE;
        const int64_t vecs = gate->numel() / l[0].N;
        if (vecs < 1 || M % vecs) Py_RETURN_NONE;
        gate_rows = M / vecs;
    }
    if (with_residual) {
        res = tensor(a[15]);
        if (!res || res->scalar_type() != x.scalar_type() || res->device() != x.device() || res->dim() != x.dim() || !res->is_contiguous() ||
            res->numel() != M * l[0].N || res->size(-1) != l[0].N)
            Py_RETURN_NONE;
        for (int64_t i = 0; i + 1 < x.dim(); ++i)
            if (res->size(i) != x.size(i)) Py_RETURN_NONE;
    }
    Owned work_object;
    if (a[16] != Py_None) {   // (the narrowest layer has the fewest tiles: what it cannot use, none can)
        int64_t narrowest = l[0].N;
        for (int i = 1; i < count; ++i) narrowest = l[i].N < narrowest ? l[i].N : narrowest;
        work_object.p = PyObject_CallFunction(a[16], "OLLL", a[0], (long long)M, (long long)narrowest, (long long)Kall);
        if (!work_object.p) return nullptr;
        if (work_object.p != Py_None && !(work = tensor(work_object.p))) Py_RETURN_NONE;
    }

    const at::ScalarType type = x.scalar_type();
    const at::Device dev = x.device();
    Size size[MAX_FANOUT];
    for (int i = 0; i < count; ++i) size[i] = output_size(x, l[i].N);
    const auto address = [](const at::Tensor *o) { return o ? o->const_data_ptr() : nullptr; };
    const void *xp = x.const_data_ptr(), *sp = address(s), *tp = address(t), *wp = address(w), *gate_p = address(gate), *res_p = address(res);
    void *work_p = work ? work->data_ptr() : nullptr;
    const int64_t work_bytes = work ? work->numel() : 0;
    at::Tensor scratch, y[MAX_FANOUT];
    int rc;
    {
        const WithoutGil released;
        // one piece of memory for the int8 rows and, behind them, their scales; it goes back to the allocator when the call
        // returns, for work behind these kernels on the same stream
        const int64_t q_bytes = (M * Kall + 255) / 256 * 256;
        scratch = empty({q_bytes + 4 * M}, at::kByte, dev);
        int8_t *q = (int8_t *)scratch.data_ptr();
        float *qs = (float *)(q + q_bytes);
        for (int i = 0; i < count; ++i) y[i] = empty(size[i], type, dev);
        const int rb = rotate ? 128 : 0;
        switch (kind) {
        case I8F_PRO_NONE: rc = lib.i8f_quant_rowwise(xp, dt, M, K, ld, rb, q, qs, st.handle); break;
        case I8F_PRO_NORM_MODULATE:
            rc = lib.i8f_quant_rowwise_norm_modulate(xp, dt, M, K, ld, eps, sp, tp, M / V, fused_add, rb, q, qs, st.handle);
            break;
        case I8F_PRO_RMS_NORM: rc = lib.i8f_quant_rowwise_rms_norm(xp, dt, M, K, ld, eps, wp, sp, tp, M / V, fused_add, rb, q, qs, st.handle); break;
        case I8F_PRO_CONCAT_GELU: rc = lib.i8f_quant_rowwise_concat_gelu(xp, dt, M, K, ld, sp, Kb, ldb, rb, q, qs, st.handle); break;
        case I8F_PRO_SILU_GATE: rc = lib.i8f_quant_rowwise_prologue(xp, dt, M, K, ld, kind, sp, nullptr, 1, rb, q, qs, st.handle); break;
        default:
            rc = lib.i8f_quant_rowwise_prologue(xp, dt, M, K, ld, kind == I8F_PRO_MODULATE && fused_add ? (int)I8F_PRO_MODULATE_FUSED : kind, sp, tp,
                                                M / V, rb, q, qs, st.handle);
        }
        if (!rc && count == 1)
            rc = lib.i8f_linear_w8a8_gated(q, qs, l[0].w, l[0].ws, l[0].ws_host, l[0].mode, l[0].bias, l[0].bias_code, gate_p, gate_rows, res_p,
                                           y[0].data_ptr(), dt, M, l[0].N, l[0].K, order, work_p, work_bytes, st.handle);
        for (int first = 0, next; count > 1 && !rc && first < count; first = next) {  // layers of one form, a launch for as many as the library puts together
            i8f_linear_group g[I8F_MAX_LINEAR_GROUPS] = {};
            int bias_code = -1;
            for (next = first; next < count && next - first < I8F_MAX_LINEAR_GROUPS; ++next) {
                const Layer &o = l[next];
                if (o.N != l[first].N || o.mode != l[first].mode || (o.bias && bias_code >= 0 && o.bias_code != bias_code)) break;
                if (o.bias) bias_code = o.bias_code;
                i8f_linear_group &e = g[next - first];
                e.a = q, e.a_scale = qs, e.w = o.w, e.w_scale = o.ws, e.w_scale_host = o.ws_host, e.bias = o.bias, e.out = y[next].data_ptr(), e.M = M;
                e.rows_per_gate = 1;
            }
            rc = lib.i8f_linear_w8a8_grouped(g, next - first, l[first].mode, bias_code < 0 ? (int)I8F_BF16 : bias_code, dt, l[first].N, Kall, order, work_p,
                                             work_bytes, st.handle);
        }
    }
    if (rc) Py_RETURN_NONE;
    return count == 1 ? THPVariable_Wrap(std::move(y[0])) : list_of(y, count);
}

// linear(x, weight, scale, bias, per_row, rotate, small_rows, order, kind, mod_scale, mod_shift, eps, norm_weight, fused_add,
//        gate, residual, workspace): kind, an i8f_prologue, names what is applied to x inside the quantiser; workspace(x, M, N,
// K) gives the memory of the K split, which the layers of one call share, or None.  It is called once a W8A8 call has passed
// every check, never for 16 rows or fewer or for a call that goes the general way, which asks for its own: the memory stays
// with the stream, or with the graph that is being captured, together with the kernel that clears it.
PyObject *linear(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 17) return PyErr_Format(PyExc_TypeError, "linear takes 17 arguments, got %zd", n);
    const at::Tensor *xt = tensor(a[0]);
    if (!lib.bound || !xt || !xt->is_cuda()) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int dt = code_of(x.scalar_type());
    const bool per_row = a[4] == Py_True, rotate = a[5] == Py_True;
    int64_t M, K, ld;
    Layer l;
    if ((dt != I8F_BF16 && dt != I8F_F16) || !rows_of(x, M, K, ld) || !layer_of(a[1], a[2], a[3], per_row, x.device(), l)) Py_RETURN_NONE;
    const Stream st(x.device());
    if (!st.ok || (rotate && K % 128)) Py_RETURN_NONE;
    if (M <= PyLong_AsLongLong(a[6])) {
        if (PyLong_AsLong(a[8]) != I8F_PRO_NONE || a[14] != Py_None || a[15] != Py_None || K != l.K) Py_RETURN_NONE;
        return small_m(x, M, K, ld, l, rotate, st.handle);
    }
    return w8a8(a, x, M, K, ld, &l, 1, st);
}

// fanout(the arguments of linear): weight, scale, bias and per_row are tuples with an entry for each layer; a list of outputs.
// Not for 16 rows or fewer.
PyObject *fanout(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 17) return PyErr_Format(PyExc_TypeError, "fanout takes 17 arguments, got %zd", n);
    const at::Tensor *xt = tensor(a[0]);
    if (!lib.bound || !xt || !xt->is_cuda()) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int dt = code_of(x.scalar_type());
    const Py_ssize_t count = PyTuple_Check(a[1]) ? PyTuple_GET_SIZE(a[1]) : 0;
    int64_t M, K, ld;
    if ((dt != I8F_BF16 && dt != I8F_F16) || count < 2 || count > MAX_FANOUT || x.dim() < 2 || !rows_of(x, M, K, ld)) Py_RETURN_NONE;
    for (int i = 2; i <= 4; ++i)
        if (!PyTuple_Check(a[i]) || PyTuple_GET_SIZE(a[i]) != count) Py_RETURN_NONE;
    Layer l[MAX_FANOUT];
    for (Py_ssize_t i = 0; i < count; ++i)
        if (!layer_of(PyTuple_GET_ITEM(a[1], i), PyTuple_GET_ITEM(a[2], i), PyTuple_GET_ITEM(a[3], i), PyTuple_GET_ITEM(a[4], i) == Py_True, x.device(), l[i]))
            Py_RETURN_NONE;
    const Stream st(x.device());
    if (!st.ok || (a[5] == Py_True && K % 128) || M <= PyLong_AsLongLong(a[6])) Py_RETURN_NONE;
    return w8a8(a, x, M, K, ld, l, (int)count, st);
}

// vector_fanout(x, weights, scales, biases, per_row, rotate): tuples with one entry per layer -> list of outputs
PyObject *vector_fanout(PyObject *, PyObject *const *a, Py_ssize_t n) {
    if (n != 6) return PyErr_Format(PyExc_TypeError, "vector_fanout takes 6 arguments, got %zd", n);
    const at::Tensor *xt = tensor(a[0]);
    if (!lib.bound || !xt || !xt->is_cuda()) Py_RETURN_NONE;
    const at::Tensor &x = *xt;
    const int dt = code_of(x.scalar_type());
    int64_t M, K, ld;
    const Stream st(x.device());
    const Py_ssize_t count = PyTuple_Check(a[1]) ? PyTuple_GET_SIZE(a[1]) : 0;
    const bool rotate = a[5] == Py_True;
    if (!st.ok || (dt != I8F_BF16 && dt != I8F_F16) || !rows_of(x, M, K, ld) || M > 16 || count < 2 || count > I8F_MAX_LINEAR_GROUPS ||
        (rotate && K % 128))
        Py_RETURN_NONE;
    for (int i = 2; i <= 4; ++i)
        if (!PyTuple_Check(a[i]) || PyTuple_GET_SIZE(a[i]) != count) Py_RETURN_NONE;
    Layer l[I8F_MAX_LINEAR_GROUPS];
    int bias_code = -1;
    for (Py_ssize_t i = 0; i < count; ++i) {
        if (!layer_of(PyTuple_GET_ITEM(a[1], i), PyTuple_GET_ITEM(a[2], i), PyTuple_GET_ITEM(a[3], i), PyTuple_GET_ITEM(a[4], i) == Py_True,
                      x.device(), l[i]) ||
            l[i].K != K || l[i].mode != l[0].mode)
            Py_RETURN_NONE;
        if (l[i].bias) {
            if (bias_code >= 0 && bias_code != l[i].bias_code) Py_RETURN_NONE;
            bias_code = l[i].bias_code;
        }
    }
    const at::ScalarType type = x.scalar_type();
    const at::Device dev = x.device();
    const void *xp = x.const_data_ptr();
    Size size[I8F_MAX_LINEAR_GROUPS];
    for (Py_ssize_t i = 0; i < count; ++i) size[i] = output_size(x, l[i].N);
    at::Tensor rotated, y[I8F_MAX_LINEAR_GROUPS];
    bool done = true;
    {
        const WithoutGil released;
        if (rotate) {
            rotated = empty({M, K}, type, dev);
            done = !lib.i8f_rotate128(xp, dt, M, K, ld, rotated.data_ptr(), st.handle);
            xp = rotated.const_data_ptr(), ld = K;
        }
        i8f_small_m_group g[I8F_MAX_LINEAR_GROUPS];
        for (Py_ssize_t i = 0; i < count; ++i) {
            y[i] = empty(size[i], type, dev);
            g[i] = {xp, M, K, ld, l[i].w, l[i].ws, l[i].ws_host, l[i].bias, y[i].data_ptr(), l[i].N};
        }
        if (done)
            done = !lib.i8f_linear_w8a16_small_m_grouped(g, (int)count, dt, l[0].mode, bias_code < 0 ? (int)I8F_BF16 : bias_code, st.handle);
    }
    if (!done) Py_RETURN_NONE;
    return list_of(y, count);
}

// No C++ exception leaves an entry point: an allocator that has nothing left, say, becomes the general path's to report.
template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *guarded(PyObject *self, PyObject *const *a, Py_ssize_t n) {
    try {
        PyObject *r = F(self, a, n);
        if (PyErr_Occurred()) {  // an operand that is no number: the general path words it
            PyErr_Clear();
            Py_XDECREF(r);
            Py_RETURN_NONE;
        }
        return r;
    } catch (const std::exception &) {
        Py_RETURN_NONE;
    }
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, "bind(path): load the kernels' library"},
    {"linear", (PyCFunction)(void (*)(void))guarded<linear>, METH_FASTCALL, "one quantised layer, or None"},
    {"fanout", (PyCFunction)(void (*)(void))guarded<fanout>, METH_FASTCALL, "several quantised layers of the same tokens, or None"},
    {"linear_lora", (PyCFunction)(void (*)(void))guarded<linear_lora>, METH_FASTCALL, "one quantised layer with a dynamic LoRA, or None"},
    {"vector_fanout", (PyCFunction)(void (*)(void))guarded<vector_fanout>, METH_FASTCALL, "several small-batch layers, or None"},
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_i8f_host", "Native host path of the INT8 linear layers.", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__i8f_host(void) { return PyModule_Create(&module); }
