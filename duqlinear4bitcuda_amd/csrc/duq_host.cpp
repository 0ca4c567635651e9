// Host side of the Python ops in native code: the module _duq_host.
//
// A decode step of one layer is 3 us of kernel and 3.3 us of HIP's launch; through Python checks, torch.empty and a
// ctypes call it was 9.5 us, all of it host time.  What the Python layer does per call is done here instead: check
// the tensors, allocate the outputs, call the C ABI of libduq_hip.so (include/duq_hip.h) on torch's current stream.
//
// Every function takes the PLAIN case only (torch tensors of the expected dtype, device, size and layout, on the
// current device) and answers None for anything else: the caller's Python code then runs its own checks, which also
// word the errors.  Nothing is computed or kept here, outputs and staging come from torch's allocator, and the
// interpreter lock is given up around the calls that launch (a full queue makes a launch wait).
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <structmember.h>

#include <vector>

#include "../../include/duq_hip.h"

namespace {

using at::ScalarType;
using at::Tensor;

PyObject *g_packed = nullptr;  // class PackedQuantizedTensor
PyObject *g_check = nullptr;   // _lib.check(status, name): raises for a status other than 0
// byte offsets of PackedQuantizedTensor's __slots__ in its instances
enum Slot { kQ, kS, kZeros, kRowsum, kShadow, kSrc, kVersion, kClip, kQmax, kSlots };
const char *const kSlotNames[kSlots] = {"_q", "_s", "zeros_x", "rowsum_x", "shadow_x", "_src", "_src_version", "_clip", "_qmax"};
Py_ssize_t g_offset[kSlots];

inline PyObject *&slot(PyObject *packed, Slot s) { return *reinterpret_cast<PyObject **>(reinterpret_cast<char *>(packed) + g_offset[s]); }

struct Unlocked {  // the interpreter lock given up for the lifetime of the object
    PyThreadState *s = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(s); }
};

PyObject *none() { Py_RETURN_NONE; }

// The result, or the error that a status other than 0 is.
PyObject *finish(int status, const char *name, PyObject *result)
{
    if (!status) return result;
    Py_XDECREF(result);
    PyObject *r = PyObject_CallFunction(g_check, "is", status, name);
    Py_XDECREF(r);
    return nullptr;
}

// A C++ exception (an allocation that fails) as the Python exception torch makes of it.
template <class F>
PyObject *guarded(F f)
{
    HANDLE_TH_ERRORS
    return f();
    END_HANDLE_TH_ERRORS
}

int current_device()
{
    int d = -1;
    return hipGetDevice(&d) == hipSuccess ? d : -1;
}

// A contiguous tensor of that type on a GPU (on device `dev` unless that is negative), by its Python object.
const Tensor *plain(PyObject *o, ScalarType type, int dev)
{
    if (!THPVariable_CheckExact(o)) return nullptr;
    const Tensor &t = THPVariable_Unpack(o);
    if (!t.is_cuda() || t.scalar_type() != type || !t.is_contiguous() || (dev >= 0 && t.get_device() != dev)) return nullptr;
    return &t;
}

// An operand of `numel` values: its address in *p.  None is accepted where `optional`.
bool operand(PyObject *o, ScalarType type, int dev, int64_t numel, bool optional, const void **p)
{
    *p = nullptr;
    if (o == Py_None) return optional;
    const Tensor *t = plain(o, type, dev);
    if (!t || t->numel() != numel) return false;
    *p = t->const_data_ptr();
    return true;
}

// An output with the leading dimensions of `like` and `last` as the last one (last < 0: without it).
Tensor output(const Tensor &like, int64_t last, ScalarType type)
{
    c10::SmallVector<int64_t, 6> shape(like.sizes().begin(), like.sizes().end() - 1);
    if (last >= 0) shape.push_back(last);
    return Tensor(at::detail::empty_cuda(shape, type, like.device(), std::nullopt));
}

struct Scratch {  // device memory of the current stream for the length of one call
    c10::DataPtr data;
    explicit Scratch(uint64_t bytes)
    {
        if (bytes) data = c10::hip::HIPCachingAllocator::get()->allocate(bytes);
    }
    void *get() const { return data.get(); }
};

PyObject *wrap(Tensor &&t) { return THPVariable_Wrap(std::move(t)); }

duq_stream_t stream_of(PyObject *o) { return reinterpret_cast<duq_stream_t>(PyLong_AsVoidPtr(o)); }

const duq_half *half(const void *p) { return static_cast<const duq_half *>(p); }
const int32_t *i32(const void *p) { return static_cast<const int32_t *>(p); }
const float *f32(const void *p) { return static_cast<const float *>(p); }
template <class T>
T *out(const Tensor &t) { return t.defined() ? static_cast<T *>(t.mutable_data_ptr()) : nullptr; }

// Tensors as a tuple, None for an undefined one.
PyObject *tuple_of(std::initializer_list<Tensor> ts)
{
    PyObject *r = PyTuple_New(static_cast<Py_ssize_t>(ts.size()));
    Py_ssize_t i = 0;
    for (const Tensor &t : ts) PyTuple_SET_ITEM(r, i++, t.defined() ? THPVariable_Wrap(t) : none());
    return r;
}

// ---- one layer's prepared call from binary16 rows ----------------------------------------------------------
// What FusedDecode (the Python class) holds: the layer's buffers, checked once, as a duq_fused_layer.
struct FusedCall {
    PyObject_HEAD
    duq_fused_layer layer;
    int dev;
    int64_t max_rows;
    PyObject *names, *tensors;        // tuples: the buffers' names in the module and the tensors the call was made of
    std::vector<int64_t> *staging;    // bytes the library stages at M rows, -1: not asked yet
};

int64_t staging_of(FusedCall *c, int64_t M)
{
    std::vector<int64_t> &v = *c->staging;
    if (v.empty()) v.assign(static_cast<size_t>(c->max_rows) + 1, -1);
    int64_t &b = v[static_cast<size_t>(M)];
    if (b < 0) {
        const duq_fused_layer &l = c->layer;
        const uint32_t m = static_cast<uint32_t>(M);
        b = static_cast<int64_t>(l.mode == DUQ_EPI_SYM || l.mode == DUQ_EPI_SYM_DUAL
                                     ? duq_quantize_linear4bit_workspace_bytes(m, l.N, l.K)
                                     : duq_quantize_linear4bit_asym_workspace_bytes(l.mode, m, l.N, l.K));
    }
    return b;
}

// Whether `buffers` (the module's dict) still holds the tensors the call was made of, where it found them.
bool still_current(FusedCall *c, PyObject *buffers)
{
    const Py_ssize_t n = PyTuple_GET_SIZE(c->names);
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject *t = PyDict_GetItemWithError(buffers, PyTuple_GET_ITEM(c->names, i));
        if ((t ? t : Py_None) != PyTuple_GET_ITEM(c->tensors, i)) return false;
    }
    return THPVariable_Unpack(PyTuple_GET_ITEM(c->tensors, 0)).const_data_ptr() == c->layer.w;
}

PyObject *run_rows(FusedCall *c, PyObject *buffers, const Tensor &x, float clip, int qmax)
{
    duq_fused_layer l = c->layer;
    if (x.dim() == 0 || x.size(-1) != static_cast<int64_t>(l.K) || x.get_device() != c->dev || l.K % 64) return none();
    const int64_t M = x.numel() / l.K;
    if (M < 1 || M > c->max_rows || current_device() != c->dev) return none();
    // more than 64 rows of a layer with a 6-bit float shadow: the Python side decides which path they take
    static PyObject *const shadow_name = PyUnicode_InternFromString("weight_shadow");
    if (M > 64) {
        PyObject *s = PyDict_GetItemWithError(buffers, shadow_name);
        if (s && s != Py_None) return none();
    }
    const int64_t bytes = staging_of(c, M);
    l.clip = clip;
    l.qmax = qmax;
    Tensor y = output(x, l.N, ScalarType::Half);
    Scratch ws(static_cast<uint64_t>(bytes));
    int st;
    {
        Unlocked u;
        st = duq_quantize_linear4bit_forward_layer(&l, half(x.const_data_ptr()), static_cast<uint32_t>(M), out<duq_half>(y),
                                                   ws.get(), static_cast<uint64_t>(bytes),
                                                   c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(c->dev)).stream());
    }
    if (st) return finish(st, "quantize_linear4bit_forward", nullptr);
    return wrap(std::move(y));
}

// take(buffers, packed): the layer's result for a PackedQuantizedTensor that was handed on unquantized
PyObject *fused_take(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    FusedCall *c = reinterpret_cast<FusedCall *>(self);
    if (n != 2 || !PyDict_Check(a[0]) || reinterpret_cast<PyObject *>(Py_TYPE(a[1])) != g_packed) return none();
    PyObject *src = slot(a[1], kSrc), *version = slot(a[1], kVersion), *clip = slot(a[1], kClip), *qmax = slot(a[1], kQmax);
    if (!src || !version || !clip || !qmax || !PyFloat_Check(clip) || !PyLong_Check(qmax)) return none();
    const Tensor *x = plain(src, ScalarType::Half, c->dev);
    if (!x || x->is_inference() || static_cast<long>(x->_version()) != PyLong_AsLong(version) || !still_current(c, a[0])) return none();
    const Tensor held = *x;  // (another thread may quantize the packed tensor, which drops its rows)
    return guarded([&] { return run_rows(c, a[0], held, static_cast<float>(PyFloat_AS_DOUBLE(clip)), static_cast<int>(PyLong_AsLong(qmax))); });
}

// take_rows(buffers, x): the same for a layer with its own quantizer
PyObject *fused_take_rows(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    FusedCall *c = reinterpret_cast<FusedCall *>(self);
    if (n != 2 || !PyDict_Check(a[0])) return none();
    const Tensor *x = plain(a[1], ScalarType::Half, c->dev);
    if (!x || reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16 || !still_current(c, a[0])) return none();
    return guarded([&] { return run_rows(c, a[0], *x, 1.0f, 6); });
}

// FusedCall(mode, N, K, device index, max_rows, addresses of (w, s1, z1, s2, z2, adj1, adj2, bias), names, tensors)
PyObject *fused_new(PyTypeObject *type, PyObject *args, PyObject *)
{
    int mode, dev;
    unsigned N, K;
    long long max_rows;
    PyObject *addr, *names, *tensors;
    if (!PyArg_ParseTuple(args, "iIIiLO!O!O!", &mode, &N, &K, &dev, &max_rows, &PyTuple_Type, &addr, &PyTuple_Type, &names,
                          &PyTuple_Type, &tensors))
        return nullptr;
    const Py_ssize_t n = PyTuple_GET_SIZE(names);
    if (PyTuple_GET_SIZE(addr) != 8 || n < 1 || PyTuple_GET_SIZE(tensors) != n || !THPVariable_Check(PyTuple_GET_ITEM(tensors, 0)) ||
        max_rows < 1 || max_rows > 65536) {
        PyErr_SetString(PyExc_ValueError, "FusedCall: eight addresses, and a tensor (the weight first) for every name");
        return nullptr;
    }
    void *p[8];
    for (int i = 0; i < 8; ++i) {
        PyObject *o = PyTuple_GET_ITEM(addr, i);
        p[i] = o == Py_None ? nullptr : PyLong_AsVoidPtr(o);
        if (PyErr_Occurred()) return nullptr;
    }
    FusedCall *c = reinterpret_cast<FusedCall *>(type->tp_alloc(type, 0));
    if (!c) return nullptr;
    c->layer = duq_fused_layer{mode, 1.0f, 6, N, K, static_cast<const uint8_t *>(p[0]), half(p[1]), half(p[2]), half(p[3]),
                               half(p[4]), i32(p[5]), i32(p[6]), half(p[7])};
    c->dev = dev;
    c->max_rows = max_rows;
    Py_INCREF(names);
    Py_INCREF(tensors);
    c->names = names;
    c->tensors = tensors;
    c->staging = new std::vector<int64_t>();
    return reinterpret_cast<PyObject *>(c);
}

void fused_dealloc(PyObject *self)
{
    FusedCall *c = reinterpret_cast<FusedCall *>(self);
    Py_XDECREF(c->names);
    Py_XDECREF(c->tensors);
    delete c->staging;
    Py_TYPE(self)->tp_free(self);
}

PyMethodDef g_fused_methods[] = {
    {"take", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fused_take)), METH_FASTCALL, nullptr},
    {"take_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fused_take_rows)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};
PyTypeObject g_fused_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// ---- quantizers --------------------------------------------------------------------------------------------

// defer(x, rows at most, shadow, rows from which it is written, clip, qmax): the PackedQuantizedTensor that hands x
// on unquantized, None for inputs that are to be quantized now (the rule: SymQuantizer.forward)
PyObject *m_defer(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 6) return none();
    const Tensor *x = plain(a[0], ScalarType::Half, -1);
    if (!x || x->dim() == 0 || x->is_inference() || !PyLong_Check(a[1])) return none();  // (inference tensors count no versions)
    const int64_t cols = x->size(-1), numel = x->numel();
    if (cols % 64 || numel <= 0 || numel > PyLong_AsLongLong(a[1]) * cols || reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16)
        return none();
    if (a[2] != Py_False && cols % 128 == 0 && (!PyLong_Check(a[3]) || numel >= PyLong_AsLongLong(a[3]) * cols)) return none();
    PyTypeObject *type = reinterpret_cast<PyTypeObject *>(g_packed);
    PyObject *p = type->tp_alloc(type, 0);
    if (!p) return nullptr;
    for (Slot s : {kQ, kS, kZeros, kRowsum, kShadow}) slot(p, s) = none();
    auto put = [&](Slot s, PyObject *v) {
        Py_INCREF(v);
        slot(p, s) = v;
    };
    put(kSrc, a[0]);
    slot(p, kVersion) = PyLong_FromLong(static_cast<long>(x->_version()));
    put(kClip, a[4]);
    put(kQmax, a[5]);
    return p;
}

// quantize_rows(x, kind, with codes, with shadow, clip, qmax, stream); kind 0 symmetric, 1 asymmetric, 2 asymmetric
// signed-shifted: (codes[, shadow], scales[, zeros[, row sums]]), codes None where not asked for
PyObject *m_quantize_rows(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 7 || !PyFloat_Check(a[4]) || !PyLong_Check(a[5])) return none();
    const Tensor *x = plain(a[0], ScalarType::Half, -1);
    if (!x || x->dim() == 0 || x->size(-1) == 0) return none();
    const long kind = PyLong_AsLong(a[1]);
    const bool with_q = a[2] == Py_True, shadow = a[3] == Py_True;
    const float clip = static_cast<float>(PyFloat_AS_DOUBLE(a[4]));
    const int qmax = static_cast<int>(PyLong_AsLong(a[5]));
    const duq_stream_t st = stream_of(a[6]);
    return guarded([&]() -> PyObject * {
        const int64_t cols = x->size(-1), rows64 = x->numel() / cols;
        if (rows64 > UINT32_MAX || cols > UINT32_MAX) return none();
        const uint32_t rows = static_cast<uint32_t>(rows64), K = static_cast<uint32_t>(cols);
        Tensor q, b, z, r, s = output(*x, 1, ScalarType::Half);
        if (with_q) q = output(*x, cols / 2, ScalarType::Byte);
        if (shadow) b = output(*x, cols * 3 / 4, ScalarType::Byte);
        if (kind) z = output(*x, 1, ScalarType::Half);
        if (kind == 2) r = output(*x, -1, ScalarType::Int);
        const duq_half *px = half(x->const_data_ptr());
        int e;
        {
            Unlocked u;
            if (shadow)
                e = kind ? duq_quantize_rows_asym_bf6(px, rows, K, out<uint8_t>(q), out<uint8_t>(b), out<duq_half>(s), out<duq_half>(z),
                                                      out<int32_t>(r), st)
                         : duq_quantize_rows_sym_bf6(px, rows, K, clip, qmax, out<uint8_t>(q), out<uint8_t>(b), out<duq_half>(s), st);
            else if (kind == 2)
                e = duq_quantize_rows_asym_shifted(px, rows, K, out<uint8_t>(q), out<duq_half>(s), out<duq_half>(z), out<int32_t>(r), st);
            else
                e = kind ? duq_quantize_rows_asym(px, rows, K, out<uint8_t>(q), out<duq_half>(s), out<duq_half>(z), st)
                         : duq_quantize_rows_sym(px, rows, K, clip, qmax, out<uint8_t>(q), out<duq_half>(s), st);
        }
        static const char *const names[2][3] = {{"quantize_rows_sym", "quantize_rows_asym", "quantize_rows_asym_shifted"},
                                                {"quantize_rows_sym_bf6", "quantize_rows_asym_bf6", "quantize_rows_asym_bf6"}};
        if (e) return finish(e, names[shadow][kind], nullptr);
        if (shadow) return kind == 0 ? tuple_of({q, b, s}) : kind == 1 ? tuple_of({q, b, s, z}) : tuple_of({q, b, s, z, r});
        return kind == 0 ? tuple_of({q, s}) : kind == 1 ? tuple_of({q, s, z}) : tuple_of({q, s, z, r});
    });
}

// quantize_rows_8bit(x, stream): (codes, scales, zeros)
PyObject *m_quantize_rows_8bit(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 2) return none();
    const Tensor *x = plain(a[0], ScalarType::Float, -1);
    if (!x || x->dim() == 0 || x->size(-1) == 0) return none();
    const duq_stream_t st = stream_of(a[1]);
    return guarded([&]() -> PyObject * {
        const int64_t cols = x->size(-1), rows = x->numel() / cols;
        if (rows > UINT32_MAX || cols > UINT32_MAX) return none();
        Tensor q = output(*x, cols, ScalarType::Char), s = output(*x, 1, ScalarType::Float), z = output(*x, 1, ScalarType::Float);
        int e;
        {
            Unlocked u;
            e = duq_quantize_rows_asym_8bit(f32(x->const_data_ptr()), static_cast<uint32_t>(rows), static_cast<uint32_t>(cols),
                                            out<int8_t>(q), out<float>(s), out<float>(z), st);
        }
        return e ? finish(e, "quantize_rows_asym_8bit", nullptr) : tuple_of({q, s, z});
    });
}

// ---- GEMM + dequant ----------------------------------------------------------------------------------------

// linear4(mode, xq, scale_x, zeros_x, w, w_scale_1, w_zeros_1, w_scale_2, w_zeros_2, bias, rowsum_x, w_rowsum_adj,
//         shadows, stream): modes 0 - 4 on packed codes, or with `shadows` on the 6-bit float shadows of both operands
PyObject *m_linear4(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 14 || !PyLong_Check(a[0])) return none();
    const int mode = static_cast<int>(PyLong_AsLong(a[0]));
    const bool shadows = a[12] == Py_True;
    const Tensor *x = plain(a[1], ScalarType::Byte, -1);
    if (!x || x->dim() == 0 || x->size(-1) == 0) return none();
    const int dev = static_cast<int>(x->get_device());
    const Tensor *w = plain(a[4], ScalarType::Byte, dev);
    if (!w || w->dim() != 2 || w->size(1) != x->size(-1) || !THPVariable_CheckExact(a[5])) return none();
    const int64_t kb = x->size(-1), M = x->numel() / kb;
    const int64_t N = shadows ? THPVariable_Unpack(a[5]).numel() : w->size(0);
    if (shadows && (kb % 96 || w->size(0) != (N + 31) / 32 * 32)) return none();
    const int64_t K = shadows ? kb * 4 / 3 : kb * 2;
    if (M > UINT32_MAX || N > UINT32_MAX || K > UINT32_MAX) return none();
    const void *p[12] = {};
    const bool rowsum = mode == DUQ_EPI_ASYM_ROWSUM;
    if (!operand(a[2], ScalarType::Half, dev, M, false, &p[2]) || !operand(a[3], ScalarType::Half, dev, M, !rowsum, &p[3]) ||
        !operand(a[10], ScalarType::Int, dev, M, !rowsum, &p[10]) || !operand(a[11], ScalarType::Int, dev, N, !rowsum, &p[11]))
        return none();
    for (int k = 5; k < 10; ++k)
        if (!operand(a[k], ScalarType::Half, dev, N, k != 5 && !(rowsum && k == 6), &p[k])) return none();
    const duq_stream_t st = stream_of(a[13]);
    return guarded([&]() -> PyObject * {
        Tensor y = output(*x, N, ScalarType::Half);
        const uint8_t *px = static_cast<const uint8_t *>(x->const_data_ptr()), *pw = static_cast<const uint8_t *>(w->const_data_ptr());
        const uint32_t m = static_cast<uint32_t>(M), nn = static_cast<uint32_t>(N), k = static_cast<uint32_t>(K);
        int e;
        {
            Unlocked u;
            if (shadows)
                e = duq_linear4bit_forward_bf6(mode, px, half(p[2]), half(p[3]), i32(p[10]), pw, half(p[5]), half(p[6]), half(p[7]),
                                               half(p[8]), i32(p[11]), half(p[9]), m, nn, k, out<duq_half>(y), st);
            else if (rowsum)
                e = duq_linear4bit_forward_rowsum(px, half(p[2]), half(p[3]), i32(p[10]), pw, half(p[5]), half(p[6]), i32(p[11]),
                                                  half(p[9]), m, nn, k, out<duq_half>(y), st);
            else
                e = duq_linear4bit_forward(mode, px, half(p[2]), half(p[3]), pw, half(p[5]), half(p[6]), half(p[7]), half(p[8]),
                                           half(p[9]), m, nn, k, out<duq_half>(y), st);
        }
        if (e) return finish(e, shadows ? "linear4bit_forward_bf6" : rowsum ? "linear4bit_forward_rowsum" : "linear4bit_forward", nullptr);
        return wrap(std::move(y));
    });
}

// linear4_batched(mode, xq, scale_x, zeros_x, w, w_scale_1, w_zeros_1, w_scale_2, w_zeros_2, bias, stream)
PyObject *m_linear4_batched(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 11 || !PyLong_Check(a[0])) return none();
    const int mode = static_cast<int>(PyLong_AsLong(a[0]));
    const Tensor *x = plain(a[1], ScalarType::Byte, -1);
    if (!x || x->dim() != 3) return none();
    const int dev = static_cast<int>(x->get_device());
    const Tensor *w = plain(a[4], ScalarType::Byte, dev);
    if (!w || w->dim() != 3 || w->size(0) != x->size(0) || w->size(2) != x->size(2)) return none();
    const int64_t b = x->size(0), M = x->size(1), N = w->size(1), K = x->size(2) * 2;
    if (b > UINT32_MAX || M > UINT32_MAX || N > UINT32_MAX || K > UINT32_MAX) return none();
    const void *p[10] = {};
    if (!operand(a[2], ScalarType::Half, dev, b * M, false, &p[2]) || !operand(a[3], ScalarType::Half, dev, b * M, true, &p[3])) return none();
    for (int k = 5; k < 10; ++k)
        if (!operand(a[k], ScalarType::Half, dev, b * N, k != 5, &p[k])) return none();
    const duq_stream_t st = stream_of(a[10]);
    return guarded([&]() -> PyObject * {
        Tensor y = output(*x, N, ScalarType::Half);
        int e;
        {
            Unlocked u;
            e = duq_batch_linear4bit_forward(mode, static_cast<const uint8_t *>(x->const_data_ptr()), half(p[2]), half(p[3]),
                                             static_cast<const uint8_t *>(w->const_data_ptr()), half(p[5]), half(p[6]), half(p[7]),
                                             half(p[8]), half(p[9]), static_cast<uint32_t>(b), static_cast<uint32_t>(M),
                                             static_cast<uint32_t>(N), static_cast<uint32_t>(K), out<duq_half>(y), st);
        }
        if (e) return finish(e, "batch_linear4bit_forward", nullptr);
        return wrap(std::move(y));
    });
}

// linear8(x, scale_x, zeros_x, w, w_tiled, w_scale, w_zeros, bias, N, stream): int8 codes with their scales and zeros
// (w_tiled not None: the GEMM reads that copy and w is not looked at), or float32 rows (scale_x and zeros_x None) that
// the call quantizes first
PyObject *m_linear8(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 10 || !PyLong_Check(a[8])) return none();
    const bool quantize = a[1] == Py_None;
    const Tensor *x = plain(a[0], quantize ? ScalarType::Float : ScalarType::Char, -1);
    if (!x || x->dim() == 0 || x->numel() == 0) return none();
    const int dev = static_cast<int>(x->get_device());
    const int64_t K = x->size(-1), M = x->numel() / K, N = PyLong_AsLongLong(a[8]);
    if (N <= 0 || M > UINT32_MAX || N > UINT32_MAX || K > UINT32_MAX) return none();
    const void *p[8] = {};
    if (!operand(a[1], ScalarType::Float, dev, M, quantize, &p[1]) || !operand(a[2], ScalarType::Float, dev, M, quantize, &p[2]) ||
        !operand(a[3], ScalarType::Char, dev, N * K, !quantize, &p[3]) ||
        !operand(a[4], ScalarType::Char, dev, (N + 31) / 32 * 32 * K, true, &p[4]) || (!p[3] && !p[4]) ||
        !operand(a[5], ScalarType::Float, dev, N, false, &p[5]) || !operand(a[6], ScalarType::Float, dev, N, false, &p[6]) ||
        !operand(a[7], ScalarType::Float, dev, N, true, &p[7]))
        return none();
    if (p[3] && THPVariable_Unpack(a[3]).dim() != 2) return none();
    const duq_stream_t st = stream_of(a[9]);
    return guarded([&]() -> PyObject * {
        Tensor y = output(*x, N, ScalarType::Float);
        const uint32_t m = static_cast<uint32_t>(M), nn = static_cast<uint32_t>(N), k = static_cast<uint32_t>(K);
        const int8_t *w = static_cast<const int8_t *>(p[3]), *wt = static_cast<const int8_t *>(p[4]);
        const uint64_t bytes = quantize ? duq_quantize_linear8bit_workspace_bytes(m, k) : 0;
        Scratch ws(bytes);
        int e;
        {
            Unlocked u;
            if (quantize)
                e = duq_quantize_linear8bit_forward(f32(x->const_data_ptr()), w, wt, f32(p[5]), f32(p[6]), f32(p[7]), m, nn, k,
                                                    out<float>(y), ws.get(), bytes, st);
            else
                e = (wt ? duq_linear8bit_forward_tiled : duq_linear8bit_forward)(
                    static_cast<const int8_t *>(x->const_data_ptr()), f32(p[1]), f32(p[2]), wt ? wt : w, f32(p[5]), f32(p[6]),
                    f32(p[7]), m, nn, k, out<float>(y), st);
        }
        if (e) return finish(e, quantize ? "quantize_linear8bit_forward" : "linear8bit_forward", nullptr);
        return wrap(std::move(y));
    });
}

// setup(PackedQuantizedTensor, check): the class defer() makes instances of, and what raises for a status
PyObject *m_setup(PyObject *, PyObject *args)
{
    PyObject *cls, *check;
    if (!PyArg_ParseTuple(args, "O!O", &PyType_Type, &cls, &check)) return nullptr;
    for (int i = 0; i < kSlots; ++i) {
        PyObject *d = PyDict_GetItemString(reinterpret_cast<PyTypeObject *>(cls)->tp_dict, kSlotNames[i]);
        if (!d || Py_TYPE(d) != &PyMemberDescr_Type) {
            PyErr_Format(PyExc_TypeError, "%s is not a slot of the class", kSlotNames[i]);
            return nullptr;
        }
        g_offset[i] = reinterpret_cast<PyMemberDescrObject *>(d)->d_member->offset;
    }
    Py_INCREF(cls);
    Py_INCREF(check);
    g_packed = cls;
    g_check = check;
    Py_RETURN_NONE;
}

#define FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(fn)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FAST("defer", m_defer),
                           FAST("quantize_rows", m_quantize_rows),
                           FAST("quantize_rows_8bit", m_quantize_rows_8bit),
                           FAST("linear4", m_linear4),
                           FAST("linear4_batched", m_linear4_batched),
                           FAST("linear8", m_linear8),
                           {"setup", m_setup, METH_VARARGS, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_duq_host", "host side of the ops (csrc/duq_host.cpp)", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__duq_host(void)
{
    g_fused_type.tp_name = "_duq_host.FusedCall";
    g_fused_type.tp_basicsize = sizeof(FusedCall);
    g_fused_type.tp_flags = Py_TPFLAGS_DEFAULT;
    g_fused_type.tp_new = fused_new;
    g_fused_type.tp_dealloc = fused_dealloc;
    g_fused_type.tp_methods = g_fused_methods;
    if (PyType_Ready(&g_fused_type) < 0) return nullptr;
    PyObject *m = PyModule_Create(&g_module);
    if (!m) return nullptr;
    Py_INCREF(&g_fused_type);
    if (PyModule_AddObject(m, "FusedCall", reinterpret_cast<PyObject *>(&g_fused_type)) < 0) return nullptr;
    return m;
}
