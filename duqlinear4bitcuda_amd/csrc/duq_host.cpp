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
#include <torch/csrc/jit/frontend/tracer.h>

#include <ATen/core/Tensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPStream.h>
#include <structmember.h>
#include <torch/version.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstdio>
#include <cstring>
#include <vector>

#include "../../include/duq_hip.h"

namespace {

using at::ScalarType;
using at::Tensor;

PyObject *g_packed = nullptr;  // class PackedQuantizedTensor
PyObject *g_check = nullptr;   // _lib.check(status, name): raises for a status other than 0
// byte offsets of PackedQuantizedTensor's __slots__ in its instances
enum Slot { kQ, kS, kZeros, kRowsum, kShadow, kSrc, kVersion, kClip, kQmax, kStaged, kSlots };
const char *const kSlotNames[kSlots] = {"_q", "_s", "zeros_x", "rowsum_x", "shadow_x", "_src", "_src_version", "_clip", "_qmax", "_staged"};
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

// The entries of the module: what throws on the way to the library (a tensor without memory of its own: a vmap or
// functional wrapper, a sparse tensor) is not the plain case, and goes to the Python code like the rest of those.
template <class F>
PyObject *plain_case(F f)
{
    try {
        return f();
    } catch (const std::exception &) {
        PyErr_Clear();
        return none();
    }
}
template <PyObject *(*F)(PyObject *, PyObject *const *, Py_ssize_t)>
PyObject *entry(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    return plain_case([&] { return F(self, a, n); });
}

// References of one's own to what was read from a module: while the interpreter lock is given up, or a finalizer runs,
// other code may put something else there, and a tensor that nobody else holds goes back to the allocator before the launch
// that was given its address is queued.
template <size_t N>
struct Held {
    PyObject *o[N];
    explicit Held(PyObject *const (&from)[N])
    {
        for (size_t i = 0; i < N; ++i) {
            o[i] = from[i];
            Py_INCREF(o[i]);
        }
    }
    ~Held()
    {
        for (PyObject *p : o) Py_DECREF(p);
    }
    Held(const Held &) = delete;
};

// A Python int, which has no largest value: what does not fit is the nearest that does.
int64_t whole(PyObject *o)
{
    int over = 0;
    const long long v = PyLong_AsLongLongAndOverflow(o, &over);
    return over > 0 ? INT64_MAX : over < 0 ? INT64_MIN : v;
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
    if (t.layout() != at::kStrided || !t.has_storage()) return nullptr;
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

// Memory that a call is faster with and does without where the device has none left.  To find that out, torch's allocator waits for the
// device and gives every cached block back, which the program around the call then has to allocate anew (asked on every call, 4096 x 4096 x
// 28672 beside four blocks of 16 MB in a process at its limit: 349 us instead of 344, and the host behind the device each time), so that
// one answer stands for a minute: until then nobody on the device asks for as much.
class Rooms {
    static constexpr int kDevices = 64;
    struct Refused {
        std::atomic<uint64_t> bytes{0};  // the least that there was no memory for (0: no answer)
        std::atomic<int64_t> until{0};
    };
    Refused refused_[kDevices];
    static int64_t seconds() { return std::chrono::duration_cast<std::chrono::seconds>(std::chrono::steady_clock::now().time_since_epoch()).count(); }

public:
    Scratch take(int dev, uint64_t bytes)
    {
        if (!bytes || dev < 0 || dev >= kDevices) return Scratch(0);
        Refused &r = refused_[dev];
        uint64_t least = r.bytes.load();
        if (least && seconds() >= r.until.load()) r.bytes.store(least = 0);
        if (least && bytes >= least) return Scratch(0);
        try {
            return Scratch(bytes);
        } catch (const c10::OutOfMemoryError &) {
            r.until.store(seconds() + 60);
            r.bytes.store(bytes);  // (less than what was refused before)
            return Scratch(0);
        }
    }
    void forget()
    {
        for (Refused &r : refused_) r.bytes.store(0);
    }
} g_rooms;

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
    std::vector<const void *> *at;    // and where these were then
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

// Whether `buffers` (the module's dict) still holds the tensors the call was made of, in the memory they had then (a tensor
// is given other memory by an assignment to its .data).
bool still_current(FusedCall *c, PyObject *buffers)
{
    const Py_ssize_t n = PyTuple_GET_SIZE(c->names);
    for (Py_ssize_t i = 0; i < n; ++i) {
        PyObject *t = PyDict_GetItemWithError(buffers, PyTuple_GET_ITEM(c->names, i));
        if ((t ? t : Py_None) != PyTuple_GET_ITEM(c->tensors, i)) return false;
        if (t && t != Py_None && THPVariable_Unpack(t).const_data_ptr() != (*c->at)[static_cast<size_t>(i)]) return false;
    }
    return true;
}

// What the first of several layers that take one deferred PackedQuantizedTensor leaves in it where it runs quantizer and GEMM as two
// launches: the codes [M, K/2] and behind them the scales [M], in memory of the stream they were written on.  The next layers on
// that stream run their GEMM alone (77 rows of 5120, two layers of 13824 columns: 29.6 -> 27.3 us, a third one 2.3 less again); on
// another stream, in another recording than the launch that writes them, or where the tensor of rows was given other memory since (an
// assignment to its .data), a layer quantizes for itself.  The rows' storage is kept, so that no other rows can come to lie at its address.
struct Staged {
    PyObject_HEAD
    c10::DataPtr data;
    c10::Storage storage;  // of the rows
    const void *at;        // the first row
    int64_t rows, cols;
    hipStream_t stream;
    unsigned long long recording;  // id of the stream's recording, 0: none
};
PyTypeObject g_staged_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

int64_t staged_codes(int64_t M, int64_t K) { return (M * (K / 2) + 255) / 256 * 256; }

// The recording that the stream is in, or false where it cannot be told.
bool recording_of(hipStream_t stream, unsigned long long *id)
{
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    *id = 0;
    if (hipStreamGetCaptureInfo(stream, &status, id) != hipSuccess) {
        (void)hipGetLastError();  // (not the launch's that follows)
        return false;
    }
    if (status == hipStreamCaptureStatusInvalidated) return false;
    if (status == hipStreamCaptureStatusNone) *id = 0;
    return true;
}

PyObject *new_staged(c10::DataPtr &&data, const Tensor &x, int64_t M, int64_t K, hipStream_t stream, unsigned long long recording)
{
    Staged *o = reinterpret_cast<Staged *>(g_staged_type.tp_alloc(&g_staged_type, 0));
    if (!o) return nullptr;
    new (&o->data) c10::DataPtr(std::move(data));
    new (&o->storage) c10::Storage(x.storage());
    o->at = x.const_data_ptr();
    o->rows = M;
    o->cols = K;
    o->stream = stream;
    o->recording = recording;
    return reinterpret_cast<PyObject *>(o);
}

// Whether the codes are those of x as [M, K] rows, on this stream and in this recording of it.
bool staged_for(const Staged *s, const Tensor &x, int64_t M, int64_t K, hipStream_t stream, unsigned long long recording)
{
    return s->stream == stream && s->recording == recording && s->rows == M && s->cols == K &&
           s->storage.unsafeGetStorageImpl() == x.storage().unsafeGetStorageImpl() && s->at == x.const_data_ptr();
}

void staged_dealloc(PyObject *self)
{
    Staged *s = reinterpret_cast<Staged *>(self);
    s->data.~DataPtr();
    s->storage.~Storage();
    Py_TYPE(self)->tp_free(self);
}

// A copy or a saved file of the packed tensor goes without it.
PyObject *staged_reduce(PyObject *, PyObject *) { return Py_BuildValue("(O())", reinterpret_cast<PyObject *>(Py_TYPE(Py_None))); }

PyMethodDef g_staged_methods[] = {{"__reduce__", staged_reduce, METH_NOARGS, nullptr}, {nullptr, nullptr, 0, nullptr}};

constexpr int64_t kFp6MinTiles = 32;  // _FP6_MIN_TILES of nn/linear.py: smaller settings are taken as they are (_fp6_pays)

// min_tiles: the module's fp6_min_tiles, negative where the caller does not know it.  packed: the deferred tensor that x is the rows
// of, or null
PyObject *run_rows(FusedCall *c, PyObject *buffers, const Tensor &x, float clip, int qmax, int64_t min_tiles = -1, PyObject *packed = nullptr)
{
    duq_fused_layer l = c->layer;
    if (x.dim() == 0 || x.size(-1) != static_cast<int64_t>(l.K) || x.get_device() != c->dev || l.K % 64) return none();
    const int64_t M = x.numel() / l.K;
    if (M < 1 || M > c->max_rows || current_device() != c->dev) return none();
    // more than 64 rows of a layer with a 6-bit float shadow: those of the 6-bit float path are not run here (the rule
    // of the layer's _fp6_pays)
    static PyObject *const shadow_name = PyUnicode_InternFromString("weight_shadow");
    if (M > 64) {
        PyObject *s = PyDict_GetItemWithError(buffers, shadow_name);
        const int64_t tiles = (M + 63) / 64 * ((l.N + 255) / 256);
        const int64_t per = l.K >= 8192 ? 8 : l.K >= 2048 ? 10 : 20;
        if (s && s != Py_None &&
            (min_tiles < 0 || ((M > 1024 || l.K < 1024 || min_tiles < kFp6MinTiles || tiles / per >= min_tiles) &&
                               (tiles >= min_tiles || (M > 256 && 8 * tiles >= 5 * min_tiles)))))
            return none();
    }
    const int64_t bytes = staging_of(c, M);
    l.clip = clip;
    l.qmax = qmax;
    const hipStream_t stream = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(c->dev)).stream();
    const bool shares = packed && bytes > 0 && (l.mode == DUQ_EPI_SYM || l.mode == DUQ_EPI_SYM_DUAL);
    unsigned long long recording = 0;
    if (shares && recording_of(stream, &recording)) {
        const int64_t at = staged_codes(M, l.K);
        PyObject *s = slot(packed, kStaged);
        if (s && Py_TYPE(s) == &g_staged_type) {
            Staged *staged = reinterpret_cast<Staged *>(s);
            if (staged_for(staged, x, M, l.K, stream, recording)) {
                const Held<1> h({s});  // (another thread may put something else there)
                Tensor y = output(x, l.N, ScalarType::Half);
                const uint8_t *q = static_cast<const uint8_t *>(staged->data.get());
                int st;
                {
                    Unlocked u;
                    st = duq_linear4bit_forward(l.mode, q, half(q + at), nullptr, l.w, l.w_scale_1, nullptr, l.w_scale_2, nullptr, l.bias,
                                                static_cast<uint32_t>(M), l.N, l.K, out<duq_half>(y), stream);
                }
                if (st) return finish(st, "linear4bit_forward", nullptr);
                return wrap(std::move(y));
            }
        }
        Tensor y = output(x, l.N, ScalarType::Half);
        Scratch ws(static_cast<uint64_t>(at + 2 * M));
        uint8_t *q = static_cast<uint8_t *>(ws.get());
        int st;
        {
            Unlocked u;
            st = duq_quantize_linear4bit_forward(l.mode, half(x.const_data_ptr()), clip, qmax, l.w, l.w_scale_1, l.w_scale_2, l.bias,
                                                 static_cast<uint32_t>(M), l.N, l.K, out<duq_half>(y), q, reinterpret_cast<duq_half *>(q + at),
                                                 nullptr, 0, stream);
        }
        if (st) return finish(st, "quantize_linear4bit_forward", nullptr);
        PyObject *left = new_staged(std::move(ws.data), x, M, l.K, stream, recording);
        if (!left) return nullptr;
        PyObject *before = slot(packed, kStaged);
        slot(packed, kStaged) = left;
        Py_XDECREF(before);
        return wrap(std::move(y));
    }
    Tensor y = output(x, l.N, ScalarType::Half);
    Scratch ws(static_cast<uint64_t>(bytes));
    int st;
    {
        Unlocked u;
        st = duq_quantize_linear4bit_forward_layer(&l, half(x.const_data_ptr()), static_cast<uint32_t>(M), out<duq_half>(y),
                                                   ws.get(), static_cast<uint64_t>(bytes), stream);
    }
    if (st) return finish(st, "quantize_linear4bit_forward", nullptr);
    return wrap(std::move(y));
}

int64_t tiles_argument(PyObject *const *a, Py_ssize_t n)
{
    return n == 3 && PyLong_Check(a[2]) ? whole(a[2]) : -1;
}

// take(buffers, packed[, the module's fp6_min_tiles]): the layer's result for a PackedQuantizedTensor that was handed on unquantized
PyObject *fused_take(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    FusedCall *c = reinterpret_cast<FusedCall *>(self);
    if (n < 2 || n > 3 || !PyDict_Check(a[0]) || reinterpret_cast<PyObject *>(Py_TYPE(a[1])) != g_packed) return none();
    PyObject *src = slot(a[1], kSrc), *version = slot(a[1], kVersion), *clip = slot(a[1], kClip), *qmax = slot(a[1], kQmax);
    if (!src || !version || !clip || !qmax || !PyFloat_Check(clip) || !PyLong_Check(qmax)) return none();
    const Tensor *x = plain(src, ScalarType::Half, c->dev);
    if (!x || x->is_inference() || x->_version() != whole(version) || !still_current(c, a[0])) return none();
    const Tensor held = *x;  // (another thread may quantize the packed tensor, which drops its rows)
    return guarded([&] { return run_rows(c, a[0], held, static_cast<float>(PyFloat_AS_DOUBLE(clip)), static_cast<int>(whole(qmax)),
                                         tiles_argument(a, n), a[1]); });
}

// take_rows(buffers, x[, fp6_min_tiles]): the same for a layer with its own quantizer
PyObject *fused_take_rows(PyObject *self, PyObject *const *a, Py_ssize_t n)
{
    FusedCall *c = reinterpret_cast<FusedCall *>(self);
    if (n < 2 || n > 3 || !PyDict_Check(a[0])) return none();
    const Tensor *x = plain(a[1], ScalarType::Half, c->dev);
    if (!x || reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16 || !still_current(c, a[0])) return none();
    return guarded([&] { return run_rows(c, a[0], *x, 1.0f, 6, tiles_argument(a, n)); });
}

// FusedCall(mode, N, K, device index, max_rows, addresses of (w, s1, z1, s2, z2, adj1, adj2, bias), names, tensors[, the
// address of each tensor, else where they are now])
PyObject *fused_new(PyTypeObject *type, PyObject *args, PyObject *)
{
    int mode, dev;
    unsigned N, K;
    long long max_rows;
    PyObject *addr, *names, *tensors, *at = nullptr;
    if (!PyArg_ParseTuple(args, "iIIiLO!O!O!|O!", &mode, &N, &K, &dev, &max_rows, &PyTuple_Type, &addr, &PyTuple_Type, &names,
                          &PyTuple_Type, &tensors, &PyTuple_Type, &at))
        return nullptr;
    const Py_ssize_t n = PyTuple_GET_SIZE(names);
    bool fits = PyTuple_GET_SIZE(addr) == 8 && n >= 1 && PyTuple_GET_SIZE(tensors) == n && (!at || PyTuple_GET_SIZE(at) == n) &&
                max_rows >= 1 && max_rows <= 65536;
    for (Py_ssize_t i = 0; fits && i < n; ++i)
        fits = THPVariable_Check(PyTuple_GET_ITEM(tensors, i)) || (i > 0 && PyTuple_GET_ITEM(tensors, i) == Py_None);
    if (!fits) {
        PyErr_SetString(PyExc_ValueError, "FusedCall: eight addresses, and a tensor (the weight first) for every name");
        return nullptr;
    }
    void *p[8];
    std::vector<const void *> where(static_cast<size_t>(n));
    auto address = [](PyObject *o) { return o == Py_None ? nullptr : PyLong_AsVoidPtr(o); };
    for (Py_ssize_t i = 0; i < 8 && !PyErr_Occurred(); ++i) p[i] = address(PyTuple_GET_ITEM(addr, i));
    for (Py_ssize_t i = 0; i < n && !PyErr_Occurred(); ++i) {
        PyObject *t = PyTuple_GET_ITEM(tensors, i);
        where[static_cast<size_t>(i)] = at             ? address(PyTuple_GET_ITEM(at, i))
                                        : t == Py_None ? nullptr
                                                       : THPVariable_Unpack(t).const_data_ptr();
    }
    if (PyErr_Occurred()) return nullptr;
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
    c->at = new std::vector<const void *>(std::move(where));
    c->staging = new std::vector<int64_t>();
    return reinterpret_cast<PyObject *>(c);
}

void fused_dealloc(PyObject *self)
{
    FusedCall *c = reinterpret_cast<FusedCall *>(self);
    Py_XDECREF(c->names);
    Py_XDECREF(c->tensors);
    delete c->staging;
    delete c->at;
    Py_TYPE(self)->tp_free(self);
}

PyMethodDef g_fused_methods[] = {
    {"take", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<fused_take>)), METH_FASTCALL, nullptr},
    {"take_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<fused_take_rows>)), METH_FASTCALL, nullptr},
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
    if (cols % 64 || numel <= 0 || numel / cols > whole(a[1]) || reinterpret_cast<uintptr_t>(x->const_data_ptr()) % 16) return none();
    if (a[2] != Py_False && cols % 128 == 0 && (!PyLong_Check(a[3]) || numel / cols >= whole(a[3]))) return none();
    PyTypeObject *type = reinterpret_cast<PyTypeObject *>(g_packed);
    const Held<3> h({a[0], a[4], a[5]});   // (the allocation may run the garbage collector)
    PyObject *p = type->tp_alloc(type, 0);
    if (!p) return nullptr;
    for (Slot s : {kQ, kS, kZeros, kRowsum, kShadow, kStaged}) slot(p, s) = none();
    auto put = [&](Slot s, PyObject *v) {
        Py_INCREF(v);
        slot(p, s) = v;
    };
    put(kSrc, h.o[0]);
    slot(p, kVersion) = PyLong_FromLong(static_cast<long>(x->_version()));
    put(kClip, h.o[1]);
    put(kQmax, h.o[2]);
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
    const int qmax = static_cast<int>(whole(a[5]));
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
//         shadows[, room_bytes], stream): modes 0 - 4 on packed codes, with at most so many bytes of room for shadows made in the call, or with
// `shadows` on the 6-bit float shadows of both operands
PyObject *m_linear4(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if ((n != 14 && n != 15) || !PyLong_Check(a[0]) || (n == 15 && !PyLong_Check(a[13]))) return none();
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
    const int64_t most = n == 15 ? whole(a[13]) : INT64_MAX;
    const duq_stream_t st = stream_of(a[n - 1]);
    return guarded([&]() -> PyObject * {
        Tensor y = output(*x, N, ScalarType::Half);
        const uint8_t *px = static_cast<const uint8_t *>(x->const_data_ptr()), *pw = static_cast<const uint8_t *>(w->const_data_ptr());
        const uint32_t m = static_cast<uint32_t>(M), nn = static_cast<uint32_t>(N), k = static_cast<uint32_t>(K);
        const uint64_t bytes = !shadows && duq_linear4bit_room_pays(mode, m, nn, k) ? duq_linear4bit_room_bytes(mode, m, nn, k) : 0;
        const Scratch room = g_rooms.take(dev, static_cast<int64_t>(bytes) <= most ? bytes : 0);
        int e;
        {
            Unlocked u;
            if (room.get())
                e = duq_linear4bit_forward_room(mode, px, half(p[2]), half(p[3]), i32(p[10]), pw, half(p[5]), half(p[6]), half(p[7]),
                                                half(p[8]), i32(p[11]), half(p[9]), m, nn, k, out<duq_half>(y), room.get(), bytes, st);
            else if (shadows)
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

// forget_refused_rooms(): calls ask for memory again, whatever the answer was
PyObject *m_forget_refused_rooms(PyObject *, PyObject *)
{
    g_rooms.forget();
    return none();
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

// int8 codes with their scales and zeros (w_tiled not None: the GEMM reads that copy and w is not looked at), or float32
// rows (scale_x and zeros_x None) that the call quantizes first.  null stream: the current one.
PyObject *linear8(PyObject *const *a, int64_t N, const duq_stream_t *stream)
{
    const bool quantize = a[1] == Py_None;
    const Tensor *x = plain(a[0], quantize ? ScalarType::Float : ScalarType::Char, -1);
    if (!x || x->dim() == 0 || x->numel() == 0) return none();
    const int dev = static_cast<int>(x->get_device());
    const int64_t K = x->size(-1), M = x->numel() / K;
    if (N <= 0 || M > UINT32_MAX || N > UINT32_MAX || K > UINT32_MAX) return none();
    const void *p[8] = {};
    if (!operand(a[1], ScalarType::Float, dev, M, quantize, &p[1]) || !operand(a[2], ScalarType::Float, dev, M, quantize, &p[2]) ||
        !operand(a[3], ScalarType::Char, dev, N * K, !quantize, &p[3]) ||
        !operand(a[4], ScalarType::Char, dev, (N + 31) / 32 * 32 * K, true, &p[4]) || (!p[3] && !p[4]) ||
        !operand(a[5], ScalarType::Float, dev, N, false, &p[5]) || !operand(a[6], ScalarType::Float, dev, N, false, &p[6]) ||
        !operand(a[7], ScalarType::Float, dev, N, true, &p[7]))
        return none();
    if (p[3] && THPVariable_Unpack(a[3]).dim() != 2) return none();
    return guarded([&]() -> PyObject * {
        const duq_stream_t st = stream ? *stream : c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream();
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

// linear8(x, scale_x, zeros_x, w, w_tiled, w_scale, w_zeros, bias, N, stream)
PyObject *m_linear8(PyObject *, PyObject *const *a, Py_ssize_t n)
{
    if (n != 10 || !PyLong_Check(a[8])) return none();
    const duq_stream_t st = stream_of(a[9]);
    return linear8(a, PyLong_AsLongLong(a[8]), &st);
}

// ---- calls of modules ----------------------------------------------------------------------------------------
// `__call__` of the framework's module classes: what torch.nn.Module.__call__ and the class's forward do in the plain
// case (no hooks, no compiled or replaced forward, no other __call__ or _call_impl on the way, plain tensors, buffers as
// they were when the layer's call was prepared), in one piece of native code: 0.2 us where the two Python frames cost 1
// (quantizer and layer of a decode step 6.6 -> 5.5 us).  Anything else goes to the __call__ that comes next in the method
// order of the object's class, as super().__call__ would: mostly torch.nn.Module's.

enum Kind { kSymQuant, kSymLayer, kOwnLayer, kEightBit, kSymProduct, kAsymProduct };
struct Entry {
    PyTypeObject *type;
    PyObject *forward;
    Kind kind;
    PyObject *call = nullptr;          // the __call__ that its instances have: a ModuleCall, or torch's for kind -1
    PyObject *mro = nullptr;           // the method order at the time,
    std::vector<PyTypeObject *> bases; // and what stands between the class and torch.nn.Module there
};
std::vector<Entry> *g_entries = nullptr;
PyTypeObject *g_module_type = nullptr;           // torch.nn.Module
PyObject *g_module_call = nullptr, *g_call_impl = nullptr;  // its __call__, and the _call_impl that this one calls
std::vector<PyObject *> *g_global_hooks = nullptr;    // torch's dicts of hooks for every module
PyObject *g_ops_dict = nullptr, *g_launch = nullptr;  // _HIP's namespace and the _launch function defined there
PyObject *g_lib_dict = nullptr;                  // attributes of the ctypes library object
PyTypeObject *g_funcptr = nullptr;               // ... and the type of its functions
PyTypeObject *g_quant8_type = nullptr, *g_asym_type = nullptr, *g_sym_type = nullptr;

struct Names {
#define NAME(n) PyObject *n = PyUnicode_InternFromString(#n)
    NAME(_forward_hooks);
    NAME(_forward_pre_hooks);
    NAME(_backward_hooks);
    NAME(_backward_pre_hooks);
    NAME(_compiled_call_impl);
    NAME(_call_impl);
    NAME(forward);
    NAME(_buffers);
    NAME(_modules);
    NAME(_decode);
    NAME(native);
    NAME(fused);
    NAME(input_clip_ratio);
    NAME(qmax);
    NAME(shadow);
    NAME(shadow_min_rows);
    NAME(shifted);
    NAME(defer_rows);
    NAME(require_quantizer);
    NAME(quantizer);
    NAME(quantizer_A);
    NAME(quantizer_B);
    NAME(tiled);
    NAME(one_call_rows);
    NAME(fp6_min_tiles);
    NAME(transpose_B);
    NAME(weight);
    NAME(weight_tiled);
    NAME(weight_shadow);
    NAME(weight_scales);
    NAME(weight_scales_1);
    NAME(weight_scales_2);
    NAME(weight_zeros);
    NAME(bias);
    NAME(_tiled_key);
    NAME(_shadow_key);
    NAME(only);
    NAME(_launch);
    NAME(duq_quantize_linear8bit_forward);
    NAME(duq_quantize_product);
    NAME(duq_quantize_rows_sym_bf6);
    NAME(duq_linear4bit_forward_bf6);
    NAME(__call__);
#undef NAME
};
const Names *g_names = nullptr;

PyObject *get(PyObject *dict, PyObject *name) { return dict ? PyDict_GetItemWithError(dict, name) : nullptr; }

// attribute of an instance: its own dict, then its class (plain values only; borrowed)
PyObject *attr(PyObject *self, PyObject *dict, PyObject *name)
{
    PyObject *v = get(dict, name);
    return v ? v : _PyType_Lookup(Py_TYPE(self), name);
}

PyObject *dict_of(PyObject *o)
{
    PyObject **d = _PyObject_GetDictPtr(o);
    return d ? *d : nullptr;
}

bool empty_dict(PyObject *d) { return d && PyDict_Check(d) && PyDict_GET_SIZE(d) == 0; }

// The entry of a module for which torch's __call__ would run its class's forward and nothing else, or null.
const Entry *plain_module(PyObject *self, PyObject *dict)
{
    const Entry *e = nullptr;
    for (const Entry &k : *g_entries)
        if (k.type == Py_TYPE(self)) e = &k;
    const Names &n = *g_names;
    if (!e || !dict || e->type->tp_mro != e->mro) return nullptr;
    if (_PyType_Lookup(e->type, n.forward) != e->forward || get(dict, n.forward)) return nullptr;
    if (_PyType_Lookup(e->type, n._call_impl) != g_call_impl || get(dict, n._call_impl)) return nullptr;
    if (attr(self, dict, n._compiled_call_impl) != Py_None) return nullptr;
    for (PyTypeObject *base : e->bases)
        if (get(base->tp_dict, n.__call__)) return nullptr;
    for (PyObject *h : {n._forward_hooks, n._forward_pre_hooks, n._backward_hooks, n._backward_pre_hooks})
        if (!empty_dict(get(dict, h))) return nullptr;
    return e;
}

// The same for a module that is not being called already: its class's __call__ has to be the one known too.
const Entry *plain_call(PyObject *self, PyObject *dict)
{
    const Entry *e = plain_module(self, dict);
    return e && _PyType_Lookup(e->type, g_names->__call__) == e->call ? e : nullptr;
}

bool plain_torch()
{
    if (get(g_module_type->tp_dict, g_names->__call__) != g_module_call) return false;
    for (PyObject *d : *g_global_hooks)
        if (PyDict_GET_SIZE(d)) return false;
    return !torch::jit::tracer::isTracing();   // (torch then calls _slow_forward)
}

// the library's own function under that name (a tracer may have put a Python one there)
bool library_function(PyObject *name)
{
    PyObject *f = get(g_lib_dict, name);
    return f && Py_TYPE(f) == g_funcptr;
}

PyObject *call_sym_quantizer(PyObject *self, PyObject *dict, PyObject *x)
{
    const Names &n = *g_names;
    PyObject *a[6] = {x,
                      attr(self, dict, n.defer_rows),
                      get(dict, n.shadow),
                      get(dict, n.shadow_min_rows),
                      get(dict, n.input_clip_ratio),
                      get(dict, n.qmax)};
    for (PyObject *v : a)
        if (!v) return none();
    PyObject *p = m_defer(nullptr, a, 6);
    if (p != Py_None || a[2] == Py_False) return p;
    // a quantizer set to write the 6-bit float shadow (True: beside the codes, "only": alone), rows enough for it
    const bool codes = a[2] == Py_True;
    const Tensor *t = plain(x, ScalarType::Half, -1);
    if (!t || t->dim() == 0 || !(codes || (PyUnicode_CheckExact(a[2]) && PyUnicode_Compare(a[2], n.only) == 0)) || !PyLong_Check(a[3]) ||
        !PyFloat_Check(a[4]) || !PyLong_Check(a[5]) || get(g_ops_dict, n._launch) != g_launch || !library_function(n.duq_quantize_rows_sym_bf6))
        return p;
    const int64_t K = t->size(-1), numel = t->numel();
    if (K % 128 || numel <= 0 || numel / K < whole(a[3]) || numel / K > UINT32_MAX || K > UINT32_MAX ||
        reinterpret_cast<uintptr_t>(t->const_data_ptr()) % 16 || t->get_device() != current_device())
        return p;
    Py_DECREF(p);
    return guarded([&]() -> PyObject * {
        const Held<1> h({x});
        const float clip = static_cast<float>(PyFloat_AS_DOUBLE(a[4]));
        const int qmax = static_cast<int>(whole(a[5]));
        Tensor q, b = output(*t, K * 3 / 4, ScalarType::Byte), s = output(*t, 1, ScalarType::Half);
        if (codes) q = output(*t, K / 2, ScalarType::Byte);
        const hipStream_t st = c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(t->get_device())).stream();
        int e;
        {
            Unlocked u;
            e = duq_quantize_rows_sym_bf6(half(t->const_data_ptr()), static_cast<uint32_t>(numel / K), static_cast<uint32_t>(K), clip, qmax,
                                          out<uint8_t>(q), out<uint8_t>(b), out<duq_half>(s), st);
        }
        if (e) return finish(e, "quantize_rows_sym_bf6", nullptr);
        PyTypeObject *type = reinterpret_cast<PyTypeObject *>(g_packed);
        PyObject *packed = type->tp_alloc(type, 0);
        if (!packed) return nullptr;
        for (Slot i : {kZeros, kRowsum, kSrc, kStaged}) slot(packed, i) = none();
        slot(packed, kQ) = codes ? wrap(std::move(q)) : none();
        slot(packed, kS) = wrap(std::move(s));
        slot(packed, kShadow) = wrap(std::move(b));
        return packed;
    });
}

// A symmetric layer whose input is a 6-bit float shadow alone (the rule for one that comes with codes: the layer's _use_shadow).
PyObject *call_layer_on_shadow(PyObject *self, PyObject *dict, PyObject *packed)
{
    const Names &n = *g_names;
    PyObject *q = slot(packed, kQ), *src = slot(packed, kSrc), *shadow = slot(packed, kShadow), *scales = slot(packed, kS);
    PyObject *buffers = get(dict, n._buffers), *key = get(dict, n._shadow_key);
    if (q != Py_None || src != Py_None || !shadow || !scales || !buffers || !key || !PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 3 ||
        attr(self, dict, n.fused) != Py_True || get(g_ops_dict, n._launch) != g_launch || !library_function(n.duq_linear4bit_forward_bf6))
        return none();
    PyObject *w = get(buffers, n.weight), *ws = get(buffers, n.weight_shadow), *s1 = get(buffers, n.weight_scales), *s2 = Py_None;
    const bool dual = !s1;
    if (dual) s1 = get(buffers, n.weight_scales_1), s2 = get(buffers, n.weight_scales_2);
    PyObject *bias = get(buffers, n.bias);
    if (!bias) bias = get(dict, n.bias) == Py_None ? Py_None : nullptr;
    if (!w || !ws || !s1 || !s2 || !bias) return none();
    const Tensor *pw = plain(w, ScalarType::Byte, -1), *px = plain(shadow, ScalarType::Byte, -1);
    // the shadow is the weight's as it is now: version, address, device (the layer's _fp6_ready)
    if (!pw || !px || pw->is_inference() || !THPVariable_CheckExact(ws) || THPVariable_Unpack(ws).get_device() != pw->get_device() ||
        whole(PyTuple_GET_ITEM(key, 0)) != pw->_version() || PyLong_AsVoidPtr(PyTuple_GET_ITEM(key, 1)) != pw->const_data_ptr() ||
        px->get_device() != current_device()) {
        PyErr_Clear();
        return none();
    }
    static PyObject *const modes[2] = {PyLong_FromLong(DUQ_EPI_SYM), PyLong_FromLong(DUQ_EPI_SYM_DUAL)};
    PyObject *st = PyLong_FromVoidPtr(c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(px->get_device())).stream());
    if (!st) return nullptr;
    const Held<14> a({modes[dual], shadow, scales, Py_None, ws, s1, Py_None, s2, Py_None, bias, Py_None, Py_None, Py_True, st});
    Py_DECREF(st);
    return m_linear4(nullptr, a.o, 14);
}

PyObject *call_layer(PyObject *self, PyObject *dict, PyObject *x, bool own_quantizer)
{
    const Names &n = *g_names;
    if (!own_quantizer && reinterpret_cast<PyObject *>(Py_TYPE(x)) == g_packed && slot(x, kQ) == Py_None && slot(x, kSrc) == Py_None)
        return call_layer_on_shadow(self, dict, x);
    PyObject *decode = get(dict, n._decode), *buffers = get(dict, n._buffers);
    if (!decode || decode == Py_None || !buffers || attr(self, dict, n.fused) != Py_True) return none();
    if (own_quantizer && get(dict, n.require_quantizer) != Py_True) return none();
    PyObject *native = PyObject_GetAttr(decode, n.native);
    if (!native) return nullptr;
    PyObject *r = none();
    if (Py_TYPE(native) == &g_fused_type) {
        Py_DECREF(r);
        PyObject *tiles = attr(self, dict, n.fp6_min_tiles), *a[3] = {buffers, x, tiles ? tiles : Py_None};
        r = own_quantizer ? fused_take_rows(native, a, 3) : fused_take(native, a, 3);
    }
    Py_DECREF(native);
    return r;
}

PyObject *call_eight_bit(PyObject *self, PyObject *dict, PyObject *x)
{
    const Names &n = *g_names;
    PyObject *buffers = get(dict, n._buffers), *modules = get(dict, n._modules), *rows = attr(self, dict, n.one_call_rows);
    if (!buffers || !modules || !rows || !PyLong_Check(rows) || get(dict, n.require_quantizer) != Py_True ||
        attr(self, dict, n.fused) != Py_True || !library_function(n.duq_quantize_linear8bit_forward))
        return none();
    PyObject *q = get(modules, n.quantizer), *qd = q ? dict_of(q) : nullptr;
    if (!q || Py_TYPE(q) != g_quant8_type || !qd || get(qd, n.fused) != Py_True) return none();
    PyObject *tiled = attr(self, dict, n.tiled), *w = get(buffers, n.weight), *wt = Py_None;
    if (!w || (tiled != Py_True && tiled != Py_False)) return none();
    const Tensor *px = plain(x, ScalarType::Float, -1), *pw = plain(w, ScalarType::Char, -1);
    if (!px || !pw || pw->dim() != 2 || px->dim() == 0 || px->size(-1) != pw->size(1) || pw->size(1) % 32 || px->numel() == 0 ||
        reinterpret_cast<uintptr_t>(px->const_data_ptr()) % 16 || px->numel() / pw->size(1) > whole(rows) ||
        px->get_device() != current_device())
        return none();
    if (tiled == Py_True) {  // the copy is the weight's as it is now: version, address, device (the layer's _tiled_weight)
        PyObject *key = get(dict, n._tiled_key);
        wt = get(buffers, n.weight_tiled);
        if (!wt || wt == Py_None || !key || !PyTuple_Check(key) || PyTuple_GET_SIZE(key) != 3 || pw->is_inference() ||
            whole(PyTuple_GET_ITEM(key, 0)) != pw->_version() ||
            PyLong_AsVoidPtr(PyTuple_GET_ITEM(key, 1)) != pw->const_data_ptr() || !THPVariable_CheckExact(wt) ||
            THPVariable_Unpack(wt).get_device() != pw->get_device()) {
            PyErr_Clear();
            return none();
        }
    }
    PyObject *s = get(buffers, n.weight_scales), *z = get(buffers, n.weight_zeros), *bias = get(buffers, n.bias);
    if (!s || !z) return none();
    const int64_t N = pw->size(0);
    const Held<8> a({x, Py_None, Py_None, w, wt, s, z, bias ? bias : Py_None});
    return linear8(a.o, N, nullptr);
}

// A product of activations: both quantizers of the module in their plain form, operands of one batch.
PyObject *call_product(PyObject *self, PyObject *dict, PyObject *pa, PyObject *pb, bool asym)
{
    const Names &n = *g_names;
    PyObject *modules = get(dict, n._modules);
    if (!modules || attr(self, dict, n.fused) != Py_True || get(g_ops_dict, n._launch) != g_launch ||
        !library_function(n.duq_quantize_product) || (asym && get(dict, n.transpose_B) != Py_False))
        return none();
    float clip[2] = {1.0f, 1.0f};
    int64_t qmax[2] = {6, 6};
    PyObject *const names[2] = {n.quantizer_A, n.quantizer_B};
    for (int i = 0; i < 2; ++i) {
        PyObject *q = get(modules, names[i]), *qd = q ? dict_of(q) : nullptr;
        if (!q || Py_TYPE(q) != (asym ? g_asym_type : g_sym_type) || !plain_call(q, qd) || get(qd, n.shadow) != Py_False) return none();
        if (asym) {
            if (get(qd, n.shifted) != Py_False) return none();
        } else {
            PyObject *c = get(qd, n.input_clip_ratio), *m = get(qd, n.qmax);
            if (!c || !m || !PyFloat_Check(c) || !PyLong_Check(m)) return none();
            clip[i] = static_cast<float>(PyFloat_AS_DOUBLE(c));
            qmax[i] = whole(m);
            if (qmax[i] < 0 || qmax[i] > 7) return none();
        }
    }
    const Tensor *a = plain(pa, ScalarType::Half, -1);
    if (!a || a->dim() < 2) return none();
    const int dev = static_cast<int>(a->get_device());
    const Tensor *b = plain(pb, ScalarType::Half, dev);
    if (!b || b->dim() < 2 || dev != current_device() || a->numel() == 0 || b->numel() == 0) return none();
    const int64_t K = a->size(-1), N = b->size(-2);
    int64_t batch = 1, M = a->size(-2);
    if (b->size(-1) != K || K % 64 || K > 131008 || reinterpret_cast<uintptr_t>(a->const_data_ptr()) % 16 ||
        reinterpret_cast<uintptr_t>(b->const_data_ptr()) % 16)
        return none();
    if (b->dim() > 2 || asym) {  // one product per entry of the same leading dimensions
        if (a->dim() != b->dim()) return none();
        for (int64_t d = 0; d < a->dim() - 2; ++d) {
            if (a->size(d) != b->size(d)) return none();
            batch *= a->size(d);
        }
    } else {
        M = a->numel() / K;  // every row of A against one B
    }
    if (M > (1 << 24) || N > (1 << 22) || batch > INT32_MAX || batch * (M + N) > INT32_MAX) return none();
    return guarded([&]() -> PyObject * {
        const int mode = asym ? DUQ_EPI_ASYM : DUQ_EPI_SYM;
        const uint32_t nb = static_cast<uint32_t>(batch), m = static_cast<uint32_t>(M), nn = static_cast<uint32_t>(N),
                       k = static_cast<uint32_t>(K);
        Tensor y = output(*a, N, ScalarType::Half);
        const uint64_t bytes = duq_quantize_product_workspace_bytes(mode, nb, m, nn, k);
        Scratch ws(bytes);
        int e;
        {
            Unlocked u;
            e = duq_quantize_product(mode, half(a->const_data_ptr()), half(b->const_data_ptr()), nb, m, nn, k, clip[0],
                                     static_cast<int>(qmax[0]), clip[1], static_cast<int>(qmax[1]), out<duq_half>(y), ws.get(), bytes,
                                     c10::hip::getCurrentHIPStream(static_cast<c10::DeviceIndex>(dev)).stream());
        }
        if (e) return finish(e, "quantize_product", nullptr);
        return wrap(std::move(y));
    });
}

struct ModuleCall {
    PyObject_HEAD
    vectorcallfunc call;
    PyTypeObject *owner;   // the class whose __call__ it is
    PyObject *dict;        // __name__, __doc__, __signature__: those of torch.nn.Module's
};

// super(owner, self).__call__(...)
PyObject *next_call(PyTypeObject *owner, PyObject *const *a, Py_ssize_t n, PyObject *kwnames)
{
    PyTypeObject *type = n && PyType_IsSubtype(Py_TYPE(a[0]), owner) ? Py_TYPE(a[0]) : owner;
    PyObject *mro = type->tp_mro, *f = nullptr;
    bool behind = false;
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(mro) && !f; ++i) {
        PyTypeObject *t = reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(mro, i));
        if (behind) f = get(t->tp_dict, g_names->__call__);
        behind |= t == owner;
    }
    if (!f) {
        PyErr_Format(PyExc_TypeError, "'%.200s' object is not callable", type->tp_name);
        return nullptr;
    }
    Py_INCREF(f);
    PyObject *r = nullptr;
    if (!n || Py_TYPE(f)->tp_flags & Py_TPFLAGS_METHOD_DESCRIPTOR) {   // (a function: takes the object as its first argument)
        r = PyObject_Vectorcall(f, a, static_cast<size_t>(n), kwnames);
    } else if (descrgetfunc bind = Py_TYPE(f)->tp_descr_get) {
        if (PyObject *bound = bind(f, a[0], reinterpret_cast<PyObject *>(Py_TYPE(a[0])))) {
            r = PyObject_Vectorcall(bound, a + 1, static_cast<size_t>(n - 1), kwnames);
            Py_DECREF(bound);
        }
    } else {
        r = PyObject_Vectorcall(f, a + 1, static_cast<size_t>(n - 1), kwnames);
    }
    Py_DECREF(f);
    return r;
}

PyObject *module_call(PyObject *self, PyObject *const *a, size_t nargsf, PyObject *kwnames)
{
    PyTypeObject *owner = reinterpret_cast<ModuleCall *>(self)->owner;
    const Py_ssize_t n = PyVectorcall_NARGS(nargsf);
    if (!kwnames && n >= 2 && n <= 3 && Py_TYPE(a[0]) == owner && plain_torch()) {
        PyObject *dict = dict_of(a[0]);
        const Entry *e = plain_module(a[0], dict);
        const bool product = e && (e->kind == kSymProduct || e->kind == kAsymProduct);
        if (e && n == (product ? 3 : 2)) {
            PyObject *r = plain_case([&] {
                return e->kind == kSymQuant   ? call_sym_quantizer(a[0], dict, a[1])
                       : e->kind == kSymLayer ? call_layer(a[0], dict, a[1], false)
                       : e->kind == kOwnLayer ? call_layer(a[0], dict, a[1], true)
                       : e->kind == kEightBit ? call_eight_bit(a[0], dict, a[1])
                                              : call_product(a[0], dict, a[1], a[2], e->kind == kAsymProduct);
            });
            if (r != Py_None) return r;
            Py_DECREF(r);
        }
    }
    return next_call(owner, a, n, kwnames);
}

PyObject *module_call_get(PyObject *self, PyObject *obj, PyObject *)
{
    if (!obj || obj == Py_None) {
        Py_INCREF(self);
        return self;
    }
    return PyMethod_New(self, obj);
}

PyTypeObject g_module_call_type = {PyVarObject_HEAD_INIT(nullptr, 0)};

// install(classes, torch's hook dicts, (torch.nn.Module, its own __call__ and _call_impl, None for one that is not torch's: no
// call is then run natively), (_HIP module, its _launch), (ctypes library, type of its functions), (SymQuantizer, AsymQuantizer,
// AsymQuantizer8bit)): `classes` is a tuple of (class, kind as in Kind, or -1 for a class that only a product looks at, the
// forward it was defined with); gives every one of them the native __call__ that has no __call__ of its own
PyObject *m_install(PyObject *, PyObject *args)
{
    PyObject *classes, *hooks, *module, *call[2], *ops, *lib, *launch, *funcptr, *sym, *asym, *quant8;
    if (!PyArg_ParseTuple(args, "O!O!(O!OO)(OO)(OO!)(O!O!O!)", &PyTuple_Type, &classes, &PyTuple_Type, &hooks, &PyType_Type, &module,
                          &call[0], &call[1], &ops, &launch, &lib, &PyType_Type, &funcptr, &PyType_Type, &sym, &PyType_Type, &asym,
                          &PyType_Type, &quant8))
        return nullptr;
    PyObject *lib_dict = dict_of(lib), *ops_dict = dict_of(ops);
    PyTypeObject *module_type = reinterpret_cast<PyTypeObject *>(module);
    if (g_names || !lib_dict || !ops_dict) {
        PyErr_SetString(PyExc_RuntimeError, "install: once, with a module and a library object");
        return nullptr;
    }
    const Names *names = new Names();
    bool found = true;
    auto *global_hooks = new std::vector<PyObject *>();
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(hooks); ++i) {
        PyObject *d = PyTuple_GET_ITEM(hooks, i);
        if (!PyDict_Check(d)) found = false;
        Py_INCREF(d);
        global_hooks->push_back(d);
    }
    auto *entries = new std::vector<Entry>();
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(classes); ++i) {
        PyObject *cls, *forward;
        int kind;
        if (!PyArg_ParseTuple(PyTuple_GET_ITEM(classes, i), "O!iO", &PyType_Type, &cls, &kind, &forward)) return nullptr;
        PyTypeObject *t = reinterpret_cast<PyTypeObject *>(cls);
        if (get(t->tp_dict, names->__call__)) continue;   // (somebody's wrapper: every call of the class goes through it)
        Py_INCREF(cls);
        Py_INCREF(forward);
        Entry e{t, forward, static_cast<Kind>(kind)};
        e.mro = t->tp_mro;
        Py_INCREF(e.mro);
        for (Py_ssize_t k = 1; k < PyTuple_GET_SIZE(e.mro) && PyTuple_GET_ITEM(e.mro, k) != module; ++k)
            e.bases.push_back(reinterpret_cast<PyTypeObject *>(PyTuple_GET_ITEM(e.mro, k)));
        entries->push_back(e);
    }
    if (!found) {
        PyErr_SetString(PyExc_RuntimeError, "install: a function or dictionary is not where it was expected");
        return nullptr;
    }
    for (PyObject *o : {module, call[0], call[1], launch, ops_dict, lib_dict, funcptr, sym, asym, quant8}) Py_INCREF(o);
    g_module_type = module_type;
    g_module_call = call[0];
    g_call_impl = call[1];
    g_ops_dict = ops_dict;
    g_launch = launch;
    g_lib_dict = lib_dict;
    g_funcptr = reinterpret_cast<PyTypeObject *>(funcptr);
    g_sym_type = reinterpret_cast<PyTypeObject *>(sym);
    g_asym_type = reinterpret_cast<PyTypeObject *>(asym);
    g_quant8_type = reinterpret_cast<PyTypeObject *>(quant8);
    g_global_hooks = global_hooks;
    g_entries = entries;
    g_names = names;
    for (Entry &e : *entries) {
        e.call = g_module_call;
        if (e.kind < 0) continue;
        ModuleCall *own = PyObject_New(ModuleCall, &g_module_call_type);
        if (!own) return nullptr;
        own->call = module_call;
        own->owner = e.type;
        own->dict = nullptr;
        e.call = reinterpret_cast<PyObject *>(own);   // (kept for good)
        if (PyObject_SetAttr(reinterpret_cast<PyObject *>(e.type), names->__call__, e.call) < 0) return nullptr;
    }
    Py_RETURN_NONE;
}

// plain_call(module): whether a call of it is its class's forward as it was written and nothing else, so that it may be
// run natively
PyObject *m_plain_call(PyObject *, PyObject *module)
{
    return PyBool_FromLong(g_names && plain_torch() && plain_call(module, dict_of(module)));
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

#define FAST(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<fn>)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FAST("defer", m_defer),
                           FAST("quantize_rows", m_quantize_rows),
                           FAST("quantize_rows_8bit", m_quantize_rows_8bit),
                           FAST("linear4", m_linear4),
                           FAST("linear4_batched", m_linear4_batched),
                           FAST("linear8", m_linear8),
                           {"setup", m_setup, METH_VARARGS, nullptr},
                           {"forget_refused_rooms", m_forget_refused_rooms, METH_NOARGS, nullptr},
                           {"install", m_install, METH_VARARGS, nullptr},
                           {"plain_call", m_plain_call, METH_O, nullptr},
                           {nullptr, nullptr, 0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_duq_host", "host side of the ops (csrc/duq_host.cpp)", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// Whether the process is of the Python and the torch that this file was compiled with: it looks into objects of both.
static bool built_for_this_process()
{
    int major = 0, minor = 0;
    if (std::sscanf(Py_GetVersion(), "%d.%d", &major, &minor) != 2 || major != PY_MAJOR_VERSION || minor != PY_MINOR_VERSION) {
        PyErr_Format(PyExc_ImportError, "_duq_host was built for Python %d.%d", PY_MAJOR_VERSION, PY_MINOR_VERSION);
        return false;
    }
    PyObject *torch = PyImport_ImportModule("torch");
    PyObject *version = torch ? PyObject_GetAttrString(torch, "__version__") : nullptr;
    const char *v = version ? PyUnicode_AsUTF8(version) : nullptr;
    const size_t len = std::strlen(TORCH_VERSION);
    const bool same = v && !std::strncmp(v, TORCH_VERSION, len) && (v[len] == 0 || v[len] == '+');   // (2.10.0+rocm7.0)
    if (v && !same) PyErr_Format(PyExc_ImportError, "_duq_host was built for torch %s, this is %s", TORCH_VERSION, v);
    Py_XDECREF(version);
    Py_XDECREF(torch);
    return same;
}

PyMODINIT_FUNC PyInit__duq_host(void)
{
    if (!built_for_this_process()) return nullptr;
    g_fused_type.tp_name = "_duq_host.FusedCall";
    g_fused_type.tp_basicsize = sizeof(FusedCall);
    g_fused_type.tp_flags = Py_TPFLAGS_DEFAULT;
    g_fused_type.tp_new = fused_new;
    g_fused_type.tp_dealloc = fused_dealloc;
    g_fused_type.tp_methods = g_fused_methods;
    if (PyType_Ready(&g_fused_type) < 0) return nullptr;
    g_staged_type.tp_name = "_duq_host.Staged";
    g_staged_type.tp_basicsize = sizeof(Staged);
    g_staged_type.tp_flags = Py_TPFLAGS_DEFAULT;
    g_staged_type.tp_dealloc = staged_dealloc;
    g_staged_type.tp_methods = g_staged_methods;
    if (PyType_Ready(&g_staged_type) < 0) return nullptr;
    g_module_call_type.tp_name = "_duq_host.ModuleCall";
    g_module_call_type.tp_basicsize = sizeof(ModuleCall);
    g_module_call_type.tp_flags = Py_TPFLAGS_DEFAULT | Py_TPFLAGS_HAVE_VECTORCALL | Py_TPFLAGS_METHOD_DESCRIPTOR;
    g_module_call_type.tp_vectorcall_offset = offsetof(ModuleCall, call);
    g_module_call_type.tp_call = PyVectorcall_Call;
    g_module_call_type.tp_descr_get = module_call_get;
    g_module_call_type.tp_dictoffset = offsetof(ModuleCall, dict);
    g_module_call_type.tp_getattro = PyObject_GenericGetAttr;
    g_module_call_type.tp_setattro = PyObject_GenericSetAttr;
    if (PyType_Ready(&g_module_call_type) < 0) return nullptr;
    PyObject *m = PyModule_Create(&g_module);
    if (!m) return nullptr;
    Py_INCREF(&g_fused_type);
    if (PyModule_AddObject(m, "FusedCall", reinterpret_cast<PyObject *>(&g_fused_type)) < 0) return nullptr;
    Py_INCREF(&g_module_call_type);
    if (PyModule_AddObject(m, "ModuleCall", reinterpret_cast<PyObject *>(&g_module_call_type)) < 0) return nullptr;
    return m;
}
