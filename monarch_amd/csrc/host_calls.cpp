// The way from a Python call on plain tensors to the C ABI, in native code.
//
// A call on small tensors is bound by the host: a HIP launch takes 2.2 to 3.2 us, and the checks of a Python wrapper, a dozen
// attribute reads and a ctypes call took 1.6 to 4 us on top (RDMABuffer.read_into 4.2, staging.pack 5.3, all_reduce of eight
// tensors 6.6, FlatBucket.unpack 0.25 per tensor).  The functions here make the same checks on the tensors' C++ objects and
// call the library.  They take a call only where every check passes on plain tensors: exactly torch.Tensor or Parameter, on a
// GPU, strided, with storage of its own and not wrapped by a transform.  Anything else (another type, a check that fails, a
// sequence that is no list or tuple) they leave alone and return NOT_TAKEN, and the Python code behind them runs as it would
// without them: it raises what it always raised and takes what it always took.  Nothing is kept from one call to the next.
//
// The library is called without the interpreter's lock, as ctypes does.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/version.h>

#include <climits>
#include <cstdint>
#include <cstring>

#include "../../include/monarch_hip.h"

namespace {

constexpr long kNotTaken = LONG_MIN;  // no status (a C int), no negated one and no count
constexpr Py_ssize_t kMaxItems = 64;  // tensors or views of one call; longer lists are left to the general path

PyTypeObject* g_slice_type = nullptr;  // monarch_amd.ndslice.Slice
PyObject* g_addr_name = nullptr;       // "_addr": the address of a Slice's mhip_slice_t

// ---- tensors ----

const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.defined()) return nullptr;
    const c10::TensorImpl* impl = t.unsafeGetTensorImpl();
    constexpr c10::DispatchKeySet wrapped({c10::DispatchKey::Python, c10::DispatchKey::FuncTorchBatched, c10::DispatchKey::FuncTorchGradWrapper,
                                           c10::DispatchKey::Functionalize, c10::DispatchKey::ZeroTensor});
    if (!t.is_cuda() || t.layout() != c10::kStrided || !impl->has_storage() || impl->has_symbolic_sizes_strides() ||
        impl->key_set().has_any(wrapped))
        return nullptr;
    return &t;
}

const at::Tensor* plain_contiguous(PyObject* o) {
    const at::Tensor* t = plain(o);
    return t != nullptr && t->is_contiguous() ? t : nullptr;
}

uint64_t bytes_of(const at::Tensor& t) { return (uint64_t)t.numel() * t.itemsize(); }

// Code of an element type the reductions take (the numbers of mhip_dtype are those of c10::ScalarType), or -1.
int reduce_code(const at::Tensor& t) {
    switch (t.scalar_type()) {
        case c10::ScalarType::Byte: case c10::ScalarType::Char: case c10::ScalarType::Int: case c10::ScalarType::Long:
        case c10::ScalarType::Half: case c10::ScalarType::Float: case c10::ScalarType::Double: case c10::ScalarType::BFloat16:
            return (int)t.scalar_type();
        default: return -1;
    }
}

mhip_stream_t current_stream() { return c10::hip::getCurrentHIPStream().stream(); }

// ---- Python objects ----

struct Items {  // of a list or a tuple, borrowed
    PyObject** at = nullptr;
    Py_ssize_t n = -1;
    explicit Items(PyObject* o) {
        if (PyList_CheckExact(o) || PyTuple_CheckExact(o)) {
            at = PySequence_Fast_ITEMS(o);
            n = PySequence_Fast_GET_SIZE(o);
        }
    }
    bool few() const { return n >= 1 && n <= kMaxItems; }
};

bool to_u64(PyObject* o, uint64_t* out) {
    if (!PyLong_Check(o)) return false;
    const unsigned long long v = PyLong_AsUnsignedLongLong(o);
    if (v == (unsigned long long)-1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    *out = v;
    return true;
}

// The C struct of a Slice; null for any other object.
const mhip_slice_t* slice_of(PyObject* o) {
    if (Py_TYPE(o) != g_slice_type) return nullptr;
    PyObject* addr = PyObject_GetAttr(o, g_addr_name);
    uint64_t v = 0;
    const bool ok = addr != nullptr && to_u64(addr, &v);
    Py_XDECREF(addr);
    if (!ok) PyErr_Clear();
    return ok ? reinterpret_cast<const mhip_slice_t*>((uintptr_t)v) : nullptr;
}

// Elements of a view and the last one it reaches; false where that overflows.
bool extent(const mhip_slice_t& s, uint64_t* len, uint64_t* hi) {
    *len = 1;
    *hi = s.offset;
    for (uint32_t k = 0; k < s.ndim; ++k)
        if (__builtin_mul_overflow(*len, s.sizes[k], len)) return false;
    if (*len == 0) return true;
    for (uint32_t k = 0; k < s.ndim; ++k) {
        uint64_t reach;
        if (__builtin_mul_overflow(s.sizes[k] - 1, s.strides[k], &reach) || __builtin_add_overflow(*hi, reach, hi)) return false;
    }
    return true;
}

// Whether a view lies inside the storage of `base` and `buffer` is a staging buffer of exactly its size.
bool fits(const at::Tensor& base, const mhip_slice_t& s, const at::Tensor& buffer) {
    uint64_t len, hi, nbytes;
    if (!extent(s, &len, &hi) || __builtin_mul_overflow(len, (uint64_t)base.itemsize(), &nbytes)) return false;
    if (len != 0 && hi >= base.storage().nbytes() / base.itemsize()) return false;
    return buffer.device() == base.device() && bytes_of(buffer) == nbytes;
}

// Holds objects of lists, tensors and Slices, while the library runs without the interpreter's lock: another thread may take
// them out of the list meanwhile, and the library reads a Slice's memory and launches on a tensor's.  (The arguments themselves
// are held by the caller.)
class Held {
public:
    ~Held() {
        for (Py_ssize_t i = 0; i < n_; ++i) Py_DECREF(at_[i]);
    }
    PyObject* add(PyObject* o) {
        Py_INCREF(o);
        return at_[n_++] = o;
    }
private:
    PyObject* at_[3 * kMaxItems];  // a call has three lists at most
    Py_ssize_t n_ = 0;
};

template <typename F>
long unlocked(F&& f) {
    struct Unlock {
        PyThreadState* state = PyEval_SaveThread();
        ~Unlock() { PyEval_RestoreThread(state); }
    } unlock;
    return f();
}

// Every function below returns the library's status or NOT_TAKEN; no C++ exception leaves it.
template <long (*F)(PyObject* const*), int NARGS>
PyObject* entry(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != NARGS) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    long rc = kNotTaken;
    try {
        rc = F(args);
    } catch (...) {
        rc = kNotTaken;
    }
    if (PyErr_Occurred()) PyErr_Clear();
    return PyLong_FromLong(rc);
}

// ---- staging ----

// (pack, base, slice, buffer)
long slice_copy(PyObject* const* a) {
    const at::Tensor *base = plain(a[1]), *buffer = plain_contiguous(a[3]);
    const mhip_slice_t* s = slice_of(a[2]);
    if (base == nullptr || buffer == nullptr || s == nullptr || !fits(*base, *s, *buffer)) return kNotTaken;
    void *mem = base->storage().mutable_data(), *packed = buffer->data_ptr();
    const uint32_t size = (uint32_t)base->itemsize();
    const mhip_stream_t stream = current_stream();
    if (a[0] == Py_True) return unlocked([&] { return mhip_slice_pack(packed, mem, s, size, stream); });
    return unlocked([&] { return mhip_slice_unpack(mem, packed, s, size, stream); });
}

// (pack, base, slices, buffers)
long slice_copy_many(PyObject* const* a) {
    const at::Tensor* base = plain(a[1]);
    const Items views(a[2]), buffers(a[3]);
    if (base == nullptr || !views.few() || views.n != buffers.n) return kNotTaken;
    mhip_slice_t slices[kMaxItems];
    void* ptrs[kMaxItems];
    Held held;
    for (Py_ssize_t i = 0; i < views.n; ++i) {
        const mhip_slice_t* s = slice_of(held.add(views.at[i]));
        const at::Tensor* buffer = plain_contiguous(held.add(buffers.at[i]));
        if (s == nullptr || buffer == nullptr || !fits(*base, *s, *buffer)) return kNotTaken;
        slices[i] = *s;
        ptrs[i] = buffer->data_ptr();
    }
    void* mem = base->storage().mutable_data();
    const uint32_t n = (uint32_t)views.n, size = (uint32_t)base->itemsize();
    const mhip_stream_t stream = current_stream();
    if (a[0] == Py_True) return unlocked([&] { return mhip_slice_pack_many(ptrs, mem, slices, n, size, stream); });
    return unlocked([&] { return mhip_slice_unpack_many(mem, ptrs, slices, n, size, stream); });
}

// (read, address, size, tensor, offset): a registered buffer's bytes into a tensor, or a tensor's into the buffer
long rdma_copy(PyObject* const* a) {
    uint64_t addr, size, offset;
    const at::Tensor* t = plain_contiguous(a[3]);
    if (t == nullptr || t->dim() != 1 || t->scalar_type() != c10::ScalarType::Byte) return kNotTaken;
    if (!to_u64(a[1], &addr) || !to_u64(a[2], &size) || !to_u64(a[4], &offset)) return kNotTaken;
    const uint64_t n = (uint64_t)t->numel();
    if (offset > size || n > size - offset) return kNotTaken;
    const mhip_rdma_buffer_t local{t->data_ptr(), (size_t)n};
    const mhip_rdma_buffer_t remote{reinterpret_cast<void*>((uintptr_t)(addr + offset)), (size_t)(size - offset)};
    const mhip_stream_t stream = current_stream();
    if (a[0] == Py_True) return unlocked([&] { return mhip_buffer_write_from(&local, &remote, stream); });
    return unlocked([&] { return mhip_buffer_read_into(&local, &remote, stream); });
}

// (destinations, sources, sizes, largest segment) -> requests posted, or minus the status
long transfer_many(PyObject* const* a) {
    const Items dst(a[0]), src(a[1]), len(a[2]);
    uint64_t max_segment;
    if (!len.few() || dst.n != len.n || src.n != len.n || !to_u64(a[3], &max_segment)) return kNotTaken;
    void *d[kMaxItems], *s[kMaxItems];
    size_t bytes[kMaxItems];
    for (Py_ssize_t i = 0; i < len.n; ++i) {
        uint64_t x, y, n;
        if (!to_u64(dst.at[i], &x) || !to_u64(src.at[i], &y) || !to_u64(len.at[i], &n)) return kNotTaken;
        d[i] = reinterpret_cast<void*>((uintptr_t)x);
        s[i] = reinterpret_cast<void*>((uintptr_t)y);
        bytes[i] = (size_t)n;
    }
    uint32_t posted = 0;
    const uint32_t n = (uint32_t)len.n;
    const mhip_stream_t stream = current_stream();
    const long rc = unlocked([&] { return mhip_buffer_transfer_many(d, s, bytes, n, (size_t)max_segment, stream, &posted); });
    return rc == MHIP_SUCCESS ? (long)posted : -rc;
}

// ---- reductions ----

// The members of a group: contiguous tensors of one type and size.
bool members(const Items& group, c10::ScalarType type, int64_t numel, const void** ptrs, Held* held) {
    if (!group.few()) return false;
    for (Py_ssize_t i = 0; i < group.n; ++i) {
        const at::Tensor* t = plain_contiguous(held->add(group.at[i]));
        if (t == nullptr || t->scalar_type() != type || t->numel() != numel) return false;
        ptrs[i] = t->data_ptr();
    }
    return true;
}

// (out, group, op)
long reduce(PyObject* const* a) {
    const at::Tensor* out = plain_contiguous(a[0]);
    const Items group(a[1]);
    uint64_t op;
    const void* ptrs[kMaxItems];
    Held held;
    if (out == nullptr || !to_u64(a[2], &op) || op > INT_MAX) return kNotTaken;
    const int code = reduce_code(*out);
    if (code < 0 || !members(group, out->scalar_type(), out->numel(), ptrs, &held)) return kNotTaken;
    void* dst = out->data_ptr();
    const uint64_t numel = (uint64_t)out->numel();
    const mhip_stream_t stream = current_stream();
    return unlocked([&] { return mhip_reduce(dst, ptrs, (uint32_t)group.n, numel, code, (int)op, stream); });
}

// (out, group): the members one after the other
long stack(PyObject* const* a) {
    const at::Tensor* out = plain_contiguous(a[0]);
    const Items group(a[1]);
    const void* ptrs[kMaxItems];
    Held held;
    if (out == nullptr || !group.few() || out->numel() % group.n != 0) return kNotTaken;
    const int64_t numel = out->numel() / group.n;
    if (!members(group, out->scalar_type(), numel, ptrs, &held)) return kNotTaken;
    void* dst = out->data_ptr();
    const uint32_t size = (uint32_t)out->itemsize();
    const mhip_stream_t stream = current_stream();
    return unlocked([&] { return mhip_stack(dst, ptrs, (uint32_t)group.n, (uint64_t)numel, size, stream); });
}

// (outs, out views, group, in view, op)
long reduce_scatter(PyObject* const* a) {
    const Items outs(a[0]), views(a[1]), group(a[2]);
    const mhip_slice_t* in_view = slice_of(a[3]);
    uint64_t op;
    if (!outs.few() || outs.n != views.n || !group.few() || in_view == nullptr || !to_u64(a[4], &op) || op > INT_MAX) return kNotTaken;
    mhip_slice_t slices[kMaxItems];
    void* dst[kMaxItems];
    const void* src[kMaxItems];
    Held held;
    int code = -1;
    for (Py_ssize_t i = 0; i < outs.n; ++i) {
        const at::Tensor* t = plain_contiguous(held.add(outs.at[i]));
        const mhip_slice_t* s = slice_of(held.add(views.at[i]));
        uint64_t len, hi;
        if (t == nullptr || s == nullptr || !extent(*s, &len, &hi) || (uint64_t)t->numel() != len) return kNotTaken;
        if (i == 0) code = reduce_code(*t);
        slices[i] = *s;
        dst[i] = t->data_ptr();
    }
    if (code < 0) return kNotTaken;
    for (Py_ssize_t i = 0; i < group.n; ++i) {
        const at::Tensor* t = plain(held.add(group.at[i]));
        if (t == nullptr) return kNotTaken;
        src[i] = t->data_ptr();
    }
    const mhip_stream_t stream = current_stream();
    return unlocked([&] {
        return mhip_reduce_scatter(dst, slices, (uint32_t)outs.n, src, in_view, 0, (uint32_t)group.n, code, (int)op, stream);
    });
}

// ---- flat buckets ----

struct Bucket {  // its device tables
    const at::Tensor* offsets = nullptr;
    void* tensors = nullptr;
    uint32_t n = 0;
    uint64_t total = 0;
    const uint32_t* index = nullptr;
};

// tables: the pointer table, the offsets table, elements, the block index or None
bool bucket_of(PyObject* ptrs, PyObject* offsets, PyObject* total, PyObject* index, Bucket* b) {
    const at::Tensor *p = plain_contiguous(ptrs), *o = plain_contiguous(offsets);
    if (p == nullptr || o == nullptr || !to_u64(total, &b->total)) return false;
    if (p->scalar_type() != c10::ScalarType::Long || p->numel() != o->numel() - 1 || p->device() != o->device()) return false;
    if (index != Py_None) {
        const at::Tensor* t = plain_contiguous(index);
        if (t == nullptr) return false;
        b->index = static_cast<const uint32_t*>(t->data_ptr());
    }
    b->offsets = o;
    b->tensors = p->data_ptr();
    b->n = (uint32_t)p->numel();
    return true;
}

// (pack, flat, pointer table, offsets, elements, index, a tensor of the flat buffer's type or None)
long flat_copy(PyObject* const* a) {
    Bucket b;
    const at::Tensor* flat = plain_contiguous(a[1]);
    if (flat == nullptr || !bucket_of(a[2], a[3], a[4], a[5], &b)) return kNotTaken;
    if (flat->device() != b.offsets->device() || (uint64_t)flat->numel() != b.total) return kNotTaken;
    if (a[6] != Py_None) {
        const at::Tensor* like = plain(a[6]);
        if (like == nullptr || like->scalar_type() != flat->scalar_type()) return kNotTaken;
    }
    void* mem = flat->data_ptr();
    const uint64_t* offsets = static_cast<const uint64_t*>(b.offsets->data_ptr());
    const uint32_t size = (uint32_t)flat->itemsize();
    const mhip_stream_t stream = current_stream();
    if (a[0] == Py_True)
        return unlocked([&] { return mhip_flat_pack(mem, static_cast<const void* const*>(b.tensors), offsets, b.n, b.total, size, b.index, stream); });
    return unlocked([&] { return mhip_flat_unpack(static_cast<void* const*>(b.tensors), mem, offsets, b.n, b.total, size, b.index, stream); });
}

// A payload of n elements on the bucket's device: one byte and a 1024th of a float each.
bool payload(PyObject* q, PyObject* scales, const Bucket& b, void** qp, float** sp) {
    const at::Tensor *c = plain_contiguous(q), *s = plain_contiguous(scales);
    if (c == nullptr || s == nullptr || c->device() != b.offsets->device() || s->device() != b.offsets->device()) return false;
    if (c->itemsize() != 1 || (uint64_t)c->numel() != b.total) return false;
    if (s->scalar_type() != c10::ScalarType::Float || (uint64_t)s->numel() != (b.total + 1023) / 1024) return false;
    *qp = c->data_ptr();
    *sp = static_cast<float*>(s->data_ptr());
    return true;
}

// (pointer table, offsets, elements, index, codes, scales)
long quantize_bucket(PyObject* const* a) {
    Bucket b;
    void* q;
    float* scales;
    if (!bucket_of(a[0], a[1], a[2], a[3], &b) || !payload(a[4], a[5], b, &q, &scales)) return kNotTaken;
    const uint64_t* offsets = static_cast<const uint64_t*>(b.offsets->data_ptr());
    const mhip_stream_t stream = current_stream();
    return unlocked([&] {
        return mhip_fp8_quantize_bucket(static_cast<uint8_t*>(q), scales, static_cast<const void* const*>(b.tensors), offsets, b.n, b.total, 1024,
                                        b.index, stream);
    });
}

// (pointer table, offsets, elements, index, codes of the peers, scales of the peers)
long dequant_accumulate_bucket(PyObject* const* a) {
    Bucket b;
    const Items qs(a[4]), ss(a[5]);
    if (!bucket_of(a[0], a[1], a[2], a[3], &b) || !qs.few() || qs.n != ss.n) return kNotTaken;
    const uint8_t* q[kMaxItems];
    const float* scales[kMaxItems];
    Held held;
    for (Py_ssize_t i = 0; i < qs.n; ++i) {
        void* qp;
        float* sp;
        if (!payload(held.add(qs.at[i]), held.add(ss.at[i]), b, &qp, &sp)) return kNotTaken;
        q[i] = static_cast<const uint8_t*>(qp);
        scales[i] = sp;
    }
    const uint64_t* offsets = static_cast<const uint64_t*>(b.offsets->data_ptr());
    const mhip_stream_t stream = current_stream();
    return unlocked([&] {
        return mhip_fp8_dequant_accumulate_bucket_many(static_cast<void* const*>(b.tensors), q, scales, (uint32_t)qs.n, offsets, b.n, b.total,
                                                       1024, b.index, stream);
    });
}

// (tensors, sizes as 64-bit integers, flat) -> the tensors' addresses as bytes, or None: contiguous tensors of these sizes,
// of the element size of the flat buffer, which holds them all, and on its device
PyObject* tensor_addresses(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    if (nargs != 3) {
        PyErr_SetString(PyExc_TypeError, "wrong number of arguments");
        return nullptr;
    }
    PyObject* out = nullptr;
    try {
        const Items tensors(a[0]);
        const at::Tensor* flat = plain_contiguous(a[2]);
        int64_t total = 0;
        if (flat != nullptr && PyBytes_CheckExact(a[1]) && tensors.n >= 0 && PyBytes_GET_SIZE(a[1]) == tensors.n * 8) {
            out = PyBytes_FromStringAndSize(nullptr, tensors.n * 8);
            if (out == nullptr) return nullptr;
            char* to = PyBytes_AS_STRING(out);
            const char* sizes = PyBytes_AS_STRING(a[1]);
            for (Py_ssize_t i = 0; i < tensors.n; ++i) {
                const at::Tensor* t = plain_contiguous(tensors.at[i]);
                int64_t size;
                memcpy(&size, sizes + i * 8, 8);
                if (t == nullptr || t->numel() != size || t->itemsize() != flat->itemsize() || t->device() != flat->device()) {
                    Py_CLEAR(out);
                    break;
                }
                const uint64_t address = (uint64_t)(uintptr_t)t->data_ptr();
                memcpy(to + i * 8, &address, 8);
                total += size;
            }
            if (out != nullptr && total != flat->numel()) Py_CLEAR(out);
        }
    } catch (...) {
        Py_CLEAR(out);
    }
    if (out != nullptr) return out;
    if (PyErr_Occurred()) PyErr_Clear();
    Py_RETURN_NONE;
}

PyObject* set_slice_type(PyObject*, PyObject* type) {
    if (!PyType_Check(type)) {
        PyErr_SetString(PyExc_TypeError, "a type is needed");
        return nullptr;
    }
    Py_INCREF(type);
    Py_XDECREF(reinterpret_cast<PyObject*>(g_slice_type));
    g_slice_type = reinterpret_cast<PyTypeObject*>(type);
    Py_RETURN_NONE;
}

template <long (*F)(PyObject* const*), int NARGS>
PyMethodDef method(const char* name) {
    return {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&entry<F, NARGS>)), METH_FASTCALL, nullptr};
}

PyMethodDef g_methods[] = {
    method<slice_copy, 4>("slice_copy"),
    method<slice_copy_many, 4>("slice_copy_many"),
    method<rdma_copy, 5>("rdma_copy"),
    method<transfer_many, 4>("transfer_many"),
    method<reduce, 3>("reduce"),
    method<stack, 2>("stack"),
    method<reduce_scatter, 5>("reduce_scatter"),
    method<flat_copy, 7>("flat_copy"),
    method<quantize_bucket, 6>("quantize_bucket"),
    method<dequant_accumulate_bucket, 6>("dequant_accumulate_bucket"),
    {"tensor_addresses", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)(void)>(&tensor_addresses)), METH_FASTCALL, nullptr},
    {"set_slice_type", set_slice_type, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr},
};

PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_host_calls", nullptr, -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host_calls() {
    g_addr_name = PyUnicode_InternFromString("_addr");
    PyObject* m = g_addr_name != nullptr ? PyModule_Create(&g_module) : nullptr;
    if (m != nullptr) {
        PyModule_AddIntConstant(m, "NOT_TAKEN", kNotTaken);
        PyModule_AddStringConstant(m, "TORCH_VERSION", TORCH_VERSION);  // whose layouts the checks read; monarch_amd/_native.py compares it
    }
    return m;
}
