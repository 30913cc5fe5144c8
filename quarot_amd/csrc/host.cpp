// Host side of the package's hot entry points: argument checks, output allocation and the call into libquarot_hip.so as
// one CPython function each, where the Python wrappers take 10 - 25 us per call -- longer than most decode kernels run.
//
// Every function returns None instead of raising when the arguments are not the plain case it serves (a tensor subclass, a
// tensor that is not contiguous or not on the current device, a wrong dtype or size, an empty input, a refusal by the
// library, a call under a transform or a tracer): the Python wrapper then takes its general route, which handles the case or
// raises the documented error.  A HIP error is raised here.
// Launches go to torch's current stream, outputs and scratch come from torch's allocator.
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ops/empty.h>
#include <c10/hip/HIPCachingAllocator.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>

#include <atomic>
#include <stdexcept>
#include <string>

#include "../../include/quarot_hip.h"

namespace {

// A tensor with memory of its own and nothing that watches what is done to it: no subclass, no wrapper of a function
// transform (vmap, jvp, functionalisation), no tangent of forward-mode differentiation, no active tracer or dispatch mode.
const at::Tensor* tensor(PyObject* o) {
    using c10::DispatchKey;
    constexpr c10::DispatchKeySet wrapped{DispatchKey::Python, DispatchKey::Functionalize, DispatchKey::FuncTorchBatched,
                                          DispatchKey::FuncTorchGradWrapper};
    constexpr c10::DispatchKeySet modes{DispatchKey::Python, DispatchKey::Functionalize, DispatchKey::Tracer,
                                        DispatchKey::FuncTorchDynamicLayerFrontMode};
    if (!THPVariable_CheckExact(o)) return nullptr;
    const at::Tensor* t = &THPVariable_Unpack(o);
    if (t->key_set().has_any(wrapped) || c10::impl::tls_local_dispatch_key_set().included_.has_any(modes) || t->_fw_grad(0).defined())
        return nullptr;
    return t;
}

bool plain(const at::Tensor* t, at::ScalarType dtype, int device) {
    return t && t->is_cuda() && t->scalar_type() == dtype && t->device().index() == device && t->is_contiguous();
}
// an optional operand: None is fine and has no address
bool plain_or_none(PyObject* o, at::ScalarType dtype, int device, const at::Tensor** out) {
    *out = nullptr;
    if (o == Py_None) return true;
    *out = tensor(o);
    return plain(*out, dtype, device);
}

constexpr auto kHalf = at::kHalf;
constexpr auto kByte = at::kByte;

// the tensor's device if it is the current one, else -1 (which no tensor on a GPU has)
int device_of(const at::Tensor* t) {
    if (!t || !t->is_cuda()) return -1;
    const int d = (int)t->device().index();
    return d == (int)c10::hip::current_device() ? d : -1;
}
void* stream(int device) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }
// Allocations and launches run without the interpreter's lock: an allocation may have to give memory back first, a launch waits
// while the queue is full, and other Python threads go on meanwhile.  Where this one is the interpreter's only thread the lock stays:
// giving it away and taking it back costs about 0.2 us of a call's 4.5.
bool only_thread() {
    PyThreadState* const own = PyThreadState_Get();
    return PyInterpreterState_ThreadHead(PyThreadState_GetInterpreter(own)) == own && !PyThreadState_Next(own);
}
struct Unlocked {
    PyThreadState* const state = only_thread() ? nullptr : PyEval_SaveThread();
    ~Unlocked() {
        if (state) PyEval_RestoreThread(state);
    }
};
at::Tensor fresh(at::IntArrayRef sizes, at::ScalarType dtype, int device) {
    return at::empty(sizes, at::TensorOptions().dtype(dtype).device(at::Device(at::kCUDA, (c10::DeviceIndex)device)));
}
void* ptr(const at::Tensor* t) { return t ? t->data_ptr() : nullptr; }

// What a call of the library came to.  Its own refusals are negative codes and leave the case to the general route.  A positive
// code is a HIP error, which the library has taken off the runtime's record: a second attempt by the general route would
// report success over it.
bool success(int rc) {
    if (rc > 0) throw std::runtime_error("libquarot_hip: " + std::string(qr_strerror(rc)) + " (code " + std::to_string(rc) + ")");
    return rc == QR_OK;
}
template <typename Call>
bool done(Call&& call) {
    int rc;
    {
        const Unlocked unlocked;
        rc = call();
    }
    return success(rc);
}

PyObject* none() { Py_RETURN_NONE; }
PyObject* wrap(at::Tensor&& t) { return THPVariable_Wrap(std::move(t)); }
PyObject* wrap2(at::Tensor&& a, at::Tensor&& b) {
    PyObject* pa = wrap(std::move(a));
    PyObject* pb = pa ? wrap(std::move(b)) : nullptr;
    if (!pb) {
        Py_XDECREF(pa);
        return nullptr;
    }
    PyObject* t = PyTuple_New(2);
    if (!t) {
        Py_DECREF(pa);
        Py_DECREF(pb);
        return nullptr;
    }
    PyTuple_SET_ITEM(t, 0, pa);
    PyTuple_SET_ITEM(t, 1, pb);
    return t;
}

// rows of a quantiser's input: fp16 [..., n], contiguous, on the current device
struct Rows {
    const at::Tensor* x;
    int device;
    int64_t rows, n;
    bool ok;
};
Rows rows_of(PyObject* o) {
    Rows r{tensor(o), -1, 0, 0, false};
    r.device = device_of(r.x);
    if (!plain(r.x, kHalf, r.device) || r.x->dim() < 1) return r;
    r.n = r.x->size(-1);
    r.ok = r.n > 0 && r.x->numel() > 0;
    if (r.ok) r.rows = r.x->numel() / r.n;
    return r;
}
// codes [..., n / 2] and scales with the shape torch.max(dim=-1)[0].unsqueeze(1) has
struct Packed {
    at::Tensor codes, scales;
};
Packed packed_for(const Rows& r, int lead) {                // lead: how many leading dimensions of x stay
    c10::SmallVector<int64_t, 6> qs(r.x->sizes().begin(), r.x->sizes().begin() + lead), ss;
    qs.push_back((r.n + 1) / 2);
    for (int i = 0; i < lead; ++i) {
        if (i == 1) ss.push_back(1);
        ss.push_back(r.x->size(i));
    }
    if (lead <= 1) ss.push_back(1);
    return Packed{fresh(qs, kByte, r.device), fresh(ss, kHalf, r.device)};
}

bool arg_int(PyObject* o, long long* v) {
    *v = PyLong_AsLongLong(o);
    if (*v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}
bool arg_float(PyObject* o, double* v) {
    *v = PyFloat_AsDouble(o);
    if (*v == -1.0 && PyErr_Occurred()) {
        PyErr_Clear();
        return false;
    }
    return true;
}

bool arg_bool(PyObject* o, bool* v) {
    const int truth = PyObject_IsTrue(o);
    if (truth < 0) PyErr_Clear();
    *v = truth > 0;
    return truth >= 0;
}

#define QR_ARGS(COUNT)                                                     \
    if (nargs != (COUNT)) {                                                \
        PyErr_SetString(PyExc_TypeError, "expected " #COUNT " arguments"); \
        return nullptr;                                                    \
    }                                                                      \
    HANDLE_TH_ERRORS
#define QR_END END_HANDLE_TH_ERRORS

// quantize_rows(x, clip) -> (codes, scales)
PyObject* quantize_rows(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(2)
    const Rows r = rows_of(a[0]);
    double clip;
    if (!r.ok || !arg_float(a[1], &clip)) return none();
    Packed p;
    const auto call = [&] {
        p = packed_for(r, (int)r.x->dim() - 1);
        return qr_quantize_rows_f16_i4(r.x->data_ptr(), (float)clip, r.rows, r.n, p.codes.data_ptr(), p.scales.data_ptr(),
                                       stream(r.device));
    };
    if (!done(call)) return none();
    return wrap2(std::move(p.codes), std::move(p.scales));
    QR_END
}

// rmsnorm(x, mean_dim, eps) -> y
PyObject* rmsnorm(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(3)
    const Rows r = rows_of(a[0]);
    long long mean_dim;
    double eps;
    if (!r.ok || !arg_int(a[1], &mean_dim) || !arg_float(a[2], &eps) || mean_dim > 0x7fffffff) return none();
    at::Tensor y;
    const auto call = [&] {
        y = fresh(r.x->sizes(), kHalf, r.device);
        return qr_rmsnorm_f16(r.x->data_ptr(), r.rows, r.n, (int)mean_dim, (float)eps, y.data_ptr(), stream(r.device));
    };
    if (!done(call)) return none();
    return wrap(std::move(y));
    QR_END
}

// rmsnorm_quantize(x, mean_dim, eps, clip) -> (codes, scales)
PyObject* rmsnorm_quantize(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(4)
    const Rows r = rows_of(a[0]);
    long long mean_dim;
    double eps, clip;
    if (!r.ok || r.n % 8 || !arg_int(a[1], &mean_dim) || !arg_float(a[2], &eps) || !arg_float(a[3], &clip) || mean_dim > 0x7fffffff)
        return none();
    Packed p;
    const auto call = [&] {
        p = packed_for(r, (int)r.x->dim() - 1);
        return qr_rmsnorm_quantize_f16_i4(r.x->data_ptr(), r.rows, r.n, (int)mean_dim, (float)eps, (float)clip, p.codes.data_ptr(),
                                          p.scales.data_ptr(), nullptr, stream(r.device));
    };
    if (!done(call)) return none();
    return wrap2(std::move(p.codes), std::move(p.scales));
    QR_END
}

// heads_hadamard_quantize(x [..., heads, 128], clip, hadK or None) -> (codes, scales) of the rows reshaped to [..., heads * 128]
PyObject* heads_hadamard_quantize(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(3)
    Rows r = rows_of(a[0]);
    double clip;
    if (!r.ok || r.x->dim() < 2 || r.n != 128 || !arg_float(a[1], &clip)) return none();
    const int64_t heads = r.x->size(-2);
    const at::Tensor* hadK;
    if (!plain_or_none(a[2], kHalf, r.device, &hadK) || heads > 64 || (hadK && hadK->numel() != heads * heads)) return none();
    r.n = heads * 128;
    r.rows = r.x->numel() / r.n;
    Packed p;
    const auto call = [&] {
        p = packed_for(r, (int)r.x->dim() - 2);
        return qr_heads_hadamard_quantize_f16_i4(r.x->data_ptr(), r.rows, (int)heads, 128, ptr(hadK), (float)clip, p.codes.data_ptr(),
                                                 p.scales.data_ptr(), nullptr, stream(r.device));
    };
    if (!done(call)) return none();
    return wrap2(std::move(p.codes), std::move(p.scales));
    QR_END
}

// A Hadamard factor as the library takes it: None (K = 1), the table of the mode's dtype, or its sign words.
bool table_arg(PyObject* o, long long mode, int64_t K, int device, const at::Tensor** out) {
    *out = nullptr;
    if (K <= 1) return true;
    const bool signs = (mode & QR_HADK_SIGNS) != 0;
    *out = tensor(o);
    const auto dtype = signs ? kByte : (mode & ~(QR_HADK_SIGNS | QR_HAD_FP32)) == QR_DTYPE_F32 || (mode & QR_HAD_FP32) ? at::kFloat : kHalf;
    return plain(*out, dtype, device) && (*out)->numel() == (signs ? K * ((K + 31) / 32) * 4 : K * K);
}

// hadamard(x, hadK or None, K, mode, scale) -> y: qr_hadamard on fp16 rows (mode QR_DTYPE_F16, optionally | QR_HAD_FP32)
PyObject* hadamard(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(5)
    const Rows r = rows_of(a[0]);
    long long K, mode;
    double scale;
    const at::Tensor* table;
    if (!r.ok || !arg_int(a[2], &K) || !arg_int(a[3], &mode) || !arg_float(a[4], &scale) || r.n > 0x7fffffff ||
        (mode & ~QR_HAD_FP32) != QR_DTYPE_F16 || !table_arg(a[1], mode, K, r.device, &table))
        return none();
    at::Tensor y;
    const auto call = [&] {
        y = fresh(r.x->sizes(), kHalf, r.device);
        return qr_hadamard(r.x->data_ptr(), y.data_ptr(), r.rows, (int)r.n, (int)K, ptr(table), (int)mode, (float)scale,
                           stream(r.device));
    };
    if (!done(call)) return none();
    return wrap(std::move(y));
    QR_END
}

// hadamard_quantize(x, table, K, mode, scale, clip) -> (codes, scales)
PyObject* hadamard_quantize(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(6)
    const Rows r = rows_of(a[0]);
    long long K, mode;
    double scale, clip;
    const at::Tensor* table;
    if (!r.ok || r.n % 2 || r.n > 0x7fffffff || !arg_int(a[2], &K) || !arg_int(a[3], &mode) || !arg_float(a[4], &scale) ||
        !arg_float(a[5], &clip) || !table_arg(a[1], mode, K, r.device, &table))
        return none();
    Packed p;
    const auto call = [&] {
        p = packed_for(r, (int)r.x->dim() - 1);
        return qr_hadamard_quantize_f16_i4(r.x->data_ptr(), r.rows, (int)r.n, (int)K, ptr(table), (int)mode, (float)scale, (float)clip,
                                           p.codes.data_ptr(), p.scales.data_ptr(), nullptr, stream(r.device));
    };
    if (!done(call)) return none();
    return wrap2(std::move(p.codes), std::move(p.scales));
    QR_END
}

// weight [N, K / 2], its scales and an optional bias
struct Weight {
    const at::Tensor *w, *s, *b;
    int64_t N;
};
bool weight_args(PyObject* w, PyObject* s, PyObject* b, int64_t half_k, int device, Weight* out) {
    out->w = tensor(w);
    out->s = tensor(s);
    if (!plain(out->w, kByte, device) || !plain(out->s, kHalf, device) || !plain_or_none(b, kHalf, device, &out->b)) return false;
    if (out->w->dim() != 2 || out->w->size(1) != half_k) return false;
    out->N = out->w->size(0);
    return out->N > 0 && out->s->numel() == out->N && (!out->b || out->b->numel() == out->N);
}

// What the library's plan uses as scratch of the product of a shape, what it would rather have to spread an operand, and what the fused call needs
// besides.  The plans behind these are 0.2 to 1.2 us of estimates, as much as a quarter of a call, and a program has few shapes: every thread keeps
// its last ones (333 tokens, norm, quantiser, 3 x 4096 x 4096 30.0 -> 29.1 us of host time, 156 tokens, Hadamard + 5120 x 5120 11.6 -> 10.9).
struct Slabs {
    size_t used, spread, fixed;
};
const Slabs& slab_bytes(int64_t M, int64_t N, int64_t K, int device) {
    struct Shape {
        int64_t M = -1, N = 0, K = 0;
        int device = -1;
        Slabs bytes;
    };
    thread_local Shape shapes[64];
    Shape& s = shapes[((uint64_t)(M * 31 + N * 17 + K * 7 + device) * 0x9E3779B97F4A7C15ull) >> 58];
    if (s.M != M || s.N != N || s.K != K || s.device != device) {
        const size_t asked = qr_workspace_bytes(M, N, K);
        Slabs bytes{0, qr_linear_spread_bytes(M, N, K), qr_quantized_linear_workspace_bytes(M, N, K) - asked};
        if (asked) qr_linear_plan(M, N, K, asked, &bytes.used);
        s.M = M, s.N = N, s.K = K, s.device = device, s.bytes = bytes;
    }
    return s.bytes;
}
// A refusal of memory is dear: torch's allocator waits for the GPU and gives back every block that it keeps before it raises, and what the program
// allocates next is new memory.  So a device that had no room for the scratch of a spread operand, which is optional, is asked again only where
// that would fit as new memory, with 64 MiB to spare for what the allocator rounds up to.
std::atomic<bool> refused[64];
bool room_for(size_t bytes, int device) {
    if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None) return false;
    auto* const allocator = c10::hip::HIPCachingAllocator::get();
    const auto [free, total] = allocator->getMemoryInfo((c10::DeviceIndex)device);
    size_t room = free;
    try {
        const double allowed = allocator->getMemoryFraction((c10::DeviceIndex)device) * (double)total;
        const auto kept = allocator->getDeviceStats((c10::DeviceIndex)device).reserved_bytes[0].current;
        const double left = allowed > (double)kept ? allowed - (double)kept : 0.0;
        if (left < (double)room) room = (size_t)left;
    } catch (const c10::Error&) {                           // an allocator without these figures
    }
    return room >= bytes + ((size_t)64 << 20);
}
// `fixed` bytes and those of the product, at least 16; *bytes: how many.  A GPU too full for a spread operand does without, whatever its
// allocator says so with (torch's own raises OutOfMemoryError; errors of the device itself are not about room).
at::Tensor scratch(size_t fixed, const Slabs& s, int device, size_t* bytes) {
    if (s.spread) {
        std::atomic<bool>& none_left = refused[device & 63];
        *bytes = fixed + s.spread;
        if (!none_left.load(std::memory_order_relaxed) || room_for(*bytes, device)) {
            try {
                at::Tensor ws = fresh({(int64_t)*bytes}, kByte, device);
                if (ws.data_ptr()) {
                    if (none_left.load(std::memory_order_relaxed)) none_left.store(false, std::memory_order_relaxed);
                    return ws;
                }
            } catch (const c10::AcceleratorError&) {
                throw;
            } catch (const std::exception&) {
            }
            none_left.store(true, std::memory_order_relaxed);
        }
    }
    *bytes = fixed + s.used;
    return *bytes ? fresh({(int64_t)(*bytes < 16 ? 16 : *bytes)}, kByte, device) : at::Tensor();
}

// linear(codes, scales, weight, weight_scales, bias or None) -> y
PyObject* linear(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(5)
    const at::Tensor *q = tensor(a[0]), *sx = tensor(a[1]);
    const int device = device_of(q);
    Weight w;
    if (!plain(q, kByte, device) || !plain(sx, kHalf, device) || q->dim() < 1 || q->numel() == 0) return none();
    const int64_t half_k = q->size(-1), M = q->numel() / half_k;
    if (sx->numel() != M || !weight_args(a[2], a[3], a[4], half_k, device, &w)) return none();
    c10::SmallVector<int64_t, 6> sizes(q->sizes().begin(), q->sizes().end());
    sizes.back() = w.N;
    const Slabs slabs = slab_bytes(M, w.N, half_k * 2, device);
    at::Tensor y, ws;
    const auto call = [&] {
        size_t need;
        y = fresh(sizes, kHalf, device);
        ws = scratch(0, slabs, device, &need);
        return qr_linear_i4_f16_ws(q->data_ptr(), sx->data_ptr(), w.w->data_ptr(), w.s->data_ptr(), ptr(w.b), M, w.N, half_k * 2,
                                   y.data_ptr(), need ? ws.data_ptr() : nullptr, need, stream(device));
    };
    if (!done(call)) return none();
    return wrap(std::move(y));
    QR_END
}

// quantized_linear(x, table or None, K, mode, scale, clip, weight, weight_scales, bias or None) -> y (K = 0: no Hadamard)
PyObject* quantized_linear(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(9)
    const Rows r = rows_of(a[0]);
    long long K, mode;
    double scale, clip;
    const at::Tensor* table;
    Weight w;
    if (!r.ok || r.n % 64 || r.n > 0x7fffffff || !arg_int(a[2], &K) || !arg_int(a[3], &mode) || !arg_float(a[4], &scale) ||
        !arg_float(a[5], &clip) || !table_arg(a[1], mode, K, r.device, &table) ||
        !weight_args(a[6], a[7], a[8], r.n / 2, r.device, &w))
        return none();
    c10::SmallVector<int64_t, 6> sizes(r.x->sizes().begin(), r.x->sizes().end());
    sizes.back() = w.N;
    const Slabs slabs = slab_bytes(r.rows, w.N, r.n, r.device);
    at::Tensor y, ws;
    const auto call = [&] {
        size_t need;
        y = fresh(sizes, kHalf, r.device);
        ws = scratch(slabs.fixed, slabs, r.device, &need);
        return qr_quantized_linear_f16(r.x->data_ptr(), r.rows, r.n, (int)K, ptr(table), (int)mode, (float)scale, (float)clip,
                                       w.w->data_ptr(), w.s->data_ptr(), ptr(w.b), w.N, y.data_ptr(), ws.data_ptr(), need,
                                       stream(r.device));
    };
    if (!done(call)) return none();
    return wrap(std::move(y));
    QR_END
}

// ---- the paged cache -------------------------------------------------------------------------------------------------
struct Cache {
    const at::Tensor *data, *param, *indptr, *indices, *last;
    int64_t pages, batch;
    int layers, heads, page_size;
};
bool cache_args(PyObject* const* a, int device, long long layer, Cache* c) {
    c->data = tensor(a[0]);
    c->param = tensor(a[1]);
    c->indptr = tensor(a[2]);
    c->indices = tensor(a[3]);
    c->last = tensor(a[4]);
    if (!plain(c->data, kByte, device) || !plain(c->param, kHalf, device) || !plain(c->indptr, at::kInt, device) ||
        !plain(c->indices, at::kInt, device) || !plain(c->last, at::kInt, device))
        return false;
    const auto d = c->data->sizes(), p = c->param->sizes();
    if (d.size() != 6 || p.size() != 6 || d[2] != 2 || d[5] != 64 || p[5] != 2) return false;
    for (int i = 0; i < 5; ++i)
        if (d[i] != p[i] || d[i] > 0x7fffffff) return false;
    c->pages = d[0];
    c->layers = (int)d[1];
    c->heads = (int)d[3];
    c->page_size = (int)d[4];
    c->batch = c->last->numel();
    return c->indptr->dim() == 1 && c->indices->dim() == 1 && c->last->dim() == 1 && c->batch > 0 &&
           c->indptr->numel() == c->batch + 1 && layer >= 0 && layer < c->layers;
}

// page_tables(batch, length, page_size, reference tensor on the device) -> (indptr, indices, last_page_offset)
PyObject* page_tables(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(4)
    long long batch, length, page;
    const int device = device_of(tensor(a[3]));
    if (device < 0 || !arg_int(a[0], &batch) || !arg_int(a[1], &length) || !arg_int(a[2], &page) || batch <= 0 || page <= 0 ||
        length <= 0 || page > 0x7fffffff)
        return none();
    at::Tensor indptr, indices, last;
    const auto call = [&] {
        indptr = fresh({batch + 1}, at::kInt, device);
        indices = fresh({batch * ((length + page - 1) / page)}, at::kInt, device);
        last = fresh({batch}, at::kInt, device);
        return qr_page_tables(batch, length, (int)page, indptr.data_ptr(), indices.data_ptr(), last.data_ptr(), stream(device));
    };
    if (!done(call)) return none();
    PyObject* t = PyTuple_New(3);
    if (!t) return nullptr;
    at::Tensor* const all[3] = {&indptr, &indices, &last};
    for (int i = 0; i < 3; ++i) {
        PyObject* o = wrap(std::move(*all[i]));
        if (!o) {
            Py_DECREF(t);
            return nullptr;
        }
        PyTuple_SET_ITEM(t, i, o);
    }
    return t;
    QR_END
}

// where(reference tensor) -> what its device's current stream is: the stream's handle, or (handle, number of the capture) while a
// graph is captured from it
PyObject* where(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(1)
    if (!THPVariable_Check(a[0])) return none();
    const at::Tensor& t = THPVariable_Unpack(a[0]);
    if (!t.is_cuda()) return none();
    void* const st = stream((int)t.device().index());
    hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
    unsigned long long id = 0;
    if (st && hipStreamGetCaptureInfo((hipStream_t)st, &status, &id) != hipSuccess) (void)hipGetLastError();     // (no capture starts on the default stream)
    if (status != hipStreamCaptureStatusActive) return PyLong_FromVoidPtr(st);
    return Py_BuildValue("(NK)", PyLong_FromVoidPtr(st), id);
    QR_END
}

// quantize_append(kv_data, kv_param, indptr, indices, last, k, v, seqlen_indptr or None, layer, hadamard) -> True
PyObject* quantize_append(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(10)
    const int device = device_of(tensor(a[0]));
    long long layer;
    bool had;
    Cache c;
    if (!arg_int(a[8], &layer) || !arg_bool(a[9], &had) || !cache_args(a, device, layer, &c)) return none();
    const at::Tensor *k = tensor(a[5]), *v = tensor(a[6]), *seq;
    if (!plain(k, kHalf, device) || !plain(v, kHalf, device) || !plain_or_none(a[7], at::kInt, device, &seq)) return none();
    if (k->dim() != 3 || k->sizes() != v->sizes() || k->size(1) != c.heads || k->size(2) != 128 || k->numel() == 0) return none();
    const int64_t tokens = k->size(0);
    if (seq ? (seq->dim() != 1 || seq->numel() != c.batch + 1) : tokens != c.batch) return none();
    const auto call = [&] {
        return qr_kv_quant_append_f16_i4(k->data_ptr(), v->data_ptr(), tokens, ptr(seq), had ? 1 : 0, c.data->data_ptr(), c.param->data_ptr(),
                                         c.indptr->data_ptr(), c.indices->data_ptr(), c.last->data_ptr(), c.pages, c.layers, (int)layer, c.heads,
                                         c.page_size, 128, c.batch, stream(device));
    };
    if (!done(call)) return none();
    Py_RETURN_TRUE;
    QR_END
}

// decode_step(kv_data, kv_param, indptr, indices, last, q, k, v, layer, q_hadamard, k_hadamard, max_seq_len, workspace or None)
// -> o.  The step's new token is quantised, stored and attended to in the same launch; a workspace has zeroed counters.
PyObject* decode_step(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(13)
    const int device = device_of(tensor(a[0]));
    long long layer, bound;
    bool q_had, k_had;
    Cache c;
    if (!arg_int(a[8], &layer) || !arg_bool(a[9], &q_had) || !arg_bool(a[10], &k_had) || !arg_int(a[11], &bound) ||
        !cache_args(a, device, layer, &c))
        return none();
    const at::Tensor *q = tensor(a[5]), *k = tensor(a[6]), *v = tensor(a[7]), *ws;
    if (!plain(q, kHalf, device) || !plain(k, kHalf, device) || !plain(v, kHalf, device) || !plain_or_none(a[12], kByte, device, &ws))
        return none();
    const int64_t vec = c.batch * c.heads * 128;
    if (q->numel() != vec || k->numel() != vec || v->numel() != vec || q->size(-1) != 128 || k->size(-1) != 128 || v->size(-1) != 128 ||
        q->dim() < 2 || q->size(-2) != c.heads || k->size(-2) != c.heads || v->size(-2) != c.heads)
        return none();
    const size_t need = bound > 0 ? qr_batch_decode_workspace_bytes(c.batch, c.heads, bound) : 0;
    const bool kept = need && ws && (size_t)ws->numel() >= need;
    const int qh = (q_had ? 1 : 0) | (kept ? QR_DECODE_COUNTERS_ZERO : 0), kh = k_had ? 1 : 0;
    at::Tensor o, own;
    const auto call = [&] {
        if (need && !kept) own = fresh({(int64_t)need}, kByte, device);
        o = fresh(q->sizes(), kHalf, device);
        return qr_kv_quant_append_batch_decode_f16_i4(o.data_ptr(), q->data_ptr(), qh, k->data_ptr(), v->data_ptr(), kh, c.data->data_ptr(),
                                                      c.param->data_ptr(), c.indptr->data_ptr(), c.indices->data_ptr(), c.last->data_ptr(),
                                                      c.pages, c.layers, (int)layer, c.heads, c.page_size, 128, c.batch, bound,
                                                      kept ? ws->data_ptr() : need ? own.data_ptr() : nullptr, need, stream(device));
    };
    if (!done(call)) return none();
    return wrap(std::move(o));
    QR_END
}

// outcome(code) -> whether the library's code means success: True, False for a refusal, RuntimeError for a HIP error
PyObject* outcome(PyObject*, PyObject* const* a, Py_ssize_t nargs) {
    QR_ARGS(1)
    long long rc;
    if (!arg_int(a[0], &rc)) return none();
    return PyBool_FromLong(success((int)rc));
    QR_END
}

#define QR_METHOD(NAME) {#NAME, (PyCFunction)(void (*)(void))NAME, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {QR_METHOD(quantize_rows),
                         QR_METHOD(rmsnorm),
                         QR_METHOD(rmsnorm_quantize),
                         QR_METHOD(heads_hadamard_quantize),
                         QR_METHOD(hadamard),
                         QR_METHOD(hadamard_quantize),
                         QR_METHOD(linear),
                         QR_METHOD(quantized_linear),
                         QR_METHOD(page_tables),
                         QR_METHOD(where),
                         QR_METHOD(quantize_append),
                         QR_METHOD(decode_step),
                         QR_METHOD(outcome),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
