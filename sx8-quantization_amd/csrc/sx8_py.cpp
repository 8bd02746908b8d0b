// sx8_py.cpp -- the per-call host path of the Python wrappers, as a CPython module.
//
// A linear layer's kernel on one token takes 4-9 us; argument conversion for a 14-argument
// ctypes call, the stream query and the output allocation in Python took 11-12 (6.0 now for
// 1024 x 2560 and one token, launch included, and 7.4 for 2560 x 9728, where the kernel bounds
// it; 512 embedding rows 13.0 -> 6.4, a whole 9728 x 2560 weight back to fp16 22.5 -> 16.9).
// Each function here does what the wrapper of the same name does for the calls a runtime makes
// all the time -- plain device tensors of the right type -- and returns None for every other
// call, which the wrapper then takes through its general path (conversions, copies, padding,
// error messages); without the module every call goes there.  The library's entry points are bound by address from the copy that ctypes
// loaded, so both paths run the same library, and as in a ctypes call the interpreter lock is
// given up while a launch or an allocation may wait.  Nothing is kept between calls.
#include <Python.h>

#include <ATen/ops/empty.h>
#include <c10/core/DeviceGuard.h>
#include <c10/core/GradMode.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include <algorithm>
#include <cstdint>
#include <cstdlib>
#include <cstring>

#include "sx8_hip.h"

namespace {

typedef const void* CP;
struct Lib {
    int32_t (*abi_version)();
    const char* (*last_error)();
    int32_t (*linear)(CP, int64_t, int64_t, int64_t, CP, CP, int32_t, CP, CP, CP, int64_t, int64_t, void*, void*);
    int32_t (*gemv)(CP, CP, CP, int32_t, CP, CP, CP, void*, int64_t, int64_t, void*, void*, int64_t, void*);
    int64_t (*gemm_ws)(int64_t, int32_t, const int64_t*, int64_t);
    int32_t (*gemm)(CP, int64_t, int64_t, int64_t, CP, CP, int32_t, CP, CP, int64_t, int64_t, void*, void*, int64_t,
                    void*);
    int32_t (*gemm_split)(CP, int64_t, int64_t, int64_t, CP, CP, CP, CP, CP, CP, CP, CP, int64_t, int64_t, void*, void*,
                          int64_t, void*);
    int32_t (*dequant)(CP, CP, CP, CP, CP, CP, CP, CP, int64_t, int64_t, int64_t, void*, void*);
    int32_t (*embed)(CP, int64_t, CP, CP, int32_t, CP, CP, int64_t, int64_t, int64_t, void*, void*);
} lib;

constexpr int32_t kUnsupported = SX8_ERR_UNSUPPORTED;
constexpr int64_t kLinearRows = 32, kLdsMaxKb = 640;

// A plain tensor (or Parameter) whose memory holds its values, else null: subclasses, the wrappers of
// function transforms (vmap, jvp) and views that negate on reading go through the general path.
const at::Tensor* plain(PyObject* o) {
    if (!THPVariable_CheckExact(o)) return nullptr;
    using K = c10::DispatchKey;
    const at::Tensor& x = THPVariable_Unpack(o);
    static const c10::DispatchKeySet other({K::FuncTorchBatched, K::FuncTorchGradWrapper, K::Batched, K::Functionalize, K::Python,
                                     K::Conjugate, K::Negative, K::ZeroTensor});
    return x.key_set().has_any(other) ? nullptr : &x;
}

const at::Tensor* dev(PyObject* o, at::ScalarType t) {
    const at::Tensor* x = plain(o);
    return x && x->is_cuda() && x->layout() == at::kStrided && x->scalar_type() == t ? x : nullptr;
}

const at::Tensor* dense(PyObject* o, at::ScalarType t) {
    const at::Tensor* x = dev(o, t);
    return x && x->is_contiguous() ? x : nullptr;
}

typedef pybind11::gil_scoped_release Unlocked;

int64_t num(PyObject* o) { return PyLong_AsLongLong(o); }

// A size that is no integer (a float, say) is the general path's to convert or refuse.
#define SX8_SIZES_OK()      \
    if (PyErr_Occurred()) { \
        PyErr_Clear();      \
        Py_RETURN_NONE;     \
    }

void* stream_of(const at::Tensor& x) { return c10::hip::getCurrentHIPStream(x.device().index()).stream(); }

PyObject* failed(const char* name, int32_t rc) {
    PyErr_Format(PyExc_RuntimeError, "%s failed (code %d): %s", name, (int)rc, lib.last_error());
    return nullptr;
}

at::Tensor empty_like_device(at::IntArrayRef sizes, at::ScalarType t, const at::Tensor& x) {
    return at::empty(sizes, at::TensorOptions().dtype(t).device(x.device()));
}

#define SX8_ARGS(n)                                                                \
    if (na != (n)) {                                                               \
        PyErr_Format(PyExc_TypeError, "expected %d arguments, got %d", n, (int)na); \
        return nullptr;                                                            \
    }

// bind({name: address}): RuntimeError for a library of another ABI version.
PyObject* py_bind(PyObject*, PyObject* d) {
    auto get = [&](const char* name) -> void* {
        PyObject* v = PyDict_GetItemString(d, name);
        if (!v) PyErr_Format(PyExc_KeyError, "%s", name);
        return v ? PyLong_AsVoidPtr(v) : nullptr;
    };
#define SX8_BIND(field, name) \
    if (!(lib.field = reinterpret_cast<decltype(lib.field)>(get(name)))) return nullptr;
    SX8_BIND(abi_version, "sx8_abi_version")
    if (lib.abi_version() != SX8_ABI_VERSION) {
        PyErr_Format(PyExc_RuntimeError, "built for ABI version %d, the library has %d", SX8_ABI_VERSION,
                     (int)lib.abi_version());
        return nullptr;
    }
    SX8_BIND(last_error, "sx8_last_error")
    SX8_BIND(linear, "sx8_linear_f16")
    SX8_BIND(gemv, "sx8_gemv")
    SX8_BIND(gemm_ws, "sx8_gemm_prefill_workspace_bytes")
    SX8_BIND(gemm, "sx8_gemm_prefill")
    SX8_BIND(gemm_split, "sx8_gemm_prefill_split")
    SX8_BIND(dequant, "sx8_dequant_f16")
    SX8_BIND(embed, "sx8_embed_gather")
#undef SX8_BIND
    Py_RETURN_NONE;
}

// linear(x, (hdr, levels, bases, scales), hdr_bytes, bias, out_f, N, in_f, n_cb): fp16(x W^T) (+ bias) of
// up to 32 rows, shape (*x.shape[:-1], out_f).
PyObject* py_linear(PyObject*, PyObject* const* a, Py_ssize_t na) {
    HANDLE_TH_ERRORS
    SX8_ARGS(8)
    const at::Tensor* x = dev(a[0], at::kHalf);
    if (!x || x->dim() < 1 || !PyTuple_Check(a[1]) || PyTuple_GET_SIZE(a[1]) != 4) Py_RETURN_NONE;
    const int64_t out_f = num(a[4]), N = num(a[5]), K = num(a[6]), n_cb = num(a[7]), hb = num(a[2]);
    SX8_SIZES_OK()
    const int64_t M = K > 0 && x->size(-1) == K ? x->numel() / K : 0;
    // (K blocks that are not the row's: decode1_v44 cuts or pads the row, the GEMM refuses)
    if (M < 1 || M > kLinearRows || out_f != N || n_cb != (K + 31) / 32) Py_RETURN_NONE;
    if (M > 1) {
        const char* wmma = std::getenv("SX8_USE_WMMA");
        if (N < 64 || (wmma && std::strcmp(wmma, "1") == 0)) Py_RETURN_NONE;
    }
    const at::Tensor* t[4];
    for (int i = 0; i < 4; ++i)
        if (!(t[i] = plain(PyTuple_GET_ITEM(a[1], i))) || t[i]->device() != x->device()) Py_RETURN_NONE;
    const at::Tensor* b = nullptr;
    if (a[3] != Py_None) {
        b = dense(a[3], at::kHalf);
        // (a bias that either mode of autograd follows is added by torch)
        if (!b || b->device() != x->device() || b->dim() != 1 || b->size(0) != N ||
            (b->requires_grad() && c10::GradMode::is_enabled()) || b->_fw_grad(0).defined())
            Py_RETURN_NONE;
    }
    c10::SmallVector<int64_t, 5> shape(x->sizes().begin(), x->sizes().end());
    shape.back() = N;
    at::Tensor y;
    int32_t rc;
    {
        Unlocked u;
        const at::Tensor xc = x->is_contiguous() ? *x : x->contiguous();
        y = empty_like_device(shape, at::kHalf, *x);
        rc = lib.linear(xc.data_ptr(), M, K, K, t[0]->data_ptr(), t[1]->data_ptr(), (int32_t)hb, t[2]->data_ptr(),
                        t[3]->data_ptr(), b ? b->data_ptr() : nullptr, N, n_cb, y.data_ptr(), stream_of(*x));
    }
    if (rc == kUnsupported) Py_RETURN_NONE;
    if (rc) return failed("sx8_linear_f16", rc);
    return THPVariable_Wrap(std::move(y));
    END_HANDLE_TH_ERRORS
}

// gemv(x, hdr, levels, bases, scales, hdr_bytes, N, n_cb, Y): True, or None.
PyObject* py_gemv(PyObject*, PyObject* const* a, Py_ssize_t na) {
    HANDLE_TH_ERRORS
    SX8_ARGS(9)
    const at::Tensor* x = dense(a[0], at::kHalf);
    const at::Tensor* y = dense(a[8], at::kFloat);
    const int64_t N = num(a[6]), n_cb = num(a[7]), hb = num(a[5]);
    SX8_SIZES_OK()
    if (!x || !y || n_cb > kLdsMaxKb || x->numel() != n_cb * 32 || y->numel() != N || x->device() != y->device())
        Py_RETURN_NONE;
    if (reinterpret_cast<uintptr_t>(x->data_ptr()) & 15) Py_RETURN_NONE;
    const at::Tensor* t[4];
    for (int i = 0; i < 4; ++i)
        if (!(t[i] = plain(a[1 + i]))) Py_RETURN_NONE;
    int32_t rc;
    {
        Unlocked u;
        rc = lib.gemv(x->data_ptr(), t[0]->data_ptr(), t[1]->data_ptr(), (int32_t)hb, t[2]->data_ptr(), t[3]->data_ptr(), nullptr,
                      nullptr, N, n_cb, y->data_ptr(), nullptr, 0, stream_of(*x));
    }
    if (rc) return failed("sx8_gemv", rc);
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// X (M, K) fp16 dense with the output and workspace of its product.
struct GemmCall {
    const at::Tensor* x;
    int64_t M, K, N, n_cb, ws_bytes;
    at::Tensor ws, y;
    bool make(PyObject* X, int64_t N_, int64_t n_cb_) {          // false: the general path
        x = dense(X, at::kHalf);
        if (!x || x->dim() != 2 || x->size(0) < 1) return false;
        M = x->size(0);
        K = x->size(1);
        N = N_;
        n_cb = n_cb_;
        ws_bytes = lib.gemm_ws(M, 1, &N, n_cb);
        return ws_bytes >= 0;
    }
    void allocate() {
        y = empty_like_device({M, N}, at::kFloat, *x);
        ws = empty_like_device({std::max<int64_t>(ws_bytes, 256)}, at::kByte, *x);
    }
};

// gemm(X, hdr, levels, bases, scales, hdr_bytes, N, in_f, n_cb): Y (M, N) float32, or None.
PyObject* py_gemm(PyObject*, PyObject* const* a, Py_ssize_t na) {
    HANDLE_TH_ERRORS
    SX8_ARGS(9)
    const at::Tensor* t[4];
    for (int i = 0; i < 4; ++i)
        if (!(t[i] = plain(a[1 + i]))) Py_RETURN_NONE;
    GemmCall c;
    const int64_t N = num(a[6]), in_f = num(a[7]), n_cb = num(a[8]), hb = num(a[5]);
    SX8_SIZES_OK()
    if (!c.make(a[0], N, n_cb) || c.K < in_f) Py_RETURN_NONE;
    int32_t rc;
    {
        Unlocked u;
        c.allocate();
        rc = lib.gemm(c.x->data_ptr(), c.M, c.K, in_f, t[0]->data_ptr(), t[1]->data_ptr(), (int32_t)hb, t[2]->data_ptr(),
                      t[3]->data_ptr(), c.N, c.n_cb, c.y.data_ptr(), c.ws.data_ptr(), c.ws_bytes, stream_of(*c.x));
    }
    if (rc) return failed("sx8_gemm_prefill", rc);
    return THPVariable_Wrap(std::move(c.y));
    END_HANDLE_TH_ERRORS
}

// gemm_split(X, dmin, dmax, config, coeff, hi, lo, basis, scales, n_cb): Y (M, N) float32, or None.
PyObject* py_gemm_split(PyObject*, PyObject* const* a, Py_ssize_t na) {
    HANDLE_TH_ERRORS
    SX8_ARGS(10)
    const at::Tensor* t[8];
    for (int i = 0; i < 8; ++i)
        if (!(t[i] = plain(a[1 + i]))) Py_RETURN_NONE;
    const int64_t n_cb = num(a[9]);
    SX8_SIZES_OK()
    GemmCall c;
    if (n_cb < 1 || !c.make(a[0], t[0]->numel() / n_cb, n_cb)) Py_RETURN_NONE;
    int32_t rc;
    {
        Unlocked u;
        c.allocate();
        rc = lib.gemm_split(c.x->data_ptr(), c.M, c.K, std::min(c.K, n_cb * 32), t[0]->data_ptr(), t[1]->data_ptr(),
                            t[2]->data_ptr(), t[3]->data_ptr(), t[4]->data_ptr(), t[5]->data_ptr(), t[6]->data_ptr(),
                            t[7]->data_ptr(), c.N, n_cb, c.y.data_ptr(), c.ws.data_ptr(), c.ws_bytes, stream_of(*c.x));
    }
    if (rc) return failed("sx8_gemm_prefill_split", rc);
    return THPVariable_Wrap(std::move(c.y));
    END_HANDLE_TH_ERRORS
}

// dequant(dmin, dmax, config, coeff, hi, lo, basis, scales, out_f, in_f, n_cb): W (out_f, in_f) fp16 on the
// current device, or None unless every field is already there in its stored type.
PyObject* py_dequant(PyObject*, PyObject* const* a, Py_ssize_t na) {
    HANDLE_TH_ERRORS
    SX8_ARGS(11)
    const at::Tensor* t[8];
    for (int i = 0; i < 8; ++i) {
        const at::ScalarType want = i < 2 ? at::kHalf : i < 6 ? at::kByte : at::kFloat;
        t[i] = dense(a[i], want);
        if (!t[i] && i < 2) t[i] = dense(a[i], at::kShort);
        if (!t[i] || t[i]->device() != t[0]->device()) Py_RETURN_NONE;
    }
    if (t[0]->device().index() != c10::hip::current_device()) Py_RETURN_NONE;
    const int64_t out_f = num(a[8]), in_f = num(a[9]), n_cb = num(a[10]);
    SX8_SIZES_OK()
    if (t[6]->numel() != n_cb * 64 || t[7]->numel() != n_cb * 2) Py_RETURN_NONE;
    at::Tensor w;
    int32_t rc;
    {
        Unlocked u;
        w = empty_like_device({out_f, in_f}, at::kHalf, *t[0]);
        rc = lib.dequant(t[0]->data_ptr(), t[1]->data_ptr(), t[2]->data_ptr(), t[3]->data_ptr(), t[4]->data_ptr(),
                         t[5]->data_ptr(), t[6]->data_ptr(), t[7]->data_ptr(), out_f, in_f, n_cb, w.data_ptr(),
                         stream_of(w));
    }
    if (rc) return failed("sx8_dequant_f16", rc);
    return THPVariable_Wrap(std::move(w));
    END_HANDLE_TH_ERRORS
}

// embed(ids, hdr, levels, basis, scales, K, N, n_cb, out): rows of ids into out's first rows, returned as
// a view (*ids.shape, K); or None.
PyObject* py_embed(PyObject*, PyObject* const* a, Py_ssize_t na) {
    HANDLE_TH_ERRORS
    SX8_ARGS(9)
    const at::Tensor* ids = dense(a[0], at::kLong);
    const at::Tensor* out = dense(a[8], at::kHalf);
    const at::Tensor* h = plain(a[1]);
    const at::Tensor* l = plain(a[2]);
    const at::Tensor* b = dense(a[3], at::kFloat);
    const at::Tensor* s = dense(a[4], at::kFloat);
    const int64_t K = num(a[5]), N = num(a[6]), n_cb = num(a[7]);
    SX8_SIZES_OK()
    if (!ids || !out || !h || !l || !b || !s || out->dim() != 2 || out->size(1) != K || ids->device() != out->device() ||
        ids->numel() < 1 || out->size(0) < ids->numel())
        Py_RETURN_NONE;
    const int64_t T = ids->numel();
    c10::SmallVector<int64_t, 5> shape(ids->sizes().begin(), ids->sizes().end());
    shape.push_back(K);
    at::Tensor rows;
    int32_t rc;
    {
        Unlocked u;
        rc = lib.embed(ids->data_ptr(), T, h->data_ptr(), l->data_ptr(), h->dim() == 2 ? (int32_t)h->size(1) : 6,
                       b->data_ptr(), s->data_ptr(), K, N, n_cb, out->data_ptr(), stream_of(*out));
        if (!rc) rows = out->narrow(0, 0, T).view(shape);
    }
    if (rc) return failed("sx8_embed_gather", rc);
    return THPVariable_Wrap(std::move(rows));
    END_HANDLE_TH_ERRORS
}

struct Event {
    hipEvent_t e = nullptr;
    ~Event() {
        if (e) (void)hipEventDestroy(e);
    }
};

void hip_ok(hipError_t e) { TORCH_CHECK(e == hipSuccess, "copy to the host: ", hipGetErrorString(e)); }

// to_host(x): a host copy of a dense device tensor of bytes; to_host(x, ((offset, bytes), ...)): host
// copies of those parts, each in memory of its own (a part kept alive keeps no other).  Through two
// pinned pieces of 1 MB (torch's caching host allocator): the GPU fills one while the host empties the
// other.  10 MB take 0.39 ms, 3 MB 0.14; the runtime's own copy to pageable memory 0.55 and 0.17 (up to
// 0.9).  Pieces of 2 and 4 MB measured no faster: the link takes 20 us a MB, one host thread about 39 to
// empty a piece.
PyObject* py_to_host(PyObject*, PyObject* const* a, Py_ssize_t na) {
    HANDLE_TH_ERRORS
    constexpr int64_t kPiece = 1 << 20;
    if (na != 2) SX8_ARGS(1)
    const at::Tensor* x = dense(a[0], at::kByte);
    if (!x || x->numel() < 1 || (na == 1 && x->numel() <= kPiece)) Py_RETURN_NONE;
    const int64_t n = x->numel(), pieces = (n + kPiece - 1) / kPiece;
    struct Part {
        int64_t off, n;
        at::Tensor y;
    };
    c10::SmallVector<Part, 8> parts;
    if (na == 1) {
        parts.push_back(Part{0, n, at::Tensor()});
    } else {
        if (!PyTuple_Check(a[1])) Py_RETURN_NONE;
        for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(a[1]); ++i) {
            PyObject* p = PyTuple_GET_ITEM(a[1], i);
            if (!PyTuple_Check(p) || PyTuple_GET_SIZE(p) != 2) Py_RETURN_NONE;
            const int64_t off = num(PyTuple_GET_ITEM(p, 0)), len = num(PyTuple_GET_ITEM(p, 1));
            SX8_SIZES_OK()
            if (off < 0 || len < 0 || off > n || len > n - off) {
                PyErr_SetString(PyExc_ValueError, "to_host: a part outside the tensor");
                return nullptr;
            }
            parts.push_back(Part{off, len, at::Tensor()});
        }
    }
    {
        Unlocked u;
        c10::DeviceGuard on(x->device());
        for (Part& p : parts) p.y = at::empty({p.n}, at::TensorOptions().dtype(at::kByte));
        const at::Tensor pin = at::empty({std::min(n, 2 * kPiece)}, at::TensorOptions().dtype(at::kByte).pinned_memory(true));
        const hipStream_t st = c10::hip::getCurrentHIPStream(x->device().index()).stream();
        Event ev[2];                      // (one piece: a copy that waits, 10-15 us less than event or stream waits)
        if (pieces > 1)
            for (Event& v : ev) hip_ok(hipEventCreateWithFlags(&v.e, hipEventDisableTiming));
        uint8_t* const stage = static_cast<uint8_t*>(pin.data_ptr());
        auto send = [&](int64_t k) {
            const int64_t off = k * kPiece;
            const auto copy = pieces > 1 ? hipMemcpyAsync : hipMemcpyWithStream;
            hip_ok(copy(stage + (k & 1) * kPiece, static_cast<const uint8_t*>(x->data_ptr()) + off,
                        std::min(kPiece, n - off), hipMemcpyDeviceToHost, st));
            if (pieces > 1) hip_ok(hipEventRecord(ev[k & 1].e, st));
        };
        send(0);
        for (int64_t k = 0; k < pieces; ++k) {
            if (k + 1 < pieces) send(k + 1);
            if (pieces > 1) hip_ok(hipEventSynchronize(ev[k & 1].e));
            const int64_t lo = k * kPiece, hi = std::min(lo + kPiece, n);
            const uint8_t* src = stage + (k & 1) * kPiece;
            for (Part& p : parts) {
                const int64_t from = std::max(lo, p.off), to = std::min(hi, p.off + p.n);
                if (from < to) std::memcpy(static_cast<uint8_t*>(p.y.data_ptr()) + (from - p.off), src + (from - lo), to - from);
            }
        }
    }
    if (na == 1) return THPVariable_Wrap(std::move(parts[0].y));
    PyObject* list = PyList_New((Py_ssize_t)parts.size());
    for (size_t i = 0; list && i < parts.size(); ++i) PyList_SET_ITEM(list, (Py_ssize_t)i, THPVariable_Wrap(std::move(parts[i].y)));
    return list;
    END_HANDLE_TH_ERRORS
}

#define SX8_FAST(f) reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(f)), METH_FASTCALL
PyMethodDef methods[] = {{"bind", py_bind, METH_O, nullptr},
                         {"linear", SX8_FAST(py_linear), nullptr},
                         {"gemv", SX8_FAST(py_gemv), nullptr},
                         {"gemm", SX8_FAST(py_gemm), nullptr},
                         {"gemm_split", SX8_FAST(py_gemm_split), nullptr},
                         {"dequant", SX8_FAST(py_dequant), nullptr},
                         {"embed", SX8_FAST(py_embed), nullptr},
                         {"to_host", SX8_FAST(py_to_host), nullptr},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_sx8py", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__sx8py() {
    PyObject* m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "torch_version", SX8_TORCH) < 0) {
        Py_DECREF(m);
        return nullptr;
    }
    return m;
}
