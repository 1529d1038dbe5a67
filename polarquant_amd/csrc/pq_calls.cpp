// The C ABI's functions as CPython builtins, and the questions a wrapper asks its tensors before it calls one.
//
// What bounds a small call is its host side: at 4096 tokens and 32 KV heads the score kernel takes 5.2 us, its call took 9.7
// through ctypes (30 arguments converted one by one 4 us, the tensors' pointers, shapes, strides and types 4 us, the launch 2).
// Here an argument is converted by the parameter's C type, a tensor is its own pointer, and a wrapper's checks are one call.
// Nothing is refused here: a tensor that is not as the fast question wants it is left to the wrapper's general path.
#include <torch/csrc/autograd/forward_grad.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/version.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/autocast_mode.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>

#include <cstring>
#include <type_traits>
#include <utility>

#include "../../include/polarquant.h"
#include "../../include/polarquant_latent.h"
#include "../../include/polarquant_recurrent.h"
#include "../../include/polarquant_steps.h"

namespace {

PyObject* argument_error = nullptr;                 // ctypes.ArgumentError, what a wrong argument raised before
PyObject* parameter_class = nullptr;                // torch.nn.Parameter
PyObject* out_of_memory_error = nullptr;            // torch.OutOfMemoryError

bool plain_tensor(PyObject* o) {
    return THPVariable_CheckExact(o) || reinterpret_cast<PyObject*>(Py_TYPE(o)) == parameter_class;
}

// ----------------------------------------------------------------------------- arguments
constexpr int kListed = 16;                         // integers of an array argument (strides), at most

struct Arg {
    int64_t list[kListed];
};

bool refuse(PyObject* o, const char* wanted) {
    if (PyErr_Occurred()) return false;             // (as an object's own method raised it)
    PyErr_Format(argument_error, "expected %s instead of %s", wanted, Py_TYPE(o)->tp_name);
    return false;
}

// (wraps around beyond the type, as ctypes does: the library then refuses the size)
bool integer(PyObject* o, uint64_t& v) {
    if (PyLong_Check(o)) {
        v = PyLong_AsUnsignedLongLongMask(o);
        return true;
    }
    PyObject* i = PyIndex_Check(o) ? PyNumber_Index(o) : nullptr;
    if (!i) return refuse(o, "an integer");
    v = PyLong_AsUnsignedLongLongMask(i);
    Py_DECREF(i);
    return true;
}

// What a parameter takes besides None and a tensor: an untyped or byte pointer an address (handles, rows of a tensor); integers and floats (a
// caller's own counts, positions, states) nothing, as a number or a tuple in their place is a mistake that the GPU would have to find; and
// strides, of the functions that have them, a tuple.
enum class Also { kNothing, kAddress, kStrides };

bool pointer(PyObject* o, Arg& a, Also also, void*& p) {
    if (o == Py_None) {
        p = nullptr;
    } else if (plain_tensor(o)) {
        p = THPVariable_Unpack(o).data_ptr();
    } else if (also == Also::kAddress && PyLong_CheckExact(o)) {
        p = reinterpret_cast<void*>(PyLong_AsUnsignedLongLongMask(o));
    } else if (also == Also::kStrides && PyTuple_Check(o)) {      // for the length of the call
        const Py_ssize_t n = PyTuple_GET_SIZE(o);
        if (n > kListed) return refuse(o, "fewer integers");
        for (Py_ssize_t i = 0; i < n; i++) {
            uint64_t v;
            if (!integer(PyTuple_GET_ITEM(o, i), v)) return false;
            a.list[i] = static_cast<int64_t>(v);
        }
        p = a.list;
    } else if (THPVariable_Check(o)) {              // (asks the class; the forms above are the common ones) a subclass says for itself what its pointer is
        PyObject* at = PyObject_CallMethod(o, "data_ptr", nullptr);
        uint64_t v = 0;
        const bool ok = at && integer(at, v);
        Py_XDECREF(at);
        if (!ok) return refuse(o, "a pointer");
        p = reinterpret_cast<void*>(v);
    } else if (also == Also::kAddress) {
        uint64_t v;
        if (!integer(o, v)) return false;
        p = reinterpret_cast<void*>(v);
    } else {
        return refuse(o, "a tensor");
    }
    return true;
}

template <typename T, bool STRIDES>
bool convert(PyObject* o, Arg& a, T& out) {
    if constexpr (std::is_pointer_v<T>) {
        using P = std::remove_cv_t<std::remove_pointer_t<T>>;
        constexpr Also also = std::is_void_v<P> || std::is_same_v<P, uint8_t> ? Also::kAddress
                              : STRIDES && std::is_same_v<P, int64_t>          ? Also::kStrides
                                                                              : Also::kNothing;
        void* p;
        if (!pointer(o, a, also, p)) return false;
        out = static_cast<T>(p);
        return true;
    } else if constexpr (std::is_floating_point_v<T>) {
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) {
            PyErr_Clear();
            return refuse(o, "a number");
        }
        out = static_cast<T>(v);
        return true;
    } else {
        uint64_t v;
        if (!integer(o, v)) return false;
        out = static_cast<T>(v);
        return true;
    }
}

// The interpreter is other threads' for as long as this lives, also where what runs meanwhile throws.
struct Released {
    PyThreadState* thread = PyEval_SaveThread();
    ~Released() { PyEval_RestoreThread(thread); }
};

template <typename F, bool STRIDES> struct Call;
template <bool STRIDES, typename R, typename... A>
struct Call<R(A...), STRIDES> {
    static_assert(std::is_integral_v<R>, "a status, a count or a size");
    template <size_t... I>
    static PyObject* run(void* at, PyObject* const* args, std::index_sequence<I...>) {
        std::tuple<std::decay_t<A>...> v;
        Arg kept[sizeof...(A) + 1];
        if (!(convert<std::decay_t<A>, STRIDES>(args[I], kept[I], std::get<I>(v)) && ...)) return nullptr;
        const R r = [&] {
            Released others;
            return reinterpret_cast<R (*)(A...)>(at)(std::get<I>(v)...);
        }();
        return std::is_signed_v<R> ? PyLong_FromLongLong(static_cast<long long>(r)) : PyLong_FromUnsignedLongLong(static_cast<unsigned long long>(r));
    }
    static PyObject* entry(PyObject* self, PyObject* const* args, Py_ssize_t n) {
        if (n != static_cast<Py_ssize_t>(sizeof...(A))) {
            PyErr_Format(PyExc_TypeError, "this function takes %d arguments (%zd given)", static_cast<int>(sizeof...(A)), n);
            return nullptr;
        }
        try {
            return run(PyCapsule_GetPointer(self, nullptr), args, std::index_sequence_for<A...>{});
        } catch (const std::exception& e) {         // (a tensor without storage)
            PyErr_SetString(PyExc_RuntimeError, e.what());
            return nullptr;
        }
    }
};

// The functions that the wrappers call: X without a parameter for strides, S with one.
#define PQ_CALLS(X, S)                                                                                                                     \
    X(pq_decode_scores) S(pq_quantize_groups) S(pq_quantize_values) X(pq_decode_attn) X(pq_decode_attn_v4) X(pq_decode_attn_plan)          \
    X(pq_decode_attn_v4_plan) X(pq_decode_attn_workspace_bytes) X(pq_rope_append) X(pq_rope_qk) X(pq_rmsnorm) X(pq_embed_rmsnorm)          \
    X(pq_rmsnorm_advance) X(pq_silu_mul) X(pq_linear_small_m) X(pq_qkv_rope_append) S(pq_prompt_attn) X(pq_norm_conv) X(pq_relu_sq)         \
    X(pq_gelu_mul) X(pq_stream_add) X(pq_embed_rows) X(pq_embed_norm_conv_takes) X(pq_embed_norm_conv) X(pq_logits) X(pq_softcap)           \
    X(pq_head_linear) X(pq_latent_norm) X(pq_latent_decode_plan) X(pq_latent_decode_workspace_bytes) X(pq_latent_decode)                   \
    X(pq_latent_prefill_takes) X(pq_latent_prefill) X(pq_qk_norm) X(pq_ring_append) X(pq_window_plan) X(pq_window_workspace_bytes)         \
    X(pq_window_attn) X(pq_delta_prep) X(pq_scan_workspace_bytes) X(pq_delta_scan) X(pq_memory_gates) X(pq_memory_scan)                    \
    X(pq_head_norm_gate) X(pq_validate_delta_token) X(pq_delta_token) X(pq_validate_memory_token) X(pq_memory_token)        \
    X(pq_validate_linear_gelu) X(pq_linear_gelu) X(pq_linear_residual) X(pq_gated_normed) X(pq_qkv_rope_append_normed)

// A prototype as ctypes writes types: the result's letter, then the parameters'.
template <typename T>
constexpr char letter() {
    if constexpr (std::is_pointer_v<T>) return 'P';
    else if constexpr (std::is_same_v<T, float>) return 'f';
    else if constexpr (sizeof(T) == 4) return std::is_signed_v<T> ? 'i' : 'I';
    else return std::is_signed_v<T> ? 'l' : 'L';
}
template <typename F> struct Prototype;
template <typename R, typename... A>
struct Prototype<R(A...)> {
    static constexpr char text[] = {letter<R>(), letter<std::decay_t<A>>()..., 0};
};

struct Bound {
    PyMethodDef method;
    const char* prototype;
};
#define PQ_BOUND(f, strides)                                                                                                               \
    {{#f, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Call<decltype(f), strides>::entry)), METH_FASTCALL, nullptr},        \
     Prototype<decltype(f)>::text},
#define PQ_METHOD(f) PQ_BOUND(f, false)
#define PQ_STRIDES(f) PQ_BOUND(f, true)
Bound bound[] = {PQ_CALLS(PQ_METHOD, PQ_STRIDES)};

// bind(name, address, prototype) -> the function at `address` of a loaded library as a builtin, None for a name that is not called from here.
// The prototype is the caller's: another one than this file was compiled with raises, as the arguments would not be the library's.
PyObject* bind(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 3 || !PyUnicode_Check(args[0]) || !PyUnicode_Check(args[2])) {
        PyErr_SetString(PyExc_TypeError, "bind(name, address, prototype)");
        return nullptr;
    }
    const char *name = PyUnicode_AsUTF8(args[0]), *prototype = PyUnicode_AsUTF8(args[2]);
    uint64_t at;
    if (!name || !prototype || !integer(args[1], at)) return nullptr;
    for (Bound& f : bound) {
        if (std::strcmp(f.method.ml_name, name) != 0) continue;
        if (std::strcmp(f.prototype, prototype) != 0) {
            PyErr_Format(PyExc_RuntimeError, "polarquant_amd: _calls.so is of another version (%s is %s there, %s here); build it with "
                         "`python -m polarquant_amd.build --calls`", name, f.prototype, prototype);
            return nullptr;
        }
        PyObject* self = PyCapsule_New(reinterpret_cast<void*>(at), nullptr, nullptr);
        if (!self) return nullptr;
        PyObject* r = PyCFunction_New(&f.method, self);
        Py_DECREF(self);
        return r;
    }
    Py_RETURN_NONE;
}

// ----------------------------------------------------------------------------- questions
// Plain eager execution, as far as can be told here: gradients off in both directions, no transform, trace, autocast or mode.
bool plain_execution() {
    return !c10::GradMode::is_enabled() && at::impl::PythonTorchFunctionTLS::stack_len() == 0 && c10::impl::TorchDispatchModeTLS::stack_len() == 0 &&
           !c10::impl::tls_is_dispatch_key_included(c10::DispatchKey::FuncTorchDynamicLayerFrontMode) && !torch::jit::tracer::isTracing() &&
           !at::autocast::is_autocast_enabled(at::kCUDA) && torch::autograd::ForwardADLevel::try_get_by_idx(0) == nullptr;
}

PyObject* yes_or_ask(bool yes) {
    PyObject* r = yes ? Py_True : Py_None;
    Py_INCREF(r);
    return r;
}

// plain_eager(*tensors) -> True, or None: the caller has to look closer
PyObject* plain_eager(PyObject*, PyObject* const* args, Py_ssize_t n) {
    for (Py_ssize_t i = 0; i < n; i++)
        if (!plain_tensor(args[i])) Py_RETURN_NONE;
    return yes_or_ask(plain_execution());
}

int half_code(const at::Tensor& t) {                // the library's code of a half-precision type, or -1
    return t.scalar_type() == at::kHalf ? PQ_F16 : t.scalar_type() == at::kBFloat16 ? PQ_BF16 : -1;
}

// plain_half(*tensors) -> True (plain eager execution, one half-precision type, one GPU, contiguous, 16-byte aligned, not empty), False (plain,
// but they do not lie like that) or None
PyObject* plain_half(PyObject*, PyObject* const* args, Py_ssize_t n) {
    for (Py_ssize_t i = 0; i < n; i++)
        if (!plain_tensor(args[i])) Py_RETURN_NONE;
    if (n == 0 || !plain_execution()) Py_RETURN_NONE;
    const at::Tensor& first = THPVariable_Unpack(args[0]);
    bool lie = half_code(first) >= 0;
    for (Py_ssize_t i = 0; lie && i < n; i++) {
        const at::Tensor& t = THPVariable_Unpack(args[i]);
        if (!t.has_storage()) Py_RETURN_NONE;
        lie = t.is_cuda() && t.scalar_type() == first.scalar_type() && t.device() == first.device() && t.is_contiguous() && t.numel() > 0 &&
              reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0;
    }
    return PyBool_FromLong(lie);
}

// One tensor of a cache as the kernels read it: plain, on the query's GPU, contiguous.  t: None is allowed where `optional`.
struct Plain {
    c10::Device device = c10::Device(at::kCPU);
    bool ok = true;
    const at::Tensor* take(PyObject* o, int dim) {
        if (!ok || !plain_tensor(o)) {
            ok = false;
            return nullptr;
        }
        const at::Tensor& t = THPVariable_Unpack(o);
        ok = t.layout() == at::kStrided && t.has_storage() && t.is_cuda() && t.dim() == dim && t.is_contiguous();
        if (ok && device.is_cpu()) device = t.device();
        ok = ok && t.device() == device;
        return ok ? &t : nullptr;
    }
    void type(const at::Tensor* t, at::ScalarType s) { ok = ok && t->scalar_type() == s; }
};

// plain_scores(query, codes, rscale, rmn, tscale, tmn) -> (B, N, Nk, groups, packed, type) where the query's and the cache's shapes and types
// are the ones scores are made of and nothing has to be copied; else None
PyObject* plain_scores(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 6) Py_RETURN_NONE;
    Plain p;
    const at::Tensor* q = p.take(args[0], 4);
    const at::Tensor* codes = p.take(args[1], 5);
    if (!p.ok) Py_RETURN_NONE;
    const int dt = half_code(*q);
    const int64_t row = codes->size(4);
    p.ok = dt >= 0 && codes->scalar_type() == at::kByte && codes->size(3) == 128 && (row == 64 || row == 48) && q->size(2) == 1 && q->size(3) == 128 &&
           q->size(0) == codes->size(0);          // (more queries than sequences: the general path answers the first ones)
    for (int i = 2; i < 6 && p.ok; i++)
        if (const at::Tensor* m = p.take(args[i], 5)) p.type(m, q->scalar_type());
    if (!p.ok) Py_RETURN_NONE;
    return Py_BuildValue("(LLLLii)", (long long)q->size(0), (long long)q->size(1), (long long)codes->size(1), (long long)codes->size(2), row == 48 ? 1 : 0, dt);
}

// plain_cache(query, codes, rscale, rmn, tscale, tmn, key window, values, value codes, value scale, value zero point, mask)
//   -> (B, N, Nk, group rows, window rows, value rows, packed, type, mask row), or None
// of decode attention, with half-precision values [B, Nk, rows, 128] (no value codes) or with 4-bit values ([B, Nk, rows, 16], and the window's
// values [B, Nk, window rows, 128]); codes, window and mask may be None as the wrappers have it.
PyObject* plain_cache(PyObject*, PyObject* const* args, Py_ssize_t n) {
    if (n != 12) Py_RETURN_NONE;
    Plain p;
    if (!plain_tensor(args[0])) Py_RETURN_NONE;
    const int qdim = static_cast<int>(THPVariable_Unpack(args[0]).dim());
    const at::Tensor* q = qdim == 3 || qdim == 4 ? p.take(args[0], qdim) : nullptr;
    if (!q || !p.ok) Py_RETURN_NONE;
    const int dt = half_code(*q);
    const int64_t B = q->size(0), N = q->size(1);
    p.ok = dt >= 0 && q->size(-1) == 128 && q->numel() == B * N * 128 && reinterpret_cast<uintptr_t>(q->const_data_ptr()) % 16 == 0;
    if (!p.ok) Py_RETURN_NONE;
    const bool four = args[8] != Py_None || args[9] != Py_None || args[10] != Py_None;
    int64_t groups = 0, window = 0, rows = 0, Nk = 0;
    int packed = 0;
    if (args[1] != Py_None) {
        const at::Tensor* codes = p.take(args[1], 5);
        if (!codes) Py_RETURN_NONE;
        p.ok = codes->scalar_type() == at::kByte;
        groups = codes->size(2);
        packed = codes->size(4) == 48;
        for (int i = 2; i < 6 && p.ok; i++)
            if (const at::Tensor* m = p.take(args[i], 5)) p.type(m, q->scalar_type());
    }
    const at::Tensor* values = p.take(args[7], 4);
    if (!values) Py_RETURN_NONE;
    p.type(values, q->scalar_type());
    Nk = values->size(1);
    rows = values->size(2);
    if (args[6] != Py_None) {
        const at::Tensor* k = p.take(args[6], 4);
        if (!k) Py_RETURN_NONE;
        p.type(k, q->scalar_type());
        window = k->size(2);
    }
    if (four) {
        const at::Tensor* codes = p.take(args[8], 4);
        if (!codes || args[1] == Py_None || args[6] == Py_None) Py_RETURN_NONE;
        p.type(codes, at::kInt);
        p.ok = p.ok && values->sizes() == THPVariable_Unpack(args[6]).sizes();
        for (int i = 9; i < 11 && p.ok; i++)
            if (const at::Tensor* m = p.take(args[i], 4)) p.type(m, q->scalar_type());
        rows = codes->size(2);
    }
    int64_t mask_row = 0;
    if (p.ok && args[11] != Py_None) {
        const at::Tensor* m = p.take(args[11], 2);
        if (!m) Py_RETURN_NONE;
        p.type(m, at::kByte);
        mask_row = m->stride(0);
    }
    if (!p.ok) Py_RETURN_NONE;
    return Py_BuildValue("(LLLLLLiiL)", (long long)B, (long long)N, (long long)Nk, (long long)groups, (long long)window, (long long)rows, packed, dt,
                         (long long)mask_row);
}

// plain_rows(x, elements, bytes) -> (sizes and strides of x [a, b, c, 128], its type's code): half precision on a GPU with unit stride inside a
// row, the other strides multiples of `elements` and the base of `bytes`; else None
PyObject* plain_rows(PyObject*, PyObject* const* args, Py_ssize_t n) {
    uint64_t elements, bytes;
    if (n != 3 || !plain_tensor(args[0]) || !integer(args[1], elements) || !integer(args[2], bytes)) Py_RETURN_NONE;
    const at::Tensor& t = THPVariable_Unpack(args[0]);
    if (t.layout() != at::kStrided || !t.has_storage() || !t.is_cuda() || t.dim() != 4 || t.size(3) != 128 || t.stride(3) != 1) Py_RETURN_NONE;
    const int dt = half_code(t);
    const auto e = static_cast<int64_t>(elements);
    if (dt < 0 || t.stride(0) % e || t.stride(1) % e || t.stride(2) % e || reinterpret_cast<uintptr_t>(t.const_data_ptr()) % bytes) Py_RETURN_NONE;
    return Py_BuildValue("(LLL(LLLL)i)", (long long)t.size(0), (long long)t.size(1), (long long)t.size(2), (long long)t.stride(0),
                         (long long)t.stride(1), (long long)t.stride(2), (long long)t.stride(3), dt);
}

// empty(like, type, *sizes): torch.empty on like's device, of its type (0), uint8 (1), int32 (2) or float32 (3), in half the time
PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t n) {
    static constexpr at::ScalarType kTypes[] = {at::kHalf, at::kByte, at::kInt, at::kFloat};
    uint64_t type, size;
    c10::SmallVector<int64_t, 6> sizes;
    if (n < 2 || !THPVariable_Check(args[0]) || !integer(args[1], type) || type > 3) {
        if (!PyErr_Occurred()) PyErr_SetString(PyExc_TypeError, "empty(like, type, *sizes)");
        return nullptr;
    }
    for (Py_ssize_t i = 2; i < n; i++) {
        if (!integer(args[i], size)) return nullptr;
        sizes.push_back(static_cast<int64_t>(size));
    }
    try {
        const at::Tensor& like = THPVariable_Unpack(args[0]);
        const auto options = at::TensorOptions().device(like.device()).dtype(type ? kTypes[type] : like.scalar_type());
        return THPVariable_Wrap([&] {
            Released others;                    // (a first allocation, or freeing and waiting on the way to one, takes milliseconds)
            return at::empty(sizes, options);
        }());
    } catch (const c10::OutOfMemoryError& e) {
        PyErr_SetString(out_of_memory_error, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    }
    return nullptr;
}

// (sizes that are symbols and wrapped tensors throw: they are the general path's)
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* asked(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    try {
        return F(self, args, n);
    } catch (const std::exception&) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
}

PyMethodDef methods[] = {
    {"bind", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&bind)), METH_FASTCALL, nullptr},
    {"plain_eager", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&asked<plain_eager>)), METH_FASTCALL, nullptr},
    {"plain_half", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&asked<plain_half>)), METH_FASTCALL, nullptr},
    {"plain_scores", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&asked<plain_scores>)), METH_FASTCALL, nullptr},
    {"plain_cache", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&asked<plain_cache>)), METH_FASTCALL, nullptr},
    {"plain_rows", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&asked<plain_rows>)), METH_FASTCALL, nullptr},
    {"empty", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&empty)), METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_calls", nullptr, -1, methods};

PyObject* attribute(const char* from, const char* name) {
    PyObject* m = PyImport_ImportModule(from);
    PyObject* a = m ? PyObject_GetAttrString(m, name) : nullptr;
    Py_XDECREF(m);
    return a;
}

// torch's C++ types are those of the version this was compiled against
bool right_torch() {
    PyObject* version = attribute("torch", "__version__");
    PyObject* text = version ? PyObject_Str(version) : nullptr;
    const char* has = text ? PyUnicode_AsUTF8(text) : nullptr;
    const bool same = has && std::strncmp(has, TORCH_VERSION, std::strlen(TORCH_VERSION)) == 0;
    if (has && !same) PyErr_Format(PyExc_ImportError, "compiled against torch %s, loaded beside %s", TORCH_VERSION, has);
    Py_XDECREF(text);
    Py_XDECREF(version);
    return same;
}

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__calls(void) {
    argument_error = attribute("ctypes", "ArgumentError");
    parameter_class = argument_error ? attribute("torch.nn", "Parameter") : nullptr;
    out_of_memory_error = parameter_class ? attribute("torch", "OutOfMemoryError") : nullptr;
    return out_of_memory_error && right_torch() ? PyModule_Create(&module) : nullptr;
}
