// Python binding of the C ABI for torch tensors: `_binding`, a module whose functions are the entry points of
// include/scmx.h that enqueue work (and four of its queries), under the same names and with the same arguments except the
// last.  A pointer argument takes a tensor (contiguous, on the GPU), None or an integer address; a format argument an object
// whose buffer is the scmx_format; the stream is the caller's current one and is not passed.  A negative status raises.
//
// A decode step is a few hundred calls of a few microseconds of GPU work each, so the host's share per call decides: through
// ctypes a call cost 8-10 us (argument conversion; pointers, stream and format descriptor made in Python each time).  One
// GEMV call 11.9 -> 5.8 us, a linear layer on 40 rows 16.7 -> 10.3, a decode step of two OLMoE blocks 320 -> 205.  The
// allocation helpers are there for the same reason.
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ops/empty.h>
#include <c10/hip/HIPStream.h>

#include <exception>
#include <tuple>
#include <type_traits>
#include <utility>

#include "../../include/scmx.h"

namespace {

// A Python exception is set.
struct Raised {};

void fail(PyObject* type, const char* text) {
    PyErr_SetString(type, text);
    throw Raised();
}

// In a catch block: the Python exception of what was thrown, torch's own types (out of memory, a Python error) among them.
PyObject* raised() {
    try {
        throw;
    } catch (const Raised&) {
    } catch (...) {
        torch::translate_exception_to_python(std::current_exception());
    }
    return nullptr;
}

int64_t as_int(PyObject* o) {
    const int64_t v = PyLong_Check(o) ? PyLong_AsLongLong(o) : [&] {
        PyObject* i = PyNumber_Index(o);
        if (!i) throw Raised();
        const int64_t r = PyLong_AsLongLong(i);
        Py_DECREF(i);
        return r;
    }();
    if (v == -1 && PyErr_Occurred()) throw Raised();
    return v;
}

void* as_pointer(PyObject* o) {
    if (o == Py_None) return nullptr;
    if (THPVariable_Check(o)) {
        const at::Tensor& t = THPVariable_Unpack(o);
        if (!t.is_cuda()) fail(PyExc_ValueError, "scmx kernels take CUDA (ROCm) tensors; got a CPU tensor");
        if (!t.is_contiguous()) fail(PyExc_ValueError, "scmx kernels take contiguous tensors");
        return t.data_ptr();
    }
    return reinterpret_cast<void*>(as_int(o));
}

template <typename T>
T convert(PyObject* o) {
    if constexpr (std::is_same_v<T, const scmx_format*>) {
        Py_buffer b;
        if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) throw Raised();
        const bool whole = b.len >= Py_ssize_t(sizeof(scmx_format));
        const T p = static_cast<T>(b.buf);   // the caller's reference to the object keeps the memory
        PyBuffer_Release(&b);
        if (!whole) fail(PyExc_ValueError, "the format argument is smaller than a scmx_format");
        return p;
    } else if constexpr (std::is_pointer_v<T>) {
        return static_cast<T>(as_pointer(o));
    } else if constexpr (std::is_floating_point_v<T>) {
        const double v = PyFloat_AsDouble(o);
        if (v == -1.0 && PyErr_Occurred()) throw Raised();
        return T(v);
    } else {
        const int64_t v = as_int(o);
        if (int64_t(T(v)) != v || (std::is_unsigned_v<T> && v < 0)) fail(PyExc_ValueError, "integer argument out of range");
        return T(v);
    }
}

PyObject* status(const char* name, int rc) {
    if (rc == SCMX_OK) Py_RETURN_NONE;
    PyErr_Format(rc == SCMX_ERR_ARG || rc == SCMX_ERR_FORMAT || rc == SCMX_ERR_WORKSPACE ? PyExc_ValueError : PyExc_RuntimeError,
                 "%s failed (%d): %s", name, rc, scmx_last_error());
    return nullptr;
}

// One entry point as a METH_FASTCALL function: its parameters but the last from the arguments, the last the current stream.
template <auto FN, typename Sig = decltype(FN)>
struct Call;
template <auto FN, typename... P>
struct Call<FN, int (*)(P...)> {
    static const char* name;
    template <size_t... I>
    static int run(PyObject* const* args, std::index_sequence<I...>) {
        using Params = std::tuple<P...>;
        std::tuple<std::tuple_element_t<I, Params>...> v{convert<std::tuple_element_t<I, Params>>(args[I])...};
        void* stream = c10::hip::getCurrentHIPStream().stream();
        int rc;
        Py_BEGIN_ALLOW_THREADS;
        rc = FN(std::get<I>(v)..., stream);
        Py_END_ALLOW_THREADS;
        return rc;
    }
    static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
        constexpr size_t N = sizeof...(P) - 1;
        try {
            if (n != Py_ssize_t(N)) {
                PyErr_Format(PyExc_TypeError, "%s takes %zu arguments (the stream is the current one), got %zd", name, N, n);
                return nullptr;
            }
            return status(name, run(args, std::make_index_sequence<N>()));
        } catch (...) {
            return raised();
        }
    }
};
template <auto FN, typename... P>
const char* Call<FN, int (*)(P...)>::name = "";

// A size or choice the library answers without device work: every argument converted, the value returned.
template <auto FN, typename Sig = decltype(FN)>
struct Query;
template <auto FN, typename R, typename... P>
struct Query<FN, R (*)(P...)> {
    template <size_t... I>
    static PyObject* run(PyObject* const* args, std::index_sequence<I...>) {
        return PyLong_FromLongLong(static_cast<long long>(FN(convert<P>(args[I])...)));
    }
    static PyObject* call(PyObject*, PyObject* const* args, Py_ssize_t n) {
        try {
            if (n != Py_ssize_t(sizeof...(P))) fail(PyExc_TypeError, "wrong number of arguments");
            return run(args, std::index_sequence_for<P...>());
        } catch (const Raised&) {
            return nullptr;
        }
    }
};

struct NoGil {
    PyThreadState* const state = PyEval_SaveThread();
    ~NoGil() { PyEval_RestoreThread(state); }
};

// empty_<type>(like, dims...): an uninitialised tensor on the device of `like`.
template <at::ScalarType TYPE>
PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t n) {
    try {
        if (n < 2 || !THPVariable_Check(args[0])) fail(PyExc_TypeError, "empty_*(tensor, dims...)");
        int64_t dims[4];
        if (n > 5) fail(PyExc_TypeError, "at most four dimensions");
        for (Py_ssize_t i = 1; i < n; ++i) dims[i - 1] = as_int(args[i]);
        const at::Tensor& like = THPVariable_Unpack(args[0]);
        const at::TensorOptions options = at::TensorOptions().dtype(TYPE).device(like.device());
        at::Tensor t;
        {
            const NoGil released;   // the allocator may ask the driver, or wait for the GPU
            t = at::empty(at::IntArrayRef(dims, size_t(n - 1)), options);
        }
        return THPVariable_Wrap(std::move(t));
    } catch (...) {
        return raised();
    }
}

// A contiguous tensor on the GPU, and if `type` is given of that type; NULL: something else.
const at::Tensor* plain(PyObject* o, at::ScalarType type = at::ScalarType::Undefined) {
    if (!THPVariable_Check(o)) return nullptr;
    const at::Tensor& t = THPVariable_Unpack(o);
    return t.is_cuda() && t.is_contiguous() && (type == at::ScalarType::Undefined || t.scalar_type() == type) ? &t : nullptr;
}

// gemv(format, xq, xscale, codes, bcodes, wscale, N, epi, res, eidx, xstride, shared, pro, nw, eps): sc_decode.gemv for the operands of
// every decode step -- plain tensors, up to eight rows -- in one call: output (and workspace) allocated, the kernel launched.  None
// where an operand is anything else: the caller's general way converts or refuses it.  With both in Python a call on one row of
// 2048 x 2048 took the host 5.0 us, in its kernel's 4.0.
PyObject* gemv(PyObject*, PyObject* const* args, Py_ssize_t n) {
    try {
        if (n != 15) fail(PyExc_TypeError, "gemv takes 15 arguments");
        for (int i : {6, 7, 10, 12})
            if (!PyLong_Check(args[i])) Py_RETURN_NONE;
        if (args[11] != Py_None && !PyLong_Check(args[11])) Py_RETURN_NONE;
        const int N = convert<int>(args[6]), epi = convert<int>(args[7]), xstride = convert<int>(args[10]), pro = convert<int>(args[12]);
        const at::Tensor* x = plain(args[1], pro == 0 ? at::ScalarType::Char : at::ScalarType::BFloat16);
        const at::Tensor *codes = plain(args[3]), *bcodes = plain(args[4]), *wscale = plain(args[5]);
        const at::Tensor* xscale = pro == 0 ? plain(args[2]) : x;
        const at::Tensor* res = epi == SCMX_EPI_RES ? plain(args[8]) : x;
        const at::Tensor* nw = pro == 2 ? plain(args[13]) : x;
        if (!x || !codes || !bcodes || !wscale || !xscale || !res || !nw || x->dim() < 1 || x->dim() > 2) Py_RETURN_NONE;
        if (pro == 2 && !PyFloat_Check(args[14])) Py_RETURN_NONE;
        const at::Tensor* eidx = args[9] == Py_None ? nullptr : plain(args[9], at::ScalarType::Int);
        const int64_t rows = x->dim() == 2 ? x->size(0) : 1, K64 = x->size(-1), slots64 = eidx ? eidx->numel() : 0;
        if ((args[9] != Py_None && !eidx) || N < 0 || K64 > INT32_MAX || slots64 > INT32_MAX - 1 || (!eidx && rows > 8)) Py_RETURN_NONE;
        const scmx_format* fmt = convert<const scmx_format*>(args[0]);
        const int K = int(K64), shared = args[11] == Py_None ? -1 : convert<int>(args[11]);
        const float eps = pro == 2 ? convert<float>(args[14]) : 0.0f;
        const int batch = !eidx && rows > 1 ? int(rows) : 1, slots = int(slots64) + (args[11] != Py_None);
        const int64_t width = epi == SCMX_EPI_SWIGLU ? N / 2 : N;
        const auto ptr = [](const at::Tensor* t) { return t->data_ptr(); };
        at::Tensor out;
        int rc;
        {
            const NoGil released;   // the allocator may ask the driver, or wait for the GPU
            const at::TensorOptions options = at::TensorOptions().dtype(at::ScalarType::BFloat16).device(x->device());
            out = eidx ? at::empty({slots, width}, options) : batch > 1 ? at::empty({batch, width}, options) : at::empty({width}, options);
            const auto *xs = pro == 0 ? static_cast<const float*>(ptr(xscale)) : nullptr;
            const auto *rs = epi == SCMX_EPI_RES ? static_cast<const uint16_t*>(ptr(res)) : nullptr;
            const auto *w = pro == 2 ? static_cast<const uint16_t*>(ptr(nw)) : nullptr;
            const auto *c = static_cast<const uint32_t*>(ptr(codes));
            const auto *b = static_cast<const uint8_t*>(ptr(bcodes));
            const auto *s = static_cast<const float*>(ptr(wscale));
            auto* o = static_cast<uint16_t*>(out.data_ptr());
            if (eidx) {
                rc = scmx_gemv(fmt, ptr(x), xs, c, b, s, rs, o, epi, pro, w, eps, batch, N, K, static_cast<const int32_t*>(ptr(eidx)),
                               int(slots64), xstride, shared, c10::hip::getCurrentHIPStream().stream());
            } else {
                const size_t need = batch > 1 ? scmx_gemv_rows_workspace(fmt, pro, batch, N, K) : 0;
                const at::Tensor work = need ? at::empty({int64_t(need)}, options.dtype(at::ScalarType::Byte)) : at::Tensor();
                rc = scmx_gemv_rows(fmt, ptr(x), xs, c, b, s, rs, o, epi, pro, w, eps, batch, N, K, need ? work.data_ptr() : nullptr, need,
                                    c10::hip::getCurrentHIPStream().stream());
            }
        }
        if (rc != SCMX_OK) return status(eidx ? "scmx_gemv" : "scmx_gemv_rows", rc);
        return THPVariable_Wrap(std::move(out));
    } catch (...) {
        return raised();
    }
}

#define ENTRY(fn) \
    {#fn, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(((Call<&fn>::name = #fn), &Call<&fn>::call))), METH_FASTCALL, nullptr}
#define QUERY(fn) {#fn, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&Query<&fn>::call)), METH_FASTCALL, nullptr}
#define EMPTY(suffix, type) \
    {"empty_" #suffix, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&empty<at::ScalarType::type>)), METH_FASTCALL, nullptr}

PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_binding", nullptr, -1, nullptr, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__binding() {
    static PyMethodDef methods[] = {
        ENTRY(scmx_unpack_i8), ENTRY(scmx_act_quant), ENTRY(scmx_act_quant_blocked), ENTRY(scmx_mm_i8_i32), ENTRY(scmx_mm_epi),
        ENTRY(scmx_mm_w4a8), ENTRY(scmx_mm_w4a8_blocked), ENTRY(scmx_linear_w4a8), ENTRY(scmx_linear_w4a8_static),
        ENTRY(scmx_rmsnorm_quant), ENTRY(scmx_rmsnorm_quant_blocked), ENTRY(scmx_rmsnorm), ENTRY(scmx_linear_bf16), ENTRY(scmx_res_norm_quant),
        ENTRY(scmx_swiglu_quant), ENTRY(scmx_qkv_headnorm), ENTRY(scmx_qkv_headnorm_rope), ENTRY(scmx_qkv_fullnorm),
        ENTRY(scmx_qkv_fullnorm_rope), ENTRY(scmx_attn_decode), ENTRY(scmx_attn_decode_qkv), ENTRY(scmx_attn_prefill), ENTRY(scmx_attn_prefill_split),
        ENTRY(scmx_gemv), ENTRY(scmx_gemv_rows), ENTRY(scmx_route_topk), ENTRY(scmx_norm_linear), ENTRY(scmx_route_sort), ENTRY(scmx_moe_mm),
        ENTRY(scmx_moe_mm_i8), ENTRY(scmx_moe_mm_blocked), ENTRY(scmx_moe_gather_blocked), ENTRY(scmx_act_quant_sorted),
        ENTRY(scmx_moe_combine), ENTRY(scmx_moe_combine_blocked), ENTRY(scmx_rot_quant), ENTRY(scmx_mxfp4_to_sc),
        ENTRY(scmx_quantize_sc), ENTRY(scmx_quantize_family),
        QUERY(scmx_linear_w4a8_workspace), QUERY(scmx_gemv_rows_workspace), QUERY(scmx_mm_w4a8_prefers_blocked),
        QUERY(scmx_moe_mm_takes_slots),
        {"gemv", reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&gemv)), METH_FASTCALL, nullptr},
        EMPTY(bf16, BFloat16), EMPTY(i8, Char), EMPTY(u8, Byte), EMPTY(i32, Int), EMPTY(f32, Float),
        {nullptr, nullptr, 0, nullptr}};
    module_def.m_methods = methods;
    return PyModule_Create(&module_def);
}
