// Operator calls on torch tensors, natively: module `_torch_call`, used by ops.py.
//
// Every operator of the C-ABI becomes a vectorcall that takes the C function's arguments in order -- tensors (or None, or
// what pinned() returns) where it takes pointers, numbers elsewhere -- without the trailing stream, which is torch's current one.
// Conversion and checks are generated from the C signature.  The same call through ctypes spent 9 us of host time on a
// launch of 2.7 us (stream object 2.9 us, 0.3 us per pointer object); this way it is 3.5 us.
//
// The functions are looked up in the library that lib.py has loaded (bind), so a build of it with other kernels is called
// through the same module.  torch supplies memory and the stream; no torch type crosses the C-ABI.
#include <torch/csrc/autograd/python_variable.h>

#include <ATen/core/CachingHostAllocator.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/hip/impl/HIPStreamMasqueradingAsCUDA.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/utils/object_ptr.h>

#include <dlfcn.h>

#include <tuple>
#include <type_traits>
#include <utility>

#include "../../../include/cpmcu_amd.h"

namespace {

const char* (*g_last_error)(void) = nullptr;

template <typename Body>
auto without_gil(Body body) {
    struct Released {
        PyThreadState* state = PyEval_SaveThread();
        ~Released() { PyEval_RestoreThread(state); }
    } released;
    return body();
}

// Every entry of the module goes through one of these.  Asking a tensor for its memory or its layout throws where it has none (vmapped,
// fake, meta or sparse tensors), as do streams without a device: that is Python's RuntimeError, and must not cross the interpreter's C frames.
template <typename Body>
PyObject* guarded(Body body) {
    try {
        return body();
    } catch (const c10::Error& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what_without_backtrace());
    } catch (const std::exception& e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
    } catch (...) {
        PyErr_SetString(PyExc_RuntimeError, "an exception of unknown type");
    }
    return nullptr;
}
template <PyObject* (*F)(PyObject*, PyObject* const*, Py_ssize_t)>
PyObject* entry(PyObject* self, PyObject* const* args, Py_ssize_t nargs) {
    return guarded([&] { return F(self, args, nargs); });
}
template <PyObject* (*F)(PyObject*, PyObject*)>
PyObject* entry(PyObject* self, PyObject* arg) {
    return guarded([&] { return F(self, arg); });
}

// The name of pinned()'s capsules.
constexpr const char* kPinned = "cpmcu pinned memory";

// One C argument from one Python object; false with a Python error set.
template <typename T>
bool convert(PyObject* o, T* out) {
    if constexpr (std::is_pointer_v<T>) {
        if (o == Py_None) {
            *out = nullptr;
            return true;
        }
        if (THPVariable_Check(o)) {
            const at::Tensor& t = THPVariable_Unpack(o);
            if (!t.is_cuda() || !t.is_contiguous()) {
                PyErr_SetString(PyExc_AssertionError, "device-resident contiguous tensor required");
                return false;
            }
            *out = reinterpret_cast<T>(t.data_ptr());
            return true;
        }
        // (a bare number is no address: only what pinned() has looked at stands for memory that is not a device tensor's)
        if (!PyCapsule_IsValid(o, kPinned)) {
            PyErr_Format(PyExc_TypeError, "a tensor or None required, not %.100s", Py_TYPE(o)->tp_name);
            return false;
        }
        *out = reinterpret_cast<T>(PyCapsule_GetPointer(o, kPinned));
        return true;
    } else if constexpr (std::is_floating_point_v<T>) {
        *out = static_cast<T>(PyFloat_AsDouble(o));
    } else if constexpr (std::is_same_v<T, int>) {
        const long v = PyLong_AsLong(o);
        if (v < INT32_MIN || v > INT32_MAX) {
            PyErr_SetString(PyExc_OverflowError, "integer argument outside 32 bits");
            return false;
        }
        *out = static_cast<int>(v);
    } else {
        *out = static_cast<T>(PyLong_AsSize_t(o));
    }
    return !PyErr_Occurred();
}

// torch's current stream.  torch's default stream is HIP's null stream, which the library has to be told apart from "its own
// blocking stream": every launch on a blocking stream is ordered behind the null stream by a marker packet, 7-8 us between two
// launches (append of 9 rows in a row: 10.5 us each, 3 on the null stream itself).
void* current_stream() {
    void* const st = reinterpret_cast<void*>(c10::hip::getCurrentHIPStream().stream());
    return st ? st : CPMCU_STREAM_LEGACY;
}

PyObject* status(int rc) {
    if (rc == CPMCU_OK) Py_RETURN_NONE;
    PyErr_SetString(rc == CPMCU_ERR_INVALID_ARGUMENT ? PyExc_ValueError : PyExc_RuntimeError, g_last_error());
    return nullptr;
}

template <typename Fn>
struct Caller;
template <typename R, typename... A>
struct Caller<R (*)(A...)> {
    using Args = std::tuple<A...>;
    static constexpr size_t kAll = sizeof...(A);
    // a status-returning function whose last argument is void* takes the stream there
    static constexpr bool kStream = std::is_same_v<R, int> && std::is_same_v<std::tuple_element_t<kAll - 1, Args>, void*>;
    static constexpr size_t kGiven = kAll - (kStream ? 1 : 0);

    template <size_t... I>
    static bool fill(Args& a, PyObject* const* args, std::index_sequence<I...>) {
        return (convert(args[I], &std::get<I>(a)) && ...);
    }
    static PyObject* call(R (*fn)(A...), PyObject* const* args, Py_ssize_t nargs) {
        if (nargs != static_cast<Py_ssize_t>(kGiven)) {
            PyErr_Format(PyExc_TypeError, "%zd arguments given, %zd expected", nargs, static_cast<Py_ssize_t>(kGiven));
            return nullptr;
        }
        Args a;
        if (!fill(a, args, std::make_index_sequence<kGiven>{})) return nullptr;
        if constexpr (kStream) std::get<kAll - 1>(a) = current_stream();
        const R r = without_gil([&] { return std::apply(fn, a); });
        if constexpr (std::is_same_v<R, int>) return status(r);
        else return PyLong_FromSize_t(r);
    }
};

#define CPMCU_TORCH_CALLS(X)                                                                                              \
    X(kv_append) X(rope_table) X(rope_apply) X(gather_rows) X(head_weight_tile) X(head_workspace_bytes)                   \
    X(frspec_head_topk) X(lm_head_argmax) X(log_softmax_sliced) X(log_softmax_workspace_bytes) X(topk)                    \
    X(topk_workspace_bytes) X(remap) X(tree_accept) X(kv_compact) X(accept_commit) X(verify_tail) X(verify_tail_inplace)  \
    X(draft_tree_begin) X(draft_tree_extend) X(draft_tree_finish) X(draft_tree_finish_root)

#define X(name)                                                                                                    \
    decltype(&cpmcu_##name) fn_##name = nullptr;                                                                   \
    PyObject* call_##name(PyObject*, PyObject* const* args, Py_ssize_t nargs) {                                    \
        return Caller<decltype(&cpmcu_##name)>::call(fn_##name, args, nargs);                                      \
    }
CPMCU_TORCH_CALLS(X)
#undef X

// The one operator with host-side results: (num_partials, partial_stride).
decltype(&cpmcu_lm_head_partials) fn_lm_head_partials = nullptr;
PyObject* call_lm_head_partials(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 11) {
        PyErr_Format(PyExc_TypeError, "%zd arguments given, 11 expected", nargs);
        return nullptr;
    }
    const void *hidden, *w;
    int layout, n, V, H, apply_scale, num = 0, stride = 0;
    float scale;
    void *logits, *ws;
    size_t ws_bytes;
    if (!(convert(args[0], &hidden) && convert(args[1], &w) && convert(args[2], &layout) && convert(args[3], &n) && convert(args[4], &V) &&
          convert(args[5], &H) && convert(args[6], &apply_scale) && convert(args[7], &scale) && convert(args[8], &logits) &&
          convert(args[9], &ws) && convert(args[10], &ws_bytes)))
        return nullptr;
    void* const st = current_stream();
    const int rc =
        without_gil([&] { return fn_lm_head_partials(hidden, w, layout, n, V, H, apply_scale, scale, logits, ws, ws_bytes, &num, &stride, st); });
    if (rc != CPMCU_OK) return status(rc);
    return Py_BuildValue("ii", num, stride);
}

// A condition on the caller's tensors; false with an AssertionError set.
bool expect(bool ok, const char* what) {
    if (!ok) PyErr_SetString(PyExc_AssertionError, what);
    return ok;
}
const at::Tensor* tensor_or_null(PyObject* o) { return THPVariable_Check(o) ? &THPVariable_Unpack(o) : nullptr; }

// kv_append_rows(k_pool, v_pool, block_table, k_new, v_new, kv_len, Hkv): rows and types from the tensors.
PyObject* call_kv_append_rows(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 7) {
        PyErr_Format(PyExc_TypeError, "%zd arguments given, 7 expected", nargs);
        return nullptr;
    }
    void *k_pool, *v_pool;
    const int32_t *table, *kv_len;
    const void *k_new, *v_new;
    int Hkv;
    if (!(convert(args[0], &k_pool) && convert(args[1], &v_pool) && convert(args[2], &table) && convert(args[3], &k_new) &&
          convert(args[4], &v_new) && convert(args[5], &kv_len) && convert(args[6], &Hkv)))
        return nullptr;
    const at::Tensor *k = tensor_or_null(args[3]), *v = tensor_or_null(args[4]), *len = tensor_or_null(args[5]);
    if (!expect(k && v && len && k->dim() >= 1, "kv_append: tensors required") ||
        !expect(k->scalar_type() == at::kHalf && v->scalar_type() == at::kHalf && len->scalar_type() == at::kInt, "kv_append: element types") ||
        !expect(k->numel() == k->size(0) * Hkv * CPMCU_HEAD_DIM && v->numel() == k->numel(), "kv_append: shapes of the rows"))
        return nullptr;
    const int T = static_cast<int>(k->size(0));
    void* const st = current_stream();
    return status(without_gil([&] { return fn_kv_append(k_pool, v_pool, table, k_new, v_new, kv_len, T, Hkv, st); }));
}

// tree_attention_rows(q, k_pool, v_pool, block_table, kv_len, max_kv_len, k_new, v_new, rope, block_window_size, mask, mask_k_range, Hkv,
// scale, out, workspace, num_splits): shapes from the tensors.  None, or the bytes needed where the workspace is too small.
decltype(&cpmcu_tree_attention_window) fn_tree_attention_window = nullptr;
decltype(&cpmcu_tree_attention_workspace_bytes) fn_tree_attention_workspace_bytes = nullptr;
PyObject* call_tree_attention_rows(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs != 17) {
        PyErr_Format(PyExc_TypeError, "%zd arguments given, 17 expected", nargs);
        return nullptr;
    }
    const void *q, *k_new, *v_new;
    void *k_pool, *v_pool, *out, *ws;
    const int32_t *table, *kv_len;
    const float* rope;
    const uint64_t* mask;
    int max_kv_len, window, mask_k_range, Hkv, splits;
    float scale;
    if (!(convert(args[0], &q) && convert(args[1], &k_pool) && convert(args[2], &v_pool) && convert(args[3], &table) && convert(args[4], &kv_len) &&
          convert(args[5], &max_kv_len) && convert(args[6], &k_new) && convert(args[7], &v_new) && convert(args[8], &rope) &&
          convert(args[9], &window) && convert(args[10], &mask) && convert(args[11], &mask_k_range) && convert(args[12], &Hkv) &&
          convert(args[13], &scale) && convert(args[14], &out) && convert(args[15], &ws) && convert(args[16], &splits)))
        return nullptr;
    const at::Tensor *tq = tensor_or_null(args[0]), *len = tensor_or_null(args[4]), *tk = tensor_or_null(args[6]), *tv = tensor_or_null(args[7]),
                     *tr = tensor_or_null(args[8]), *tm = tensor_or_null(args[10]), *tw = tensor_or_null(args[15]);
    if (!expect(tq && len && tq->dim() == 3 && tq->size(2) == CPMCU_HEAD_DIM && tq->scalar_type() == at::kHalf, "tree_attention: q is [T, Hq, 128] of 16-bit floats") ||
        !expect(len->scalar_type() == at::kInt, "tree_attention: kv_len is int32"))
        return nullptr;
    const int64_t T = tq->size(0), Hq = tq->size(1);
    int W = 0;
    if (tm) {
        if (!expect((tm->scalar_type() == at::kLong || tm->scalar_type() == at::kUInt64) && T > 0 && tm->numel() % T == 0, "tree_attention: mask of 64-bit words, rows alike"))
            return nullptr;
        W = static_cast<int>(tm->numel() / T);
    }
    if (tk && !expect(tv && tk->scalar_type() == at::kHalf && tv->scalar_type() == at::kHalf && tk->numel() == T * Hkv * CPMCU_HEAD_DIM && tv->numel() == tk->numel(),
                      "tree_attention: k_new and v_new are [T, Hkv, 128] of 16-bit floats"))
        return nullptr;
    if (tr && !expect(tr->scalar_type() == at::kFloat && tr->numel() == T * CPMCU_HEAD_DIM, "tree_attention: rope is [T, 64, 2] of floats")) return nullptr;
    const size_t need = fn_tree_attention_workspace_bytes(static_cast<int>(T), static_cast<int>(Hq), Hkv, max_kv_len);
    const size_t have = tw ? static_cast<size_t>(tw->nbytes()) : 0;
    if (have < need) return PyLong_FromSize_t(need);
    void* const st = current_stream();
    return status(without_gil([&] {
        return fn_tree_attention_window(q, k_pool, v_pool, table, kv_len, max_kv_len, k_new, v_new, rope, window, mask, W, mask_k_range,
                                        static_cast<int>(T), static_cast<int>(Hq), Hkv, scale, out, ws, have, splits, st);
    }));
}

// empty(like, dtype, rows, cols, dtype, rows, cols, ...): uninitialised [rows, cols] tensors ([rows] where cols is 0) on like's
// device, as a tuple.  dtype: 'h' 16-bit float, 'f' fp32, 'i' int32, 'l' int64.
PyObject* empty(PyObject*, PyObject* const* args, Py_ssize_t nargs) {
    if (nargs < 4 || (nargs - 1) % 3 != 0 || !THPVariable_Check(args[0])) {
        PyErr_SetString(PyExc_TypeError, "empty(tensor, dtype, rows, cols, ...) expected");
        return nullptr;
    }
    if (!expect(THPVariable_Unpack(args[0]).is_cuda(), "device-resident contiguous tensor required")) return nullptr;
    const Py_ssize_t n = (nargs - 1) / 3;
    THPObjectPtr out(PyTuple_New(n));
    if (!out) return nullptr;
    const auto device = THPVariable_Unpack(args[0]).device();
    for (Py_ssize_t i = 0; i < n; ++i) {
        const char* code = PyUnicode_AsUTF8(args[1 + 3 * i]);
        const long rows = PyLong_AsLong(args[2 + 3 * i]), cols = PyLong_AsLong(args[3 + 3 * i]);
        if (PyErr_Occurred()) return nullptr;
        const auto type = code[0] == 'h' ? at::kHalf : code[0] == 'f' ? at::kFloat : code[0] == 'l' ? at::kLong : at::kInt;
        const int64_t sizes[2] = {rows, cols};
        PyObject* t = THPVariable_Wrap(at::detail::empty_cuda(at::IntArrayRef(sizes, cols ? 2 : 1), type, device, std::nullopt));
        if (!t) return nullptr;
        PyTuple_SET_ITEM(out.get(), i, t);
    }
    return out.release();
}

// pinned(tensor): a contiguous pinned host tensor's memory, in the place of a device tensor, for a call on the current stream: the GPU writes
// it through the mapped address.  The allocator is told of the stream, so that a tensor dropped before the work is done is not
// given to somebody else ahead of it (device memory is reused in stream order by itself).
PyObject* pinned(PyObject*, PyObject* o) {
    if (!THPVariable_Check(o)) {
        PyErr_SetString(PyExc_TypeError, "pinned(tensor) expected");
        return nullptr;
    }
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!expect(t.is_contiguous() && t.is_pinned(), "device-resident or pinned contiguous tensor required")) return nullptr;
    at::getHostAllocator(at::kCUDA)->record_event(t.data_ptr(), t.storage().data_ptr().get_context(), c10::hip::getCurrentHIPStreamMasqueradingAsCUDA().unwrap());
    return PyCapsule_New(t.data_ptr(), kPinned, nullptr);
}

// synchronize(): waits for torch's current stream.
PyObject* synchronize(PyObject*, PyObject*) {
    const auto stream = c10::hip::getCurrentHIPStream();
    without_gil([&] { stream.synchronize(); });
    Py_RETURN_NONE;
}

// bind(handle): the library's functions, from the handle lib.py loaded it under.
PyObject* bind(PyObject*, PyObject* handle) {
    void* h = PyLong_AsVoidPtr(handle);
    if (PyErr_Occurred()) return nullptr;
    auto find = [&](const char* name, auto* slot) {
        *slot = reinterpret_cast<std::remove_pointer_t<decltype(slot)>>(dlsym(h, name));
        if (!*slot) PyErr_Format(PyExc_ImportError, "the library does not export %s", name);
        return *slot != nullptr;
    };
    bool ok = find("cpmcu_last_error", &g_last_error) && find("cpmcu_lm_head_partials", &fn_lm_head_partials) &&
              find("cpmcu_tree_attention_window", &fn_tree_attention_window) &&
              find("cpmcu_tree_attention_workspace_bytes", &fn_tree_attention_workspace_bytes);
#define X(name) ok = ok && find("cpmcu_" #name, &fn_##name);
    CPMCU_TORCH_CALLS(X)
#undef X
    if (!ok) return nullptr;
    Py_RETURN_NONE;
}

#define ENTRY(name, fn) {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void*>(static_cast<PyObject* (*)(PyObject*, PyObject* const*, Py_ssize_t)>(entry<fn>))), METH_FASTCALL, nullptr},
#define X(name) ENTRY(#name, call_##name)
PyMethodDef g_methods[] = {
    CPMCU_TORCH_CALLS(X)
    X(lm_head_partials)
    X(kv_append_rows)
    X(tree_attention_rows)
    ENTRY("empty", empty)
    {"pinned", entry<pinned>, METH_O, nullptr},
    {"synchronize", entry<synchronize>, METH_NOARGS, nullptr},
    {"bind", entry<bind>, METH_O, nullptr},
    {nullptr, nullptr, 0, nullptr}};
#undef X
#undef ENTRY
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_torch_call", "The library's operators on torch tensors.", -1, g_methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__torch_call(void) { return PyModule_Create(&g_module); }
