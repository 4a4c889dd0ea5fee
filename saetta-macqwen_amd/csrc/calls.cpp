// The calls that a program makes per chunk and per token, from Python without ctypes: the tensors' checks and pointers, the
// current stream and the call of the C ABI in one step.  A small launch is 2.7 us of the host in the HIP runtime; a call through
// ctypes, with its checks in Python, was 2 to 3.5 us more.  (Host code only: the kernels are the library's, which is
// loaded from the path that `setup` was given when the first call needs it.)
#include <Python.h>

#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cstdarg>
#include <cstdio>
#include <cstring>
#include <exception>

#include "../../include/saetta_hip.h"

namespace {

struct Library {
    bool loaded;
    decltype(&saetta_last_error) last_error;
    decltype(&saetta_to_half) to_half;
    decltype(&saetta_kv_quantize) kv_quantize;
    decltype(&saetta_attn_prefill) attn_prefill;
    decltype(&saetta_attn_prefill_quant) attn_prefill_quant;
    decltype(&saetta_token_params_set) token_params_set;
    decltype(&saetta_plan_run) plan_run;
};

// What a copy of the package has set up (`setup`), kept with its module.
struct State {
    PyObject *error, *flash_params, *path;  // SaettaError, FlashParamsC, the library's path
    Library lib;
};
State &state_of(PyObject *module) { return *static_cast<State *>(PyModule_GetState(module)); }

// A Python exception is set.
struct Raised {};

[[noreturn]] void raise(PyObject *type, const char *fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    PyErr_FormatV(type, fmt, ap);
    va_end(ap);
    throw Raised{};
}

// (the GIL is held: one thread at a time gets here)
const Library &library(State &st) {
    Library &lib = st.lib;
    if (!lib.loaded) {
        if (!st.path) raise(PyExc_RuntimeError, "_saetta_calls: not set up");
        const char *path = PyUnicode_AsUTF8(st.path);
        if (!path) throw Raised{};
        void *h = dlopen(path, RTLD_NOW | RTLD_LOCAL);
        if (!h) raise(st.error, "%s is missing: run __graft_entry__.build() (make -C csrc): %s", path, dlerror());
        auto find = [&](auto &f, const char *name) {
            f = reinterpret_cast<std::remove_reference_t<decltype(f)>>(dlsym(h, name));
            if (!f) raise(st.error, "%s has no %s", path, name);
        };
        find(lib.last_error, "saetta_last_error"), find(lib.to_half, "saetta_to_half"), find(lib.kv_quantize, "saetta_kv_quantize");
        find(lib.attn_prefill, "saetta_attn_prefill"), find(lib.attn_prefill_quant, "saetta_attn_prefill_quant");
        find(lib.token_params_set, "saetta_token_params_set"), find(lib.plan_run, "saetta_plan_run");
        lib.loaded = true;
    }
    return lib;
}

// A contiguous tensor of `dtype` on the GPU.
const at::Tensor &need(PyObject *o, at::ScalarType dtype, const char *what) {
    if (THPVariable_Check(o)) {
        const at::Tensor &t = THPVariable_Unpack(o);
        if (t.scalar_type() == dtype && t.is_cuda() && t.is_contiguous()) return t;
    }
    raise(PyExc_TypeError, "%s: expected a contiguous torch.%s tensor on the GPU", what,
          dtype == at::kFloat ? "float32" : dtype == at::kHalf ? "float16" : "uint8");
}
template <class T>
T *pointer(const at::Tensor &t) {
    return static_cast<T *>(t.data_ptr());
}
// A tensor that a kernel can reach.
template <class T>
T *pointer_of(PyObject *o, const char *what) {
    if (THPVariable_Check(o)) {
        const at::Tensor &t = THPVariable_Unpack(o);
        if (t.is_cuda() || t.is_pinned()) return pointer<T>(t);
    }
    raise(PyExc_TypeError, "%s: expected a tensor on the GPU or in pinned memory", what);
}

long long integer(PyObject *o) {
    const long long v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) throw Raised{};
    return v;
}
uint32_t u32(PyObject *o) { return uint32_t(PyLong_AsUnsignedLongMask(o)); }

// None: torch's current stream of the current device.
saetta_stream_t stream_of(PyObject *o) {
    if (o == Py_None) return reinterpret_cast<saetta_stream_t>(c10::hip::getCurrentHIPStream().stream());
    void *p = PyLong_AsVoidPtr(o);
    if (!p && PyErr_Occurred()) throw Raised{};
    return reinterpret_cast<saetta_stream_t>(p);
}

saetta_flash_params flash_params(const State &st, PyObject *o, const char *what) {
    const int is = st.flash_params ? PyObject_IsInstance(o, st.flash_params) : 0;
    if (is < 0) throw Raised{};
    if (!is) raise(PyExc_TypeError, "%s: expected FlashParams", what);
    Py_buffer b;
    if (PyObject_GetBuffer(o, &b, PyBUF_SIMPLE)) throw Raised{};
    saetta_flash_params p;
    const bool fits = size_t(b.len) >= sizeof p;
    if (fits) memcpy(&p, b.buf, sizeof p);
    PyBuffer_Release(&b);
    if (!fits) raise(PyExc_TypeError, "%s: expected FlashParams", what);
    return p;
}

// Calls the library with the GIL released, as ctypes does (a launch waits where the queue is full).
template <class F>
PyObject *call(const char *what, const State &st, F f) {
    PyThreadState *thread = PyEval_SaveThread();
    const int rc = f();
    PyEval_RestoreThread(thread);
    if (rc) raise(st.error, "%s: %s (code %d)", what, st.lib.last_error(), rc);
    Py_RETURN_NONE;
}

template <class F>
PyObject *guarded(Py_ssize_t n, Py_ssize_t wanted, const char *what, F f) {
    try {
        if (n != wanted) raise(PyExc_TypeError, "%s takes %zd arguments (%zd given)", what, wanted, n);
        return f();
    } catch (const Raised &) {
        return nullptr;
    } catch (const std::exception &e) {
        PyErr_SetString(PyExc_RuntimeError, e.what());
        return nullptr;
    } catch (...) {
        PyErr_Format(PyExc_RuntimeError, "%s: unknown error", what);
        return nullptr;
    }
}

// setup(path, SaettaError, FlashParamsC)
PyObject *setup(PyObject *module, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 3, "setup", [&]() -> PyObject * {
        State &st = state_of(module);
        Py_INCREF(a[0]), Py_INCREF(a[1]), Py_INCREF(a[2]);
        Py_XSETREF(st.path, a[0]);
        Py_XSETREF(st.error, a[1]);
        Py_XSETREF(st.flash_params, a[2]);
        Py_RETURN_NONE;
    });
}

// to_half(x, out, stream)
PyObject *to_half(PyObject *module, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 3, "to_half", [&] {
        const at::Tensor &x = need(a[0], at::kFloat, "to_half x"), &out = need(a[1], at::kHalf, "to_half out");
        if (out.numel() < x.numel()) raise(PyExc_ValueError, "to_half: out does not hold x's values");
        State &st = state_of(module);
        const Library &lib = library(st);
        const saetta_stream_t s = stream_of(a[2]);
        const float *from = pointer<float>(x);
        uint16_t *to = pointer<uint16_t>(out);
        const size_t count = size_t(x.numel());
        return call("to_half", st, [&] { return lib.to_half(s, from, to, count); });
    });
}

// kv_encode(bits, per_token, capacity, data, scales, biases, x, pos, tokens, stream)
PyObject *kv_encode(PyObject *module, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 10, "kv_encode", [&] {
        const long long per_token = integer(a[1]), capacity = integer(a[2]), pos = integer(a[7]), tokens = integer(a[8]);
        const bool fit = tokens >= 0 && tokens <= capacity && pos >= 0 && pos <= capacity - tokens;
        if (!fit) raise(PyExc_ValueError, "QuantRows.encode: tokens do not fit");
        const at::Tensor &x = need(a[6], at::kFloat, "QuantRows.encode x");
        if (x.numel() < tokens * per_token * SAETTA_QUANT_GROUP) raise(PyExc_ValueError, "QuantRows.encode: tokens do not fit");
        const saetta_quant_rows rows{pointer_of<uint32_t>(a[3], "QuantRows.encode data"), pointer_of<uint16_t>(a[4], "QuantRows.encode scales"),
                                     pointer_of<uint16_t>(a[5], "QuantRows.encode biases")};
        State &st = state_of(module);
        const Library &lib = library(st);
        const saetta_stream_t s = stream_of(a[9]);
        const saetta_kv_quant_params p{uint32_t(per_token * tokens), uint32_t(per_token)};
        const int bits = int(integer(a[0]));
        const float *from = pointer<float>(x);
        return call("kv_quantize", st, [&] { return lib.kv_quantize(s, bits, from, rows, p, nullptr, uint32_t(pos)); });
    });
}

// prefill(kernel, q, keys, values, q_and_gate, out, p, workspace, stream)
PyObject *prefill(PyObject *module, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 9, "prefill", [&] {
        State &st = state_of(module);
        const saetta_flash_params p = flash_params(st, a[6], "prefill attention");
        if (p.heads != p.kv_heads * SAETTA_GQA_GROUP) raise(PyExc_ValueError, "%S needs 8 q heads per kv head", a[0]);
        const at::Tensor &q = need(a[1], at::kHalf, "q"), &keys = need(a[2], at::kHalf, "keys"), &values = need(a[3], at::kHalf, "values"),
                         &qg = need(a[4], at::kFloat, "q_and_gate"), &out = need(a[5], at::kFloat, "out"), &ws = need(a[7], at::kByte, "workspace");
        const Library &lib = library(st);
        const saetta_stream_t s = stream_of(a[8]);
        const uint16_t *q_ptr = pointer<uint16_t>(q), *k = pointer<uint16_t>(keys), *v = pointer<uint16_t>(values);
        const float *g = pointer<float>(qg);
        float *o = pointer<float>(out);
        void *w = ws.data_ptr();
        const size_t bytes = size_t(ws.numel());
        return call("attn_prefill", st, [&] { return lib.attn_prefill(s, q_ptr, k, v, g, o, p, w, bytes); });
    });
}

// prefill_quant(bits, q, keys' data, scales, biases, values' data, scales, biases, q_and_gate, out, p, workspace, stream)
PyObject *prefill_quant(PyObject *module, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 13, "prefill_quant", [&] {
        State &st = state_of(module);
        const saetta_flash_params p = flash_params(st, a[10], "prefill attention");
        if (p.heads != p.kv_heads * SAETTA_GQA_GROUP) raise(PyExc_ValueError, "prefill attention needs 8 q heads per kv head");
        const at::Tensor &q = need(a[1], at::kHalf, "q"), &qg = need(a[8], at::kFloat, "q_and_gate"), &out = need(a[9], at::kFloat, "out"),
                         &ws = need(a[11], at::kByte, "workspace");
        const saetta_quant_rows keys{pointer_of<uint32_t>(a[2], "keys"), pointer_of<uint16_t>(a[3], "keys"), pointer_of<uint16_t>(a[4], "keys")},
            values{pointer_of<uint32_t>(a[5], "values"), pointer_of<uint16_t>(a[6], "values"), pointer_of<uint16_t>(a[7], "values")};
        const Library &lib = library(st);
        const saetta_stream_t s = stream_of(a[12]);
        const int bits = int(integer(a[0]));
        const uint16_t *q_ptr = pointer<uint16_t>(q);
        const float *g = pointer<float>(qg);
        float *o = pointer<float>(out);
        void *w = ws.data_ptr();
        const size_t bytes = size_t(ws.numel());
        return call("attn_prefill_quant", st, [&] { return lib.attn_prefill_quant(s, bits, q_ptr, keys, values, g, o, p, w, bytes); });
    });
}

// token_params_set(params, token, position, kv_len, pad)
PyObject *token_params_set(PyObject *module, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 5, "token_params_set", [&] {
        saetta_token_params *to = pointer_of<saetta_token_params>(a[0], "token_params_set params");
        const saetta_token_params value{u32(a[1]), u32(a[2]), u32(a[3]), u32(a[4])};
        if (PyErr_Occurred()) throw Raised{};
        State &st = state_of(module);
        const Library &lib = library(st);
        const saetta_stream_t s = stream_of(Py_None);
        return call("token_params_set", st, [&] { return lib.token_params_set(s, to, value); });
    });
}

// plan_run(the plan's address, stream)
PyObject *plan_run(PyObject *module, PyObject *const *a, Py_ssize_t n) {
    return guarded(n, 2, "plan_run", [&] {
        const saetta_plan *plan = static_cast<const saetta_plan *>(PyLong_AsVoidPtr(a[0]));
        if (!plan && PyErr_Occurred()) throw Raised{};
        State &st = state_of(module);
        const Library &lib = library(st);
        const saetta_stream_t s = stream_of(a[1]);
        return call("plan_run", st, [&] { return lib.plan_run(s, plan); });
    });
}

#define FUNCTION(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(name)), METH_FASTCALL, nullptr}
PyMethodDef g_methods[] = {FUNCTION(setup), FUNCTION(to_half), FUNCTION(kv_encode), FUNCTION(prefill), FUNCTION(prefill_quant),
                           FUNCTION(token_params_set), FUNCTION(plan_run), {nullptr, nullptr, 0, nullptr}};
#undef FUNCTION

int traverse(PyObject *module, visitproc visit, void *arg) {
    const State &st = state_of(module);
    Py_VISIT(st.path);
    Py_VISIT(st.error);
    Py_VISIT(st.flash_params);
    return 0;
}
int clear(PyObject *module) {
    State &st = state_of(module);
    Py_CLEAR(st.path);
    Py_CLEAR(st.error);
    Py_CLEAR(st.flash_params);
    return 0;
}
// (a state per module object: a process may hold more than one copy of the package)
PyModuleDef_Slot g_slots[] = {{0, nullptr}};
PyModuleDef g_module = {PyModuleDef_HEAD_INIT, "_saetta_calls", nullptr, sizeof(State), g_methods, g_slots, traverse, clear, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__saetta_calls() { return PyModuleDef_Init(&g_module); }
