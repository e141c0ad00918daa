// Native host side of the operators that run once per layer and step: argument checks, output and scratch tensors and
// the call through the C ABI, as CPython functions.
//
// A decode-sized call keeps the GPU busy for 3 to 10 us, and through ctypes the same checks, allocations and argument
// conversions took 10 us of interpreter time per call (fp8 linear layer of one row, 4096 x 4096, quantiser and GEMM:
// 21 us of host time for 9 us of kernels), so the host was what such a layer ran at.  Here a call costs about 1 us
// beside the launches themselves.  The library is still reached only through include/llmk.h: bind() resolves the entry
// points of the library that the ctypes binding loaded.
//
// A function reads its arguments under the interpreter's lock and gives the lock up for everything that may wait:
// allocations, conversions of an operand, and the launches (a full queue, code that is loaded on first use).  Other Python
// threads run meanwhile, this function's other callers among them, so no two calls under way share scratch (see Scratch).
#include <dlfcn.h>
#include <string>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <ATen/ATen.h>
#include <ATen/hip/EmptyTensor.h>
#include <ATen/record_function.h>
#include <c10/core/DefaultDtype.h>
#include <c10/hip/HIPStream.h>
#include <hip/hip_runtime_api.h>

#include "../../include/llmk.h"

namespace {

#define LLMK_HOST_API(X)                                                                                              \
    X(llmk_last_error) X(llmk_gemm_workspace_bytes) X(llmk_act_quant_fp8) X(llmk_act_quant_i8) X(llmk_comm_quant_fp8) \
    X(llmk_quant_i8_rowwise) X(llmk_gemm_fp8_block) X(llmk_gemm_i8_block) X(llmk_gemm_i8_rowcol) X(llmk_gemm_w4a8)    \
    X(llmk_gemm_i8_rowcol_workspace_bytes) X(llmk_grouped_gemm_workspace_bytes)                                       \
    X(llmk_gemm_w4a8_workspace_bytes) X(llmk_gemm_w4a16_marlin) X(llmk_gemm_w4a16_marlin_workspace_bytes)             \
    X(llmk_gemm_w4a16_nk) X(llmk_gemm_w4a16_nk_workspace_bytes) X(llmk_moe_ep_preprocess)                             \
    X(llmk_moe_pre_reorder_quant) X(llmk_moe_act_and_mul_quant) X(llmk_moe_post_reorder) X(llmk_grouped_gemm)         \
    X(llmk_grouped_gemm_swiglu_quant) X(llmk_grouped_gemm_swiglu_quant_fused) X(llmk_moe_softmax_topk)                \
    X(llmk_weight_quant_w4a8) X(llmk_weight_quant_i8_block) X(llmk_weight_quant_fp8_block)                            \
    X(llmk_weight_dequant_fp8_block) X(llmk_weight_dequant_i8_block) X(llmk_weight_dequant_w4a8) X(llmk_quant_w4_nk)

// one per imported module object: the package and the top-level module layout may both be imported
struct State {
    PyObject* error;        // LlmkError of the binding module
    PyObject* workspaces;   // its {(device, stream): uint8 tensor}
#define X(name) decltype(&::name) name;
    LLMK_HOST_API(X)
#undef X
};

// Ends a call with a Python exception; call() sets it, with the interpreter's lock held again (no type: it is set already).
struct Raised {
    PyObject* type = nullptr;
    std::string msg;
};

[[noreturn]] void raise(PyObject* type, std::string msg) { throw Raised{type, std::move(msg)}; }
inline void require(bool ok, const char* msg) {
    if (!ok) raise(PyExc_AssertionError, msg);
}

// positional arguments of a METH_FASTCALL function (the Python wrappers pass all of them)
struct Args {
    State* st;
    PyObject* const* v;
    Args(PyObject* self, PyObject* const* args, Py_ssize_t n, Py_ssize_t want) : st((State*)PyModule_GetState(self)), v(args) {
        if (n != want) raise(PyExc_TypeError, "expected " + std::to_string(want) + " arguments, got " + std::to_string(n));
        if (!st->llmk_last_error) raise(PyExc_RuntimeError, "the kernel library is not bound");
    }
    const at::Tensor& tensor(int i) const {
        if (!THPVariable_Check(v[i])) raise(PyExc_TypeError, std::string("expected a torch.Tensor, got ") + Py_TYPE(v[i])->tp_name);
        return THPVariable_Unpack(v[i]);
    }
    bool none(int i) const { return v[i] == Py_None; }
    int64_t integer(int i) const {
        const long long r = PyLong_AsLongLong(v[i]);
        if (r == -1 && PyErr_Occurred()) throw Raised{};
        return r;
    }
    void on_gpu(const at::Tensor& t) const {
        if (!t.is_cuda())
            raise(st->error, "llm_kernels_amd kernels run on a HIP device only; got a " + t.device().str() +
                                 " tensor (no CPU fallback exists)");
    }
    template <class... T> void on_gpu(const at::Tensor& t, const T&... more) const {
        on_gpu(t);
        on_gpu(more...);
    }
    void check(int rc, const char* name, PyObject* type = nullptr) const {
        if (rc == 0) return;
        const char* msg = st->llmk_last_error();
        raise(type ? type : st->error, std::string(name) + " failed (rc=" + std::to_string(rc) + "): " + (msg ? msg : ""));
    }
};

inline int float_code(at::ScalarType t) {
    switch (t) {
        case at::kFloat: return LLMK_F32;
        case at::kHalf: return LLMK_F16;
        case at::kBFloat16: return LLMK_BF16;
        default: raise(PyExc_TypeError, std::string("unsupported floating dtype ") + c10::toString(t) + " (need float32/float16/bfloat16)");
    }
}
inline int id_bytes(const at::Tensor& t) {
    if (t.scalar_type() == at::kLong) return 8;
    if (t.scalar_type() == at::kInt) return 4;
    raise(PyExc_TypeError, std::string("expert id tensors must be int32 or int64, got ") + c10::toString(t.scalar_type()));
}
// torch.empty.  Where nothing but eager execution looks at the call, straight from its CUDA function, which saves 0.25 us
// a tensor (fp8 layer of one row, 4096 x 4096, three tensors: 9.5 us all through the dispatcher, 8.7 so).  Modes, tracing,
// functorch and autocast put a key into the thread's dispatch set, a profiler has callbacks, and
// torch.use_deterministic_algorithms fills a new tensor above that function.
inline at::Tensor empty(at::IntArrayRef sizes, at::ScalarType dt, const at::Tensor& like) {
    const c10::DispatchKeySet looking = c10::impl::tls_local_dispatch_key_set().included_ - c10::default_included_set;
    if (!looking.empty() || at::hasCallbacks() || at::globalContext().deterministicAlgorithms())
        return at::empty(sizes, at::TensorOptions(like.device()).dtype(dt));
    return at::Tensor(at::detail::empty_cuda(sizes, dt, like.device(), std::nullopt));
}
// sizes of t with the last one replaced
inline c10::SmallVector<int64_t, 6> with_last(const at::Tensor& t, int64_t last) {
    c10::SmallVector<int64_t, 6> s(t.sizes().begin(), t.sizes().end());
    s.back() = last;
    return s;
}
inline at::ScalarType default_dtype() { return c10::get_default_dtype_as_scalartype(); }
inline void* stream_of(const at::Tensor& t) { return (void*)c10::hip::getCurrentHIPStream(t.device().index()).stream(); }
inline at::Tensor as_type(const at::Tensor& t, at::ScalarType dt) { return t.scalar_type() == dt ? t : t.to(dt); }
inline int64_t last_size(const at::Tensor& t) { return t.size(-1); }
inline int64_t rows_of(const at::Tensor& t, int64_t cols) {
    if (cols == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    return t.numel() / cols;
}

// f() without the interpreter's lock: nothing in it touches a Python object
template <class F> auto unlocked(F&& f) {
    struct Release {
        PyThreadState* ts = PyEval_SaveThread();
        ~Release() { PyEval_RestoreThread(ts); }
    } release;
    return f();
}

// Scratch of one call: taken out of the dictionary {(device, stream): uint8 tensor} for as long as the call lasts, and put
// back once its launches are queued.  Calls on one stream run one after the other there, so the next one may have the same
// buffer; a call that another thread makes on that stream meanwhile finds none and allocates its own, because the launches
// of the two may alternate.  Of two buffers that come back the larger one is kept.
// Under capture a call takes a buffer from the graph's own pool instead: a graph goes on using it after the call, when one
// from the dictionary may have been replaced by a larger one and its memory given to another tensor.
// (Made and destroyed under the interpreter's lock, get() anywhere.)
class Scratch {
    const Args& a;
    const at::Tensor& like;
    const int64_t need;
    PyObject *key = nullptr, *held = nullptr;            // held: the dictionary's tensor, this call's while it lasts
    at::Tensor fresh;                                    // or one of its own

    bool capturing() const {
        hipStreamCaptureStatus status = hipStreamCaptureStatusNone;
        if (hipStreamIsCapturing((hipStream_t)stream_of(like), &status) != hipSuccess) (void)hipGetLastError();
        return status != hipStreamCaptureStatusNone;
    }
    static int64_t size(PyObject* o) { return o && THPVariable_Check(o) ? THPVariable_Unpack(o).numel() : 0; }

public:
    Scratch(const Args& args, const at::Tensor& t, int64_t bytes) : a(args), like(t), need(std::max<int64_t>(bytes, 0)) {
        if (!need || capturing()) return;
        key = Py_BuildValue("(iK)", (int)t.device().index(), (unsigned long long)(uintptr_t)stream_of(t));
        if (!key) throw Raised{};
        PyObject* o = PyDict_GetItemWithError(a.st->workspaces, key);
        if (!o) {
            PyErr_Clear();
            return;
        }
        if (size(o) >= need) Py_INCREF(held = o);
        PyDict_DelItem(a.st->workspaces, key);           // one that is too small goes before its successor is allocated
    }
    Scratch(const Scratch&) = delete;
    ~Scratch() {
        if (!key) return;
        PyObject *type, *value, *trace;
        PyErr_Fetch(&type, &value, &trace);
        if (fresh.defined()) held = THPVariable_Wrap(std::move(fresh));
        if (held && size(PyDict_GetItemWithError(a.st->workspaces, key)) < size(held)) PyDict_SetItem(a.st->workspaces, key, held);
        PyErr_Clear();                                   // a buffer that cannot be kept is freed, and the next call allocates
        Py_XDECREF(held);
        Py_DECREF(key);
        PyErr_Restore(type, value, trace);
    }
    void* get() {
        if (!need) return nullptr;
        if (held) return THPVariable_Unpack(held).data_ptr();
        if (!fresh.defined()) fresh = empty({std::max<int64_t>(need, 1 << 20)}, at::kByte, like);
        return fresh.data_ptr();
    }
    // the size asked for, not the size of the buffer: what a kernel does with its scratch (K splits) then depends on the
    // shape alone, never on what an earlier call left behind
    int64_t bytes() const { return need; }
};

PyObject* wrap(at::Tensor t) {
    PyObject* o = THPVariable_Wrap(std::move(t));
    if (!o) throw Raised{};
    return o;
}
template <class... T> PyObject* wrap_all(T... t) {
    PyObject* tup = PyTuple_New(sizeof...(T));
    if (!tup) throw Raised{};
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(tup, i++, wrap(std::move(t))), ...);
    return tup;
}

// ------------------------------------------------------------------ quantisers
// act_quant(x, block, form): form 0 e4m3 with fp32 scales, 1 / 2 int8 half-away / half-up with fp16 scales, 3 / 4 the
// payload forms (int8 half-up, e4m3 with fp16 scales), which report a refused shape as an AssertionError
PyObject* act_quant(const Args& a) {
    const at::Tensor& x = a.tensor(0);
    const int64_t block = a.integer(1);
    const int form = (int)a.integer(2);
    require(x.is_contiguous(), "Input tensor must be contiguous");
    const int64_t cols = last_size(x);
    if (block == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    if (cols % block)
        raise(PyExc_AssertionError, "Last dimension size must be divisible by block_size (block_size=" + std::to_string(block) + ")");
    a.on_gpu(x);
    const int dt = float_code(x.scalar_type());
    const bool fp8 = form == 0 || form == 4;
    const int64_t groups = x.numel() / block;
    at::Tensor y, s;
    unlocked([&] {
        y = empty(x.sizes(), fp8 ? at::kFloat8_e4m3fn : at::kChar, x);
        s = empty(with_last(x, cols / block), form == 0 ? at::kFloat : at::kHalf, x);
        if (form == 0)
            a.check(a.st->llmk_act_quant_fp8(x.data_ptr(), dt, y.data_ptr(), (float*)s.data_ptr(), groups, (int)block, stream_of(x)), "llmk_act_quant_fp8");
        else if (form == 4)
            a.check(a.st->llmk_comm_quant_fp8(x.data_ptr(), dt, y.data_ptr(), s.data_ptr(), LLMK_F16, groups, (int)block, stream_of(x)), "llmk_comm_quant_fp8", PyExc_AssertionError);
        else
            a.check(a.st->llmk_act_quant_i8(x.data_ptr(), dt, (int8_t*)y.data_ptr(), s.data_ptr(), groups, (int)block,
                                            form == 1 ? LLMK_ROUND_HALF_AWAY : LLMK_ROUND_HALF_UP, stream_of(x)),
                    "llmk_act_quant_i8", form == 3 ? PyExc_AssertionError : nullptr);
    });
    return wrap_all(std::move(y), std::move(s));
}

PyObject* rowwise_quant(const Args& a) {
    at::Tensor x = a.tensor(0);
    require(x.is_contiguous(), "Input tensor must be contiguous");
    a.on_gpu(x);
    const at::ScalarType t = x.scalar_type();
    at::Tensor y, s;
    unlocked([&] {
        if (t != at::kFloat && t != at::kHalf && t != at::kBFloat16) x = x.to(at::kFloat);
        const int64_t cols = last_size(x), rows = cols ? x.numel() / cols : 0;
        y = empty(x.sizes(), at::kChar, x);
        s = empty(x.sizes().slice(0, x.dim() - 1), at::kFloat, x);
        a.check(a.st->llmk_quant_i8_rowwise(x.data_ptr(), float_code(x.scalar_type()), (int8_t*)y.data_ptr(), (float*)s.data_ptr(), rows, cols, stream_of(x)),
                "llmk_quant_i8_rowwise");
    });
    return wrap_all(std::move(y), std::move(s));
}

// weight_quant(x, block, fp8): block x block tiles, e4m3 with fp32 scales or int8 (half-away) with fp16 scales
PyObject* weight_quant(const Args& g) {
    const at::Tensor& x = g.tensor(0);
    const int64_t block = g.integer(1);
    const bool fp8 = g.integer(2) != 0;
    require(x.is_contiguous(), "Input tensor must be contiguous");
    require(x.dim() == 2, "Input tensors must have 2 dimensions");
    g.on_gpu(x);
    if (block == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    const int dt = float_code(x.scalar_type());
    const int64_t N = x.size(0), K = x.size(1), nb = std::max<int64_t>(0, (N + block - 1) / block), kb = std::max<int64_t>(0, (K + block - 1) / block);
    at::Tensor y, s;
    unlocked([&] {
        y = empty(x.sizes(), fp8 ? at::kFloat8_e4m3fn : at::kChar, x);
        s = empty({nb, kb}, fp8 ? at::kFloat : at::kHalf, x);
        if (fp8) g.check(g.st->llmk_weight_quant_fp8_block(x.data_ptr(), dt, y.data_ptr(), (float*)s.data_ptr(), N, K, (int)block, stream_of(x)), "llmk_weight_quant_fp8_block");
        else g.check(g.st->llmk_weight_quant_i8_block(x.data_ptr(), dt, (int8_t*)y.data_ptr(), s.data_ptr(), N, K, (int)block, 127.f, LLMK_ROUND_HALF_AWAY, 0, stream_of(x)),
                     "llmk_weight_quant_i8_block");
    });
    return wrap_all(std::move(y), std::move(s));
}

// weight_dequant(y, s, block, fp8) in the default dtype
PyObject* weight_dequant(const Args& g) {
    const at::Tensor &x = g.tensor(0), &s = g.tensor(1);
    const int64_t block = g.integer(2);
    const bool fp8 = g.integer(3) != 0;
    require(x.is_contiguous() && s.is_contiguous(), "Input tensors must be contiguous");
    require(x.dim() == 2 && s.dim() == 2, "Input tensors must have 2 dimensions");
    g.on_gpu(x, s);
    const at::ScalarType out = default_dtype();
    at::Tensor y;
    unlocked([&] {
        y = empty(x.sizes(), out, x);
        if (fp8) {
            const at::Tensor s32 = as_type(s, at::kFloat);
            g.check(g.st->llmk_weight_dequant_fp8_block(x.data_ptr(), (const float*)s32.data_ptr(), y.data_ptr(), float_code(out), x.size(0), x.size(1), (int)block, stream_of(x)),
                    "llmk_weight_dequant_fp8_block");
        } else {
            g.check(g.st->llmk_weight_dequant_i8_block((const int8_t*)x.data_ptr(), s.data_ptr(), float_code(s.scalar_type()), y.data_ptr(), float_code(out), x.size(0), x.size(1), (int)block,
                                                       stream_of(x)), "llmk_weight_dequant_i8_block");
        }
    });
    return wrap(std::move(y));
}

// w4a8_weight_quant(x, group): 128 x 128 blocks, both levels and the packing
PyObject* w4a8_weight_quant(const Args& g) {
    const at::Tensor& x = g.tensor(0);
    const int64_t group = g.integer(1), N = x.size(0), K = x.size(1);
    at::Tensor packed, s, s4, z4;
    unlocked([&] {
        packed = empty({N / 8, K}, at::kInt, x);
        s = empty({(N + 127) / 128, K / 128}, at::kHalf, x);
        s4 = empty({N, K / group}, at::kChar, x);
        z4 = empty({N, K / group}, at::kChar, x);
        g.check(g.st->llmk_weight_quant_w4a8(x.data_ptr(), float_code(x.scalar_type()), (int32_t*)packed.data_ptr(), s.data_ptr(), (int8_t*)s4.data_ptr(), (int8_t*)z4.data_ptr(), N, K, (int)group,
                                             stream_of(x)), "llmk_weight_quant_w4a8");
    });
    return wrap_all(std::move(packed), std::move(s), std::move(s4), std::move(z4));
}

// w4a8_weight_dequant(packed, s, s4, z4, block, group) -> fp16
PyObject* w4a8_weight_dequant(const Args& g) {
    const at::Tensor &y = g.tensor(0), &s_in = g.tensor(1), &s4_in = g.tensor(2), &z4_in = g.tensor(3);
    g.on_gpu(y, s_in, s4_in, z4_in);
    const int block = (int)g.integer(4), group = (int)g.integer(5);
    at::Tensor out;
    unlocked([&] {
        const at::Tensor s = s_in.contiguous(), s4 = s4_in.contiguous(), z4 = z4_in.contiguous();
        const int64_t K = y.size(1), N = y.size(0) * 8;
        out = empty({N, K}, at::kHalf, y);
        g.check(g.st->llmk_weight_dequant_w4a8((const int32_t*)y.data_ptr(), s.data_ptr(), (const int8_t*)s4.data_ptr(), (const int8_t*)z4.data_ptr(), out.data_ptr(), N, K, block, group,
                                               stream_of(y)), "llmk_weight_dequant_w4a8");
    });
    return wrap(std::move(out));
}

// w4_quantize_nk(w, group) -> (packed, scales, codes)
PyObject* w4_quantize_nk(const Args& g) {
    const int64_t group = g.integer(1);
    if (group == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
    const at::Tensor& in = g.tensor(0);
    require(in.dim() == 2 && in.size(1) % group == 0, "");
    const at::ScalarType t = in.scalar_type();
    require(t == at::kFloat || t == at::kHalf || t == at::kBFloat16, "weights must be fp32, fp16 or bf16");
    g.on_gpu(in);
    at::Tensor packed, s, q;
    unlocked([&] {
        const at::Tensor w = in.contiguous();
        const int64_t N = w.size(0), K = w.size(1);
        packed = empty({N, K / 8}, at::kInt, w);
        s = empty({N, K / group}, at::kHalf, w);
        q = empty({N, K}, at::kByte, w);
        g.check(g.st->llmk_quant_w4_nk(w.data_ptr(), float_code(t), (int32_t*)packed.data_ptr(), s.data_ptr(), (uint8_t*)q.data_ptr(), N, K, (int)group, stream_of(w)), "llmk_quant_w4_nk",
                PyExc_AssertionError);
    });
    return wrap_all(std::move(packed), std::move(s), std::move(q));
}

// ------------------------------------------------------------------ dense GEMMs
void check_gemm(const Args& g, const at::Tensor& a, const at::Tensor& a_s, const at::Tensor& b, const at::Tensor& b_s) {
    require(a.is_contiguous() && b.is_contiguous(), "Input tensors must be contiguous");
    require(a_s.is_contiguous() && b_s.is_contiguous(), "Scaling factor tensors must be contiguous");
    g.on_gpu(a, a_s, b, b_s);
}

PyObject* fp8_gemm(const Args& g) {
    const at::Tensor &a = g.tensor(0), &a_s = g.tensor(1), &b = g.tensor(2), &b_s = g.tensor(3);
    check_gemm(g, a, a_s, b, b_s);
    const int64_t K = last_size(a), M = rows_of(a, K), N = b.size(0);
    require(a_s.scalar_type() == at::kFloat && b_s.scalar_type() == at::kFloat, "fp8 scales must be float32");
    const at::ScalarType out = default_dtype();
    Scratch ws(g, a, g.st->llmk_gemm_workspace_bytes(M, N, K));
    at::Tensor c;
    unlocked([&] {
        c = empty(with_last(a, N), out, a);
        g.check(g.st->llmk_gemm_fp8_block(a.data_ptr(), (const float*)a_s.data_ptr(), b.data_ptr(), (const float*)b_s.data_ptr(), c.data_ptr(), float_code(out), M, N, K,
                                          ws.get(), ws.bytes(), stream_of(a)), "llmk_gemm_fp8_block", PyExc_AssertionError);
    });
    return wrap(std::move(c));
}

PyObject* int8_gemm(const Args& g) {
    const at::Tensor &a = g.tensor(0), &a_s = g.tensor(1), &b = g.tensor(2), &b_s = g.tensor(3);
    check_gemm(g, a, a_s, b, b_s);
    const int64_t K = last_size(a), M = rows_of(a, K), N = b.size(0);
    require(a_s.scalar_type() == b_s.scalar_type(), "activation and weight scales must share a dtype");
    const at::ScalarType out = default_dtype();
    Scratch ws(g, a, g.st->llmk_gemm_workspace_bytes(M, N, K));
    at::Tensor c;
    unlocked([&] {
        c = empty(with_last(a, N), out, a);
        g.check(g.st->llmk_gemm_i8_block((const int8_t*)a.data_ptr(), a_s.data_ptr(), (const int8_t*)b.data_ptr(), b_s.data_ptr(), float_code(a_s.scalar_type()), c.data_ptr(),
                                         float_code(out), M, N, K, ws.get(), ws.bytes(), stream_of(a)), "llmk_gemm_i8_block", PyExc_AssertionError);
    });
    return wrap(std::move(c));
}

// int8_gemm_per_token(a, a_s, b, b_s, with int32 accumulators)
PyObject* int8_gemm_per_token(const Args& g) {
    const at::Tensor &a = g.tensor(0), &a_s_in = g.tensor(1), &b = g.tensor(2), &b_s_in = g.tensor(3);
    require(a.is_contiguous() && b.is_contiguous(), "Input tensors must be contiguous");
    g.on_gpu(a, a_s_in, b, b_s_in);
    const int64_t K = last_size(a), M = rows_of(a, K), N = b.size(0);
    require(a_s_in.numel() == M && b_s_in.numel() == N, "need one scale per token and per output channel");
    const at::ScalarType out = default_dtype();
    const bool want_acc = g.integer(4) != 0;
    Scratch ws(g, a, g.st->llmk_gemm_i8_rowcol_workspace_bytes(M, N, K));
    at::Tensor c, acc;
    unlocked([&] {
        const at::Tensor a_s = as_type(a_s_in, at::kFloat).contiguous(), b_s = as_type(b_s_in, at::kFloat).contiguous();
        c = empty(with_last(a, N), out, a);
        if (want_acc) acc = empty(with_last(a, N), at::kInt, a);
        g.check(g.st->llmk_gemm_i8_rowcol((const int8_t*)a.data_ptr(), (const float*)a_s.data_ptr(), (const int8_t*)b.data_ptr(), (const float*)b_s.data_ptr(), c.data_ptr(), float_code(out),
                                          want_acc ? (int32_t*)acc.data_ptr() : nullptr, M, N, K, ws.get(), ws.bytes(), stream_of(a)), "llmk_gemm_i8_rowcol", PyExc_AssertionError);
    });
    return want_acc ? wrap_all(std::move(c), std::move(acc)) : wrap(std::move(c));
}

// w4a8_gemm(a, a_s, b, b_s, b_s4, b_z4, group)
PyObject* w4a8_gemm(const Args& g) {
    const at::Tensor &a = g.tensor(0), &a_s = g.tensor(1), &b = g.tensor(2), &b_s = g.tensor(3), &s4 = g.tensor(4), &z4 = g.tensor(5);
    require(a.is_contiguous() && b.is_contiguous(), "Input tensors must be contiguous");
    require(a_s.is_contiguous() && b_s.is_contiguous(), "Scaling factor tensors must be contiguous");
    require(s4.is_contiguous() && z4.is_contiguous(), "Scaling factor and zero point tensors must be contiguous");
    g.on_gpu(a, a_s, b, b_s, s4, z4);
    const int64_t K = last_size(a), M = rows_of(a, K), N = b.size(0) * 8;
    const int group = (int)g.integer(6);
    require(a_s.scalar_type() == b_s.scalar_type(), "activation and weight scales must share a dtype");
    const at::ScalarType out = default_dtype();
    // what this shape's kernels use: fp32 sums of K slices, or the expanded int8 weights and the int8 GEMM's scratch
    Scratch ws(g, a, g.st->llmk_gemm_w4a8_workspace_bytes(M, N, K, group));
    at::Tensor c;
    unlocked([&] {
        c = empty(with_last(a, N), out, a);
        g.check(g.st->llmk_gemm_w4a8((const int8_t*)a.data_ptr(), a_s.data_ptr(), (const int32_t*)b.data_ptr(), b_s.data_ptr(), float_code(a_s.scalar_type()), (const int8_t*)s4.data_ptr(),
                                     (const int8_t*)z4.data_ptr(), c.data_ptr(), float_code(out), M, N, K, group, ws.get(), ws.bytes(), stream_of(a)), "llmk_gemm_w4a8", PyExc_AssertionError);
    });
    return wrap(std::move(c));
}

// w4a16_gemm(x, packed, scales, group)
PyObject* w4a16_gemm(const Args& g) {
    const at::Tensor &x = g.tensor(0), &w = g.tensor(1), &s = g.tensor(2);
    const int group = (int)g.integer(3);
    require(x.is_contiguous() && w.is_contiguous() && s.is_contiguous(), "Input tensors must be contiguous");
    require(w.scalar_type() == at::kInt && s.scalar_type() == at::kHalf, "");
    g.on_gpu(x, w, s);
    const int64_t K = last_size(x), M = rows_of(x, K), N = w.size(0);
    require(w.size(1) * 8 == K, "packed weight must be [N, K/8]");
    require(x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16, "activations must be fp16 or bf16");
    const int dt = float_code(x.scalar_type());
    Scratch ws(g, x, g.st->llmk_gemm_w4a16_nk_workspace_bytes(M, N, K, group, dt));
    at::Tensor y;
    unlocked([&] {
        y = empty(with_last(x, N), x.scalar_type(), x);
        g.check(g.st->llmk_gemm_w4a16_nk(x.data_ptr(), (const int32_t*)w.data_ptr(), y.data_ptr(), s.data_ptr(), dt, M, N, K, group, ws.get(), ws.bytes(), stream_of(x)),
                "llmk_gemm_w4a16_nk", PyExc_AssertionError);
    });
    return wrap(std::move(y));
}

// marlin_mul(A, B, C, s)
PyObject* marlin_mul(const Args& g) {
    const at::Tensor &A = g.tensor(0), &B = g.tensor(1), &C = g.tensor(2), &s = g.tensor(3);
    auto fail = [](const std::string& m) { raise(PyExc_RuntimeError, m); };
    const int64_t M = A.size(0), K = A.size(1), N = C.size(1);
    if (M % 16 || N % 16 || K % 16)
        fail("Matrix dimensions must be divisible by 16. Got M=" + std::to_string(M) + ", N=" + std::to_string(N) + ", K=" + std::to_string(K));
    if (!(A.is_cuda() && B.device() == A.device() && C.device() == A.device() && s.device() == A.device())) fail("All tensors must be on the same CUDA device");
    if (A.scalar_type() != at::kHalf || C.scalar_type() != at::kHalf) fail("A and C matrices must be of type torch.float16");
    if (s.scalar_type() != at::kHalf) fail("Scale tensor must be of type torch.float16");
    if (B.scalar_type() != at::kInt) fail("B matrix must be packed INT4 data (torch.int32)");
    if (!C.is_contiguous()) fail("C must be contiguous (the result is written in place)");
    if (C.size(0) != M) fail("C must have as many rows as A");
    int64_t group = -1;
    if (s.dim() == 2) {
        if (s.size(1) != N) fail("Scale tensor N dimension mismatch: expected " + std::to_string(N) + " but got " + std::to_string(s.size(1)));
        if (s.size(0) == 0) raise(PyExc_ZeroDivisionError, "integer division or modulo by zero");
        group = K / s.size(0);
        if (group == 0 || K % group) fail("K dimension not divisible by groupsize: K=" + std::to_string(K) + ", groupsize=" + std::to_string(group));
    }
    if (B.numel() * 8 != K * N) fail("B does not hold K*N packed 4-bit values");
    Scratch ws(g, A, g.st->llmk_gemm_w4a16_marlin_workspace_bytes(M, N, K));
    unlocked([&] {
        const at::Tensor a = A.contiguous(), b = B.contiguous(), sc = s.contiguous();
        g.check(g.st->llmk_gemm_w4a16_marlin(a.data_ptr(), (const int32_t*)b.data_ptr(), C.data_ptr(), sc.data_ptr(), M, N, K, (int)group, ws.get(), ws.bytes(), stream_of(A)),
                "llmk_gemm_w4a16_marlin", PyExc_RuntimeError);
    });
    Py_RETURN_NONE;
}

// ------------------------------------------------------------------ mixture of experts
// softmax_topk(logits [.., E], topk, renormalize) -> (ids int64, weights fp32)
PyObject* softmax_topk(const Args& g) {
    const at::Tensor& in = g.tensor(0);
    const int64_t topk = g.integer(1), E = last_size(in), T = rows_of(in, E);
    const bool renorm = g.integer(2) != 0;
    at::Tensor ids, w;
    unlocked([&] {
        const at::Tensor x = in.contiguous();
        ids = empty(with_last(x, topk), at::kLong, x);
        w = empty(with_last(x, topk), at::kFloat, x);
        g.check(g.st->llmk_moe_softmax_topk(x.data_ptr(), float_code(x.scalar_type()), (int64_t*)ids.data_ptr(), (float*)w.data_ptr(), T, (int)E, (int)topk, renorm, stream_of(x)),
                "llmk_moe_softmax_topk");
    });
    return wrap_all(std::move(ids), std::move(w));
}

// ep_preprocess(topk_ids, num_experts) -> (sorted ids, src2dst, seg_indptr); contiguous int32 / int64 ids within the limits
PyObject* ep_preprocess(const Args& g) {
    const at::Tensor& ids = g.tensor(0);
    g.on_gpu(ids);
    const int64_t n = ids.numel(), E = g.integer(1);
    at::Tensor sorted, src2dst, seg;
    unlocked([&] {
        sorted = empty({n}, ids.scalar_type(), ids);
        src2dst = empty({n}, at::kInt, ids);
        seg = empty({E + 1}, at::kLong, ids);
        g.check(g.st->llmk_moe_ep_preprocess(ids.data_ptr(), id_bytes(ids), n, (int)E, sorted.data_ptr(), (int32_t*)src2dst.data_ptr(), (int64_t*)seg.data_ptr(), stream_of(ids)),
                "llmk_moe_ep_preprocess");
    });
    return wrap_all(std::move(sorted), std::move(src2dst), std::move(seg));
}

struct QuantBuffers {
    at::Tensor q, s;
    int kind;
};
// the 1 x 128 activation format that goes with a weight dtype (0 int8, 1 e4m3)
QuantBuffers quant_buffers(int64_t rows, int64_t cols, int64_t fp8, const at::Tensor& like) {
    require(cols % 128 == 0, "row length must be a multiple of 128");
    return {empty({rows, cols}, fp8 ? at::kFloat8_e4m3fn : at::kChar, like), empty({rows, cols / 128}, fp8 ? at::kFloat : at::kHalf, like),
            fp8 ? LLMK_KIND_FP8 : LLMK_KIND_I8};
}
// an optional tensor argument (undefined for None), and its fp32 / int64 form
at::Tensor optional(const Args& g, int i) { return g.none(i) ? at::Tensor() : g.tensor(i); }
at::Tensor f32_contiguous(const at::Tensor& t) { return t.defined() ? as_type(t, at::kFloat).contiguous() : t; }
inline void* ptr_or_null(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
at::Tensor long_contiguous(const at::Tensor& t) { return t.defined() ? as_type(t, at::kLong).contiguous() : t; }

// pre_reorder_quant(input, src2dst, topk_ids, a1_scales, start, end, topk, hidden, fp8)
PyObject* pre_reorder_quant(const Args& g) {
    const at::Tensor &x = g.tensor(0), &src2dst = g.tensor(1), &ids = g.tensor(2);
    g.on_gpu(x, src2dst, ids);
    require(x.is_contiguous() && src2dst.is_contiguous() && ids.is_contiguous(), "");
    require(x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16, "");
    const int64_t start = g.integer(4), end = g.integer(5), topk = g.integer(6), hidden = g.integer(7), fp8 = g.integer(8), T = rows_of(x, hidden);
    const at::Tensor scales = optional(g, 3);
    QuantBuffers o;
    unlocked([&] {
        o = quant_buffers(T * topk, hidden, fp8, x);
        const at::Tensor sc = f32_contiguous(scales);
        g.check(g.st->llmk_moe_pre_reorder_quant(x.data_ptr(), float_code(x.scalar_type()), o.q.data_ptr(), o.s.data_ptr(), o.kind, LLMK_ROUND_HALF_AWAY, (const int32_t*)src2dst.data_ptr(),
                                                 ids.data_ptr(), id_bytes(ids), (const float*)ptr_or_null(sc), (int)start, (int)end, (int)topk, T, hidden, stream_of(x)),
                "llmk_moe_pre_reorder_quant");
    });
    return wrap_all(std::move(o.q), std::move(o.s));
}

// act_and_mul_quant(gateup, two_i, reorder_ids, scales, start, end, fp8, act)
PyObject* act_and_mul_quant(const Args& g) {
    const at::Tensor &x = g.tensor(0), &ids = g.tensor(2);
    g.on_gpu(x, ids);
    require(x.is_contiguous() && ids.is_contiguous(), "");
    require(x.scalar_type() == at::kHalf || x.scalar_type() == at::kBFloat16, "");
    const int64_t two_i = g.integer(1), start = g.integer(4), end = g.integer(5), fp8 = g.integer(6), act = g.integer(7), M = rows_of(x, two_i);
    const at::Tensor scales = optional(g, 3);
    QuantBuffers o;
    unlocked([&] {
        o = quant_buffers(M, two_i / 2, fp8, x);
        const at::Tensor sc = f32_contiguous(scales);
        g.check(g.st->llmk_moe_act_and_mul_quant(x.data_ptr(), float_code(x.scalar_type()), o.q.data_ptr(), o.s.data_ptr(), o.kind, LLMK_ROUND_HALF_AWAY, ids.data_ptr(), id_bytes(ids),
                                                 (const float*)ptr_or_null(sc), (int)start, (int)end, M, two_i, (int)act, stream_of(x)),
                "llmk_moe_act_and_mul_quant");
    });
    return wrap_all(std::move(o.q), std::move(o.s));
}

// post_reorder(down, out, src2dst, topk_ids, topk_weights, start, end, topk, hidden)
PyObject* post_reorder(const Args& g) {
    const at::Tensor &down = g.tensor(0), &out = g.tensor(1), &src2dst = g.tensor(2), &ids = g.tensor(3), &w = g.tensor(4);
    g.on_gpu(down, out, src2dst, ids, w);
    require(down.is_contiguous() && out.is_contiguous() && w.is_contiguous(), "");
    require(down.scalar_type() == out.scalar_type(), "");
    const int64_t start = g.integer(5), end = g.integer(6), topk = g.integer(7), hidden = g.integer(8), T = rows_of(out, hidden);
    unlocked([&] {
        g.check(g.st->llmk_moe_post_reorder(down.data_ptr(), out.data_ptr(), float_code(out.scalar_type()), (const int32_t*)src2dst.data_ptr(), ids.data_ptr(), id_bytes(ids), w.data_ptr(),
                                            float_code(w.scalar_type()), (int)start, (int)end, (int)topk, T, hidden, stream_of(out)), "llmk_moe_post_reorder");
    });
    Py_INCREF(g.v[1]);
    return g.v[1];
}

inline int operand_kind(at::ScalarType t) {
    switch (t) {
        case at::kChar: return LLMK_KIND_I8;
        case at::kFloat8_e4m3fn: return LLMK_KIND_FP8;
        case at::kHalf: return LLMK_KIND_F16;
        case at::kBFloat16: return LLMK_KIND_BF16;
        default: raise(PyExc_AssertionError, std::string("unsupported operand dtype ") + c10::toString(t));
    }
}

// grouped_gemm(a, b, c, batch_size, seg_indptr, weight_indices, scale_a, scale_b): operands already in the weights' type
PyObject* grouped_gemm(const Args& g) {
    const at::Tensor &a = g.tensor(0), &b = g.tensor(1), &c = g.tensor(2);
    require(a.is_contiguous() && b.is_contiguous() && c.is_contiguous(), "Input tensors must be contiguous");
    require(b.dim() == 3 && last_size(a) == last_size(b) && last_size(c) == b.size(1) && c.size(0) == a.size(0), "");
    require(a.scalar_type() == b.scalar_type(), "a and b must share a dtype after activation quantisation");
    const int kind = operand_kind(b.scalar_type());
    const bool scaled = kind == LLMK_KIND_I8 || kind == LLMK_KIND_FP8;
    const int64_t E = g.integer(3), M = a.size(0), N = b.size(1), K = b.size(2);
    const at::Tensor& seg_in = g.tensor(4);
    const at::Tensor wi_in = optional(g, 5), sa = scaled ? g.tensor(6) : at::Tensor(), sb_in = scaled ? g.tensor(7) : at::Tensor();
    Scratch ws(g, a, g.st->llmk_grouped_gemm_workspace_bytes(kind, scaled ? float_code(sa.scalar_type()) : 0, M, N, K));
    unlocked([&] {
        const at::Tensor seg = long_contiguous(seg_in), wi = long_contiguous(wi_in);
        const at::Tensor sb = scaled ? as_type(sb_in, sa.scalar_type()).contiguous() : sb_in;
        g.check(g.st->llmk_grouped_gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), kind, float_code(c.scalar_type()), (int)E, M, N, K, (const int64_t*)seg.data_ptr(),
                                        (const int64_t*)ptr_or_null(wi), ptr_or_null(sa), ptr_or_null(sb), scaled ? float_code(sa.scalar_type()) : 0, ws.get(), ws.bytes(), stream_of(a)),
                "llmk_grouped_gemm", PyExc_AssertionError);
    });
    Py_INCREF(g.v[2]);
    return g.v[2];
}

// grouped_gemm_swiglu_quant_fused(a, b, batch_size) -> bool
PyObject* swiglu_fused(const Args& g) {
    const at::Tensor &a = g.tensor(0), &b = g.tensor(1);
    const at::ScalarType t = b.scalar_type();
    if ((t != at::kChar && t != at::kFloat8_e4m3fn) || a.scalar_type() != t || b.dim() != 3) Py_RETURN_FALSE;
    return PyBool_FromLong(g.st->llmk_grouped_gemm_swiglu_quant_fused(operand_kind(t), (int)g.integer(2), a.size(0), b.size(1), b.size(2)));
}

// grouped_gemm_swiglu_quant(a, scale_a, b, scale_b, batch_size, seg_indptr, weight_indices, mid dtype code, act)
PyObject* swiglu_quant(const Args& g) {
    const at::Tensor &a = g.tensor(0), &sa_in = g.tensor(1), &b = g.tensor(2), &sb_in = g.tensor(3), &seg_in = g.tensor(5);
    g.on_gpu(a, b, sa_in, sb_in, seg_in);
    require(a.is_contiguous() && b.is_contiguous() && a.scalar_type() == b.scalar_type() && b.dim() == 3 && last_size(a) == last_size(b), "");
    const int kind = operand_kind(b.scalar_type());
    require(kind == LLMK_KIND_I8 || kind == LLMK_KIND_FP8, "quant_dtype must be torch.int8 or torch.float8_e4m3fn");
    const int64_t M = a.size(0), two_i = b.size(1), K = b.size(2), E = g.integer(4), mid = g.integer(7), act = g.integer(8);
    const at::Tensor wi_in = optional(g, 6);
    Scratch ws(g, a, sa_in.scalar_type() == at::kFloat ? 0 : M * (K / 128) * 4);
    QuantBuffers o;
    unlocked([&] {
        o = quant_buffers(M, two_i / 2, kind == LLMK_KIND_FP8, a);
        const at::Tensor sa = sa_in.contiguous(), sb = as_type(sb_in, sa.scalar_type()).contiguous();
        const at::Tensor seg = long_contiguous(seg_in), wi = long_contiguous(wi_in);
        g.check(g.st->llmk_grouped_gemm_swiglu_quant(a.data_ptr(), b.data_ptr(), o.q.data_ptr(), o.s.data_ptr(), kind, (int)mid, LLMK_ROUND_HALF_AWAY, (int)E, M, two_i, K,
                                                     (const int64_t*)seg.data_ptr(), (const int64_t*)ptr_or_null(wi), sa.data_ptr(), sb.data_ptr(), float_code(sa.scalar_type()),
                                                     (int)act, ws.get(), ws.bytes(), stream_of(a)), "llmk_grouped_gemm_swiglu_quant", PyExc_AssertionError);
    });
    return wrap_all(std::move(o.q), std::move(o.s));
}

// ------------------------------------------------------------------ module
// bind(library path, LlmkError, workspace dictionary)
PyObject* bind(PyObject* self, PyObject* args) {
    State* st = (State*)PyModule_GetState(self);
    const char* path;
    PyObject *error, *workspaces;
    if (!PyArg_ParseTuple(args, "sOO!", &path, &error, &PyDict_Type, &workspaces)) return nullptr;
    void* lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!lib) return PyErr_Format(PyExc_OSError, "%s", dlerror());
#define X(name)                                                             \
    st->name = (decltype(st->name))dlsym(lib, #name);                       \
    if (!st->name) {                                                        \
        st->llmk_last_error = nullptr;                                      \
        return PyErr_Format(PyExc_AttributeError, "%s: no %s", path, #name); \
    }
    LLMK_HOST_API(X)
#undef X
    Py_INCREF(error);
    Py_INCREF(workspaces);
    Py_XSETREF(st->error, error);
    Py_XSETREF(st->workspaces, workspaces);
    Py_RETURN_NONE;
}

template <PyObject* (*F)(const Args&), int N>
PyObject* call(PyObject* self, PyObject* const* args, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    try {
        return F(Args(self, args, n, N));
    } catch (const Raised& r) {
        if (r.type) PyErr_SetString(r.type, r.msg.c_str());
        return nullptr;
    }
    END_HANDLE_TH_ERRORS
}
#define FN(name, n) {#name, (PyCFunction)(void (*)())call<name, n>, METH_FASTCALL, nullptr}

PyMethodDef methods[] = {
    {"bind", bind, METH_VARARGS, nullptr},
    FN(act_quant, 3), FN(rowwise_quant, 1), FN(weight_quant, 3), FN(weight_dequant, 4), FN(w4a8_weight_quant, 2),
    FN(w4a8_weight_dequant, 6), FN(w4_quantize_nk, 2), FN(softmax_topk, 3), FN(fp8_gemm, 4), FN(int8_gemm, 4), FN(int8_gemm_per_token, 5), FN(w4a8_gemm, 7),
    FN(w4a16_gemm, 4), FN(marlin_mul, 4), FN(ep_preprocess, 2), FN(pre_reorder_quant, 9), FN(act_and_mul_quant, 8),
    FN(post_reorder, 9), FN(grouped_gemm, 8), FN(swiglu_fused, 3), FN(swiglu_quant, 9),
    {nullptr, nullptr, 0, nullptr}};

int traverse(PyObject* self, visitproc visit, void* arg) {
    State* st = (State*)PyModule_GetState(self);
    if (st) { Py_VISIT(st->error); Py_VISIT(st->workspaces); }
    return 0;
}
int clear(PyObject* self) {
    State* st = (State*)PyModule_GetState(self);
    if (st) { Py_CLEAR(st->error); Py_CLEAR(st->workspaces); }
    return 0;
}
// the torch this module's C++ interface is that of: the loader refuses another
int exec(PyObject* self) { return PyModule_AddStringConstant(self, "torch_version", LLMK_TORCH_VERSION); }
PyModuleDef_Slot slots[] = {{Py_mod_exec, (void*)exec}, {0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "llmk_host", nullptr, sizeof(State), methods, slots, traverse, clear, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_llmk_host(void) { return PyModuleDef_Init(&module); }
