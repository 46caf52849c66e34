// Host side of the Python binding: the calls a decoding program makes for every layer and token, from the
// Python arguments to the kernel launch in one native function.
//
// A batch-1 call costs 4 to 7 us on the GPU; checking six tensors, looking up buffers and passing sixteen
// arguments through ctypes costs two to three times that in Python, so single calls are bound by the
// host.  These functions do the same checks on the tensor objects directly.  They take the call only when
// everything is as the kernels need it and return None otherwise, launching nothing: the caller's Python code then
// takes the general route (other devices, released layers, large prompts) or words the error.
//
// Host-only translation unit (g++).  The library's C entry points come in as addresses (bind()), so it links
// against torch alone.
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <c10/core/InferenceMode.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>

#include <algorithm>
#include <array>
#include <cstdint>
#include <cstring>
#include <map>
#include <mutex>
#include <utility>
#include <vector>

#include "cherryq.h"

namespace {

using at::Tensor;

using VecquantFn = int (*)(const void *, const void *, const void *, const void *, const void *, void *, int, int, int, int,
                           int, int, void *, size_t, void *, size_t, void *);
using SizeFn = size_t (*)(int, int, int, int);
using PrepackedScratchFn = size_t (*)(int, int, int, int, int);
using MatvecPrepackedFn = int (*)(int, const void *, const void *, size_t, void *, int, int, int, int, int, void *);
using MatmulPrepackedFn = int (*)(int, const void *, const void *, size_t, void *, int, int, int, int, int, void *, size_t,
                                  void *);
using ShapeFn = int (*)(int, int, int, int, int, int);
using TakenFn = int (*)(int, int, int, int, int, int, void *);

struct Api {
    VecquantFn vecquant4, vecquant3, vecquant3_f32;
    SizeFn workspace, scratch, scratch_f32;
    PrepackedScratchFn prepacked_scratch;
    MatvecPrepackedFn matvec_prepacked;
    MatmulPrepackedFn matmul_prepacked;
    ShapeFn prepack_supported, rows_recommended;
} api;
TakenFn prompt_taken;  // cherryq_prompt_taken
using CapturingFn = int (*)(void *);
CapturingFn capturing;  // cherryq_stream_capturing

using FakeQuantFn = int (*)(int, const void *, const void *, void *, int, int, int, int, int, void *);
using GemmSizeFn = size_t (*)(int, int, int);
using GemmPreferredFn = int (*)(int, int, int, int, int);
using GemmFn = int (*)(int, int, int, const void *, const void *, void *, int, int, int, void *, size_t, void *, size_t, void *);
struct TrainApi {
    FakeQuantFn fake_quant_f16, fake_quant_bf16, fake_quant_f32;
    GemmSizeFn gemm_workspace, gemm_scratch;
    GemmPreferredFn gemm_preferred;
    GemmFn gemm;
} train;

// ---- buffers kept per (device, stream) -----------------------------------------------------------
// A zero-initialised workspace (the kernels leave it all zero after every call, so it is reusable as is)
// and an uninitialised scratch buffer for the batched paths.  Both grow on demand, at least doubling.  An
// outgrown buffer is kept alive rather than freed: a HIP graph captured earlier on that stream may still hold
// its address (doubling bounds what is kept to the size of the live buffer).
struct Pool {
    std::map<std::pair<int, uintptr_t>, Tensor> live;
    std::vector<Tensor> outgrown;
    std::mutex lock;
    bool zeroed;
    int64_t floor;

    Tensor get(int device, void *stream, int64_t bytes) {
        const std::pair<int, uintptr_t> key{device, reinterpret_cast<uintptr_t>(stream)};
        int64_t size = std::max(bytes, floor);
        {
            std::lock_guard<std::mutex> hold(lock);
            const Tensor &t = live[key];
            if (t.defined() && t.numel() >= bytes) return t;
            if (t.defined()) size = std::max(size, 2 * t.numel());
        }
        // Zeros that a graph writes are there only from its first replay on, so a call of another graph or outside would count from
        // whatever lies there: while the stream records, what is missing is made for the call alone (a warm stream has it).
        const bool own = zeroed && capturing && capturing(stream);
        if (own) size = std::max<int64_t>(bytes, 1);
        // Without the lock: callers come with and without the interpreter's, and an allocation may ask for that one (a record of
        // allocations with Python's stacks).  Who comes second drops what they made.
        Tensor made;
        {
            // plain tensors, whatever mode or function transform the first caller is in
            using K = c10::DispatchKey;
            c10::InferenceMode normal(false);
            c10::impl::ExcludeDispatchKeyGuard untouched(c10::DispatchKeySet({K::FuncTorchDynamicLayerFrontMode, K::FuncTorchDynamicLayerBackMode,
                                                                              K::FuncTorchVmapMode, K::Python, K::PythonTLSSnapshot}));
            const auto opts = at::TensorOptions().dtype(at::kByte).device(at::kCUDA, device);
            made = zeroed ? at::zeros({size}, opts) : at::empty({size}, opts);
        }
        if (own) return made;
        std::lock_guard<std::mutex> hold(lock);
        Tensor &t = live[key];
        if (!t.defined() || t.numel() < bytes) {
            if (t.defined()) outgrown.push_back(t);
            t = made;
        }
        return t;
    }
};
Pool &workspaces = *new Pool{{}, {}, {}, true, 1 << 18};  // never destroyed: the runtime may be gone by then
Pool &scratches = *new Pool{{}, {}, {}, false, 1};

inline const Tensor *tensor(PyObject *o) { return THPVariable_CheckExact(o) ? &THPVariable_Unpack(o) : nullptr; }

inline bool is(const Tensor *t, at::ScalarType type, int64_t dims, int device) {
    return t && t->scalar_type() == type && t->dim() == dims && t->is_cuda() && t->get_device() == device &&
           t->is_contiguous();
}

inline const void *ptr(const Tensor &t) { return t.numel() ? t.const_data_ptr() : nullptr; }
inline void *mut(const Tensor &t) { return t.numel() ? t.mutable_data_ptr() : nullptr; }

inline void *current_stream(int device) { return c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }

// From so many rows QuantLinear has a dense product to go to (llama/qlinear.py); the prompt kernel is taken where it is sure to answer.
constexpr int64_t kDenseRows = 512;

// Whether a call is only that: nothing records, replaces or transforms the operations, which a launch of ours is not among.
bool ordinary(const Tensor &x) {
    using K = c10::DispatchKey;
    return x.has_storage() && !at::tracer::impl::is_dispatch_enabled() && !c10::impl::TorchDispatchModeTLS::any_modes_set() &&
           !at::impl::torch_function_mode_enabled() &&
           !c10::impl::tls_local_dispatch_key_set().included_.has_any(
               c10::DispatchKeySet({K::FuncTorchDynamicLayerFrontMode, K::FuncTorchDynamicLayerBackMode, K::FuncTorchVmapMode}));
}

struct Packed {  // the checkpoint buffers of one layer
    const Tensor *qweight, *cherry_weight, *cherry_indices, *scales;
};

// The interpreter's lock is given up for a launch.  Another thread may replace a module's buffers meanwhile, so a call's
// tensors are held; what can throw (a tensor without memory has no address) is done before, and the lock comes back
// whichever way the scope is left.
template <typename... T>
struct Unlocked {
    std::array<Tensor, sizeof...(T)> held;
    PyThreadState *thread;
    explicit Unlocked(const T &...t) : held{t...}, thread(PyEval_SaveThread()) {}
    ~Unlocked() { PyEval_RestoreThread(thread); }
    Unlocked(const Unlocked &) = delete;
};

// The fused matmul over the checkpoint buffers; -1 where a buffer is not what the kernels take.
int fused(int kind, const Tensor &vec, int64_t batch, int64_t k, const Packed &p, const Tensor &out, int64_t group,
          bool accumulate) {
    const bool f32 = kind == 32;
    const int bits = kind == 4 ? 4 : 3, device = vec.get_device();
    const auto io = f32 ? at::kFloat : at::kHalf;
    if (!is(p.qweight, at::kByte, 2, device) || !is(p.cherry_weight, io, 2, device) ||
        !is(p.cherry_indices, f32 ? at::kInt : at::kShort, 1, device) || !is(p.scales, io, 2, device))
        return -1;
    const int64_t n = p.qweight->size(1), c = p.cherry_indices->size(0), kn = k - c;
    if (p.qweight->size(0) * 8 != kn * bits || p.cherry_weight->size(0) != c || p.cherry_weight->size(1) != n || group <= 0 ||
        (bits == 4 && group < 128) || p.scales->size(0) != (kn + group - 1) / group || p.scales->size(1) != n ||
        out.numel() != batch * n || batch <= 0)
        return -1;
    if (std::max({batch, k, n, group}) > INT32_MAX || c10::hip::current_device() != device) return -1;
    const int B = (int)batch, K = (int)k, N = (int)n, C = (int)c;
    void *stream = current_stream(device);
    const size_t wsb = api.workspace(B, K, N, C);
    const size_t scb = f32 ? api.scratch_f32(B, K, N, C) : B > 1 ? api.scratch(B, K, N, C) : 0;
    const Tensor ws = workspaces.get(device, stream, (int64_t)wsb);
    const Tensor sc = scb ? scratches.get(device, stream, (int64_t)scb) : Tensor();
    const VecquantFn fn = f32 ? api.vecquant3_f32 : bits == 4 ? api.vecquant4 : api.vecquant3;
    const void *x = ptr(vec), *w = ptr(*p.qweight), *cw = ptr(*p.cherry_weight), *ci = ptr(*p.cherry_indices), *scale = ptr(*p.scales);
    void *y = mut(out), *work = mut(ws), *extra = scb ? mut(sc) : nullptr;
    const size_t work_bytes = ws.numel(), extra_bytes = scb ? sc.numel() : 0;
    int rc;
    {
        const Unlocked launch(*p.qweight, *p.cherry_weight, *p.cherry_indices, *p.scales, vec, out);
        rc = fn(x, w, cw, ci, scale, y, B, K, N, C, (int)group, accumulate, work, work_bytes, extra, extra_bytes, stream);
    }
    return rc < 0 ? -1 : rc;  // a refusal of the library is worded by the general route
}

// 1 to 16 rows over a weight stream; -1 as above.
int over_stream(int bits, const Tensor &vec, int64_t batch, const Tensor &weights, const Tensor &out, int64_t k, int64_t n,
                int64_t c, bool accumulate) {
    const int device = vec.get_device();
    if (batch <= 0 || std::max({batch, k, n, c}) > INT32_MAX || c10::hip::current_device() != device) return -1;
    const int B = (int)batch, K = (int)k, N = (int)n, C = (int)c;
    void *stream = current_stream(device);
    Tensor sc;
    const size_t scb = B > 1 ? api.prepacked_scratch(bits, B, K, N, C) : 0;
    if (scb) sc = scratches.get(device, stream, (int64_t)scb);
    const void *x = ptr(vec), *w = ptr(weights);
    void *y = mut(out), *extra = scb ? mut(sc) : nullptr;
    const size_t bytes = weights.numel();
    int rc;
    {
        const Unlocked launch(weights, vec, out);
        rc = B == 1 ? api.matvec_prepacked(bits, x, w, bytes, y, B, K, N, C, accumulate, stream)
                    : api.matmul_prepacked(bits, x, w, bytes, y, B, K, N, C, accumulate, extra, scb, stream);
    }
    return rc < 0 ? -1 : rc;
}

PyObject *answer(int rc) {
    if (rc < 0) Py_RETURN_NONE;
    return PyLong_FromLong(rc);
}

// vecquant(kind, vec, qweight, cherry_weight, cherry_indices, scales, mul, group_size, accumulate): kind 4 and 3 are the
// fp16 operators of that many bits, 32 the 3-bit one over fp32 tensors.  0, a HIP error code, or None.
PyObject *vecquant(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 9 || !PyLong_CheckExact(a[7])) Py_RETURN_NONE;
    const int kind = (int)PyLong_AsLong(a[0]);
    const int64_t group = PyLong_AsLongLong(a[7]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const Tensor *vec = tensor(a[1]), *mul = tensor(a[6]);
    const auto io = kind == 32 ? at::kFloat : at::kHalf;
    if (!vec || !vec->is_cuda()) Py_RETURN_NONE;
    const int device = vec->get_device();
    if (!is(vec, io, 2, device) || !is(mul, io, 2, device) || mul->size(0) != vec->size(0)) Py_RETURN_NONE;
    const Packed p{tensor(a[2]), tensor(a[3]), tensor(a[4]), tensor(a[5])};
    const int accumulate = PyObject_IsTrue(a[8]);
    if (accumulate < 0) return nullptr;
    return answer(fused(kind, *vec, vec->size(0), vec->size(1), p, *mul, group, accumulate));
    END_HANDLE_TH_ERRORS
}

// matvec_prepacked(bits, vec, stream, out, in_features, num_cherries, accumulate)
PyObject *matvec_prepacked(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 7) Py_RETURN_NONE;
    for (int i : {0, 4, 5})
        if (!PyLong_CheckExact(a[i])) Py_RETURN_NONE;
    const int bits = (int)PyLong_AsLong(a[0]);
    const int64_t k = PyLong_AsLongLong(a[4]), c = PyLong_AsLongLong(a[5]);
    if (PyErr_Occurred()) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    const Tensor *vec = tensor(a[1]), *weights = tensor(a[2]), *out = tensor(a[3]);
    if (!vec || !vec->is_cuda()) Py_RETURN_NONE;
    const int device = vec->get_device();
    if (!is(vec, at::kHalf, 2, device) || !is(weights, at::kByte, 1, device) || !is(out, at::kHalf, 2, device) ||
        vec->size(1) != k || out->size(0) != vec->size(0))
        Py_RETURN_NONE;
    const int accumulate = PyObject_IsTrue(a[6]);
    if (accumulate < 0) return nullptr;
    return answer(over_stream(bits, *vec, vec->size(0), *weights, *out, k, out->size(1), c, accumulate));
    END_HANDLE_TH_ERRORS
}

// ---- QuantLinear.forward ----------------------------------------------------------------------------
struct Names {
    PyObject *dict, *buffers, *stream, *released, *dequantized, *layerwise, *prefill_rows, *w_bits, *group_size, *in_features,
        *out_features, *num_cherries, *qweight, *cherry_weight, *cherry_indices, *scales, *bias, *forward, *forward_hooks,
        *forward_pre_hooks;
} names;

// An integer entry of a module's dictionary (negative: none).
inline int64_t number(PyObject *dict, PyObject *name) {
    PyObject *v = PyDict_GetItemWithError(dict, name);
    return v && PyLong_CheckExact(v) ? PyLong_AsLongLong(v) : -1;
}

struct Ref {
    PyObject *o;
    ~Ref() { Py_XDECREF(o); }
};

// linear(module, x): the output, or None.  Everything is read from the module at every call (its dictionaries are
// plain lookups), so replaced buffers, a dropped stream or a changed mode need no notice.
PyObject *linear(PyObject *, PyObject *const *a, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 2) Py_RETURN_NONE;
    const Tensor *x = tensor(a[1]);
    if (!x || !x->is_cuda() || x->dim() < 1 || x->numel() == 0 || !x->is_floating_point()) Py_RETURN_NONE;
    Ref dict{PyObject_GetAttr(a[0], names.dict)};
    Ref layerwise{PyObject_GetAttr(a[0], names.layerwise)};
    if (!dict.o || !layerwise.o || !PyDict_CheckExact(dict.o)) {
        PyErr_Clear();
        Py_RETURN_NONE;
    }
    PyObject *buffers = PyDict_GetItemWithError(dict.o, names.buffers);
    const int bits = (int)number(dict.o, names.w_bits);
    const int64_t group = number(dict.o, names.group_size), k = number(dict.o, names.in_features),
                  n = number(dict.o, names.out_features), c = number(dict.o, names.num_cherries);
    if (layerwise.o != Py_True || PyDict_GetItemWithError(dict.o, names.dequantized) != Py_False || (bits != 3 && bits != 4) ||
        !buffers || !PyDict_Check(buffers) || group <= 0 || k <= 0 || n <= 0 || c < 0 || x->size(-1) != k ||
        std::max({group, k, n, c}) > INT32_MAX)
        Py_RETURN_NONE;
    const int64_t rows = x->numel() / k;
    const bool released = PyDict_GetItemWithError(dict.o, names.released) != Py_False;
    const int device = x->get_device();
    PyObject *so = PyDict_GetItemWithError(dict.o, names.stream);
    if (!so) Py_RETURN_NONE;
    const Tensor *weights = so != Py_None ? tensor(so) : nullptr;
    if (so != Py_None && !is(weights, at::kByte, 1, device)) Py_RETURN_NONE;
    bool streamed = false;
    // over the weight stream: one row, and the small batches that measured faster there than on the checkpoint
    // layout's kernels; with the checkpoint buffers released, everything its kernels take
    if (weights)
        streamed = rows == 1 || (rows <= 16 && (released ? api.prepack_supported : api.rows_recommended)(
                                                   bits, (int)rows, (int)k, (int)n, (int)c, (int)group));
    Packed p{};
    if (!streamed) {
        if (released) Py_RETURN_NONE;
        Ref limit{PyObject_GetAttr(a[0], names.prefill_rows)};
        const int64_t most = limit.o && PyLong_Check(limit.o) ? PyLong_AsLongLong(limit.o) : -1;
        if (PyErr_Occurred()) PyErr_Clear();
        if (rows >= most) Py_RETURN_NONE;  // dequantise once and a dense product
        if (rows >= kDenseRows && (!prompt_taken || !ordinary(*x) ||
                                   !prompt_taken(bits, (int)std::min<int64_t>(rows, INT32_MAX), (int)k, (int)n, (int)c, (int)group, current_stream(device))))
            Py_RETURN_NONE;
        auto buffer = [&](PyObject *name) {
            PyObject *o = PyDict_GetItemWithError(buffers, name);
            return o ? tensor(o) : nullptr;
        };
        p = Packed{buffer(names.qweight), buffer(names.cherry_weight), buffer(names.cherry_indices), buffer(names.scales)};
        if (!p.qweight || p.qweight->dim() != 2 || p.qweight->size(1) != n) Py_RETURN_NONE;
    }
    // The bias where attribute lookup finds it: the class, the module's own dictionary (None, or set by pack() where no
    // buffer was registered), its buffers.  One that lies elsewhere (a parameter, a property) is left to the general route.
    if (_PyType_Lookup(Py_TYPE(a[0]), names.bias)) Py_RETURN_NONE;
    PyObject *bo = PyDict_GetItemWithError(dict.o, names.bias);
    if (!bo) bo = PyDict_GetItemWithError(buffers, names.bias);
    if (!bo) Py_RETURN_NONE;
    const Tensor *bias = bo != Py_None ? tensor(bo) : nullptr;
    if (bo != Py_None && !bias) Py_RETURN_NONE;

    c10::InferenceMode inference(true);
    const Tensor row = x->scalar_type() == at::kHalf ? x->contiguous() : x->to(at::kHalf).contiguous();
    c10::SmallVector<int64_t, 6> sizes(x->sizes().begin(), x->sizes().end());
    sizes.back() = n;
    Tensor out = at::empty(sizes, row.options());
    const int rc = streamed ? over_stream(bits, row, rows, *weights, out, k, n, c, false)
                            : fused(bits, row, rows, k, p, out, group, false);
    if (rc != 0) Py_RETURN_NONE;
    if (x->scalar_type() != at::kHalf) out = out.to(x->scalar_type());
    if (bias) out.add_(*bias);
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// describe(address, rows, device, class, held, *modules): fills the cherryq_prefill_product at the address and appends the
// buffers it points to to the list `held`.  False where a module's own call would do anything but multiply `rows` rows
// by its checkpoint buffers with the prompt kernel: another class, hooks, a bias, another mode or shape.
PyObject *describe(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n < 6 || n > 8 || !PyList_CheckExact(a[4])) Py_RETURN_FALSE;
    auto *product = static_cast<cherryq_prefill_product *>(PyLong_AsVoidPtr(a[0]));
    const int64_t rows = PyLong_AsLongLong(a[1]);
    const int device = (int)PyLong_AsLong(a[2]);
    if (PyErr_Occurred()) return nullptr;
    if (!product) Py_RETURN_FALSE;
    product->n_layers = (int)(n - 5);
    for (Py_ssize_t i = 5; i < n; i++) {
        PyObject *m = a[i];
        if ((PyObject *)Py_TYPE(m) != a[3] || _PyType_Lookup(Py_TYPE(m), names.bias)) Py_RETURN_FALSE;
        Ref dict{PyObject_GetAttr(m, names.dict)}, layerwise{PyObject_GetAttr(m, names.layerwise)}, limit{PyObject_GetAttr(m, names.prefill_rows)};
        if (!dict.o || !layerwise.o || !limit.o || !PyDict_CheckExact(dict.o)) {
            PyErr_Clear();
            Py_RETURN_FALSE;
        }
        auto entry = [&](PyObject *name) { return PyDict_GetItemWithError(dict.o, name); };
        PyObject *buffers = entry(names.buffers), *hooks = entry(names.forward_hooks), *pre_hooks = entry(names.forward_pre_hooks);
        const int64_t bits = number(dict.o, names.w_bits), group = number(dict.o, names.group_size), k = number(dict.o, names.in_features),
                      columns = number(dict.o, names.out_features), c = number(dict.o, names.num_cherries),
                      most = PyLong_Check(limit.o) ? PyLong_AsLongLong(limit.o) : -1;
        if (PyErr_Occurred()) PyErr_Clear();
        if (entry(names.forward) || !buffers || !PyDict_Check(buffers) || !hooks || !PyDict_Check(hooks) || PyDict_GET_SIZE(hooks) ||
            !pre_hooks || !PyDict_Check(pre_hooks) || PyDict_GET_SIZE(pre_hooks) || layerwise.o != Py_True ||
            entry(names.dequantized) != Py_False || entry(names.released) != Py_False || rows >= most || (bits != 3 && bits != 4) ||
            group <= 0 || k <= 0 || columns <= 0 || c < 0 || c >= k || std::max({group, k, columns}) > INT32_MAX)
            Py_RETURN_FALSE;
        PyObject *bias = entry(names.bias);
        if (!bias) bias = PyDict_GetItemWithError(buffers, names.bias);
        if (bias != Py_None) Py_RETURN_FALSE;
        PyObject *const o[4] = {PyDict_GetItemWithError(buffers, names.qweight), PyDict_GetItemWithError(buffers, names.cherry_weight),
                                PyDict_GetItemWithError(buffers, names.cherry_indices), PyDict_GetItemWithError(buffers, names.scales)};
        const Tensor *t[4];
        for (int j = 0; j < 4; j++) t[j] = o[j] ? tensor(o[j]) : nullptr;
        if (!is(t[0], at::kByte, 2, device) || !is(t[1], at::kHalf, 2, device) || !is(t[2], at::kShort, 1, device) ||
            !is(t[3], at::kHalf, 2, device) || t[0]->size(0) * 8 != (k - c) * bits || t[0]->size(1) != columns || t[1]->size(0) != c ||
            t[1]->size(1) != columns || t[2]->size(0) != c || t[3]->size(0) != (k - c + group - 1) / group || t[3]->size(1) != columns)
            Py_RETURN_FALSE;
        if (i == 5) {
            product->w_bits = (int)bits, product->in_features = (int)k, product->num_cherries = (int)c, product->group_size = (int)group;
        } else if (product->w_bits != bits || product->in_features != k || product->num_cherries != c || product->group_size != group) {
            Py_RETURN_FALSE;
        }
        // what the entry point takes; other layers' own calls may go to a dense product
        auto misaligned = [](const Tensor &t, uintptr_t bytes) { return reinterpret_cast<uintptr_t>(ptr(t)) % bytes; };
        if (group % 32 || (bits == 4 && group < 128) || misaligned(*t[0], 16) || misaligned(*t[1], 16) || misaligned(*t[2], 4) || misaligned(*t[3], 16) ||
            (rows >= kDenseRows && (!prompt_taken || !prompt_taken((int)bits, (int)rows, (int)k, (int)columns, (int)c, (int)group, current_stream(device)))))
            Py_RETURN_FALSE;
        for (int j = 0; j < 4; j++)
            if (PyList_Append(a[4], o[j])) return nullptr;
        product->layers[i - 5] = {static_cast<const uint8_t *>(ptr(*t[0])), ptr(*t[1]), static_cast<const int16_t *>(ptr(*t[2])), ptr(*t[3]),
                                  nullptr, (int)columns};
    }
    Py_RETURN_TRUE;
    END_HANDLE_TH_ERRORS
}

// plain(tensor, device, *shape): whether a launch may read the tensor's memory as fp16 of this shape, in 16-byte pieces
PyObject *plain(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    const Tensor *t = n >= 2 ? tensor(a[0]) : nullptr;
    if (!t || !PyLong_Check(a[1]) || !is(t, at::kHalf, n - 2, (int)PyLong_AsLong(a[1])) || !t->has_storage()) Py_RETURN_FALSE;
    for (Py_ssize_t i = 2; i < n; i++) {
        const int64_t size = PyLong_AsLongLong(a[i]);
        if (size == -1 && PyErr_Occurred()) return nullptr;
        if (t->size(i - 2) != size) Py_RETURN_FALSE;
    }
    return PyBool_FromLong((reinterpret_cast<uintptr_t>(ptr(*t)) & 15) == 0);
    END_HANDLE_TH_ERRORS
}

// workspace(device, stream, bytes) / scratch(device, stream, bytes): the kept buffers, for the other callers
PyObject *kept(Pool &pool, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 3) {
        PyErr_SetString(PyExc_TypeError, "device, stream and bytes expected");
        return nullptr;
    }
    const int device = (int)PyLong_AsLong(a[0]);
    void *stream = reinterpret_cast<void *>(PyLong_AsUnsignedLongLong(a[1]));
    const int64_t bytes = PyLong_AsLongLong(a[2]);
    if (PyErr_Occurred()) return nullptr;
    return THPVariable_Wrap(pool.get(device, stream, bytes));
    END_HANDLE_TH_ERRORS
}
PyObject *workspace(PyObject *, PyObject *const *a, Py_ssize_t n) { return kept(workspaces, a, n); }
PyObject *scratch(PyObject *, PyObject *const *a, Py_ssize_t n) { return kept(scratches, a, n); }

// bind(addresses): the library's entry points in the order of struct Api
PyObject *bind(PyObject *, PyObject *seq) {
    constexpr Py_ssize_t count = sizeof(Api) / sizeof(void *);
    if (!PyTuple_Check(seq) || PyTuple_GET_SIZE(seq) != count) {
        PyErr_SetString(PyExc_TypeError, "one address per entry point expected");
        return nullptr;
    }
    void *at[count];
    for (Py_ssize_t i = 0; i < count; i++) {
        at[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(seq, i));
        if (!at[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
            return nullptr;
        }
    }
    memcpy(&api, at, sizeof(api));
    Py_RETURN_NONE;
}

// bind_prompt(address): cherryq_prompt_taken.  Without it no call of kDenseRows rows and more is taken.
PyObject *bind_prompt(PyObject *, PyObject *address) {
    prompt_taken = reinterpret_cast<TakenFn>(PyLong_AsVoidPtr(address));
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
}

// bind_capturing(address): cherryq_stream_capturing.  Without it no stream is taken to record a graph.
PyObject *bind_capturing(PyObject *, PyObject *address) {
    capturing = reinterpret_cast<CapturingFn>(PyLong_AsVoidPtr(address));
    if (PyErr_Occurred()) return nullptr;
    Py_RETURN_NONE;
}

// ---- the training layer ----------------------------------------------------------------------------
// A pass over a small layer is bound by the host: the fake quantisation's and the product's autograd nodes in Python, their checks, and
// torch's own linear took 180 us for a forward and a backward whose kernels take 30.

// Whether a launch may take the tensor's memory for its values, now: a gradient, or what a saved-tensor hook hands back, may be batched, a
// wrapper, sparse, lazily negated, zeros without memory or carry a tangent, and modes may have been entered since the forward pass.  Asked
// before the tensor's address, which some of these do not have.
bool plain_memory(const Tensor &t) {
    using K = c10::DispatchKey;
    return t.layout() == at::kStrided && ordinary(t) && !t.is_nested() &&
           !t.key_set().has_any(c10::DispatchKeySet({K::Negative, K::Conjugate, K::ZeroTensor, K::Python, K::Functionalize})) && !t._fw_grad(0).defined();
}

inline bool whole(const Tensor &t) { return t.is_contiguous() && reinterpret_cast<uintptr_t>(t.const_data_ptr()) % 16 == 0; }

// out[m, n] = sum_k a(m, k) b(n, k) of 16-bit matrices (an operand by_k lies as [k, n]) where the kernel takes it and is faster than
// torch's product; undefined elsewhere.  The result is laid out as `shape`.
Tensor product(const Tensor &a, bool a_by_k, const Tensor &b, bool b_by_k, int64_t m, int64_t n, int64_t k, at::IntArrayRef shape) {
    constexpr int64_t most = INT32_MAX;
    if ((a.scalar_type() != at::kHalf && a.scalar_type() != at::kBFloat16) || a.scalar_type() != b.scalar_type() || a.device() != b.device() ||
        !plain_memory(a) || !plain_memory(b) || m > most || n > most || k > most || a.numel() != m * k || b.numel() != n * k || !whole(a) || !whole(b))
        return {};
    const int device = a.get_device();
    if (c10::hip::current_device() != device || at::autocast::is_autocast_enabled(a.device().type()) ||
        !train.gemm_preferred(a_by_k, b_by_k, (int)m, (int)n, (int)k))
        return {};
    void *const stream = current_stream(device);
    const Tensor out = at::empty(shape, a.options());
    const int64_t zero_bytes = (int64_t)train.gemm_workspace((int)m, (int)n, (int)k), bytes = (int64_t)train.gemm_scratch((int)m, (int)n, (int)k);
    // the call's own, given back behind it in the stream's order: two streams never share it
    const Tensor scratch = bytes ? at::empty({bytes}, a.options().dtype(at::kByte)) : Tensor();
    // (so are a recorded call's tickets, zeroed in the graph: the stream's kept ones are other graphs' and other calls', too, and zeros that
    // were only recorded are not there yet when another graph is replayed first)
    const Tensor zero = !zero_bytes                       ? Tensor()
                        : capturing && capturing(stream) ? at::zeros({zero_bytes}, a.options().dtype(at::kByte))
                                                         : workspaces.get(device, stream, zero_bytes);
    const int rc = train.gemm(a.scalar_type() == at::kBFloat16, a_by_k, b_by_k, a.const_data_ptr(), b.const_data_ptr(), out.mutable_data_ptr(), (int)m, (int)n,
                              (int)k, bytes ? zero.mutable_data_ptr() : nullptr, bytes ? (size_t)zero.numel() : 0,
                              bytes ? scratch.mutable_data_ptr() : nullptr, (size_t)bytes, stream);
    TORCH_CHECK(rc == 0, "training product: status ", rc);
    return out;
}

// A gradient handed on as it is
struct StraightThrough : torch::autograd::Node {
    torch::autograd::variable_list apply(torch::autograd::variable_list &&grads) override { return {grads[0]}; }
};

// `quantised` with the gradient of the weight that it was made from, for second derivatives.  The node that runs holds where that leads since
// the forward pass; the weight itself may have been changed, replaced or given back.
Tensor of_the_weight(const Tensor &quantised) {
    const auto node = torch::autograd::get_current_node();
    TORCH_CHECK(node, "second derivatives of the training layer are taken by autograd's engine");
    const Tensor value = quantised.detach();
    const auto &edge = node->next_edge(1);
    if (edge.is_valid()) {
        const std::shared_ptr<StraightThrough> on(new StraightThrough(), torch::autograd::deleteNode);
        on->add_next_edge(edge);
        torch::autograd::impl::set_gradient_edge(value, {on, on->add_input_metadata(value)});
    }
    return value;
}

// linear(x, quantised) with the straight-through gradient for the weight that was quantised (llama/cherry_linear.py:97-98)
struct TrainLinear : torch::autograd::Function<TrainLinear> {
    static Tensor forward(torch::autograd::AutogradContext *ctx, const Tensor &x, const Tensor &weight, const Tensor &quantised) {
        // what a gradient reads and no more: the other may be changed in place or given back
        ctx->save_for_backward({weight.requires_grad() ? x : Tensor(), x.requires_grad() ? quantised : Tensor()});
        const int64_t n = weight.size(0), k = weight.size(1), rows = x.numel() / k;
        std::vector<int64_t> shape(x.sizes().begin(), x.sizes().end());
        shape.back() = n;
        Tensor out = product(x, false, quantised, false, rows, n, k, shape);
        return out.defined() ? out : at::linear(x, quantised);
    }
    static torch::autograd::variable_list backward(torch::autograd::AutogradContext *ctx, torch::autograd::variable_list grads) {
        const auto saved = ctx->get_saved_variables();
        const Tensor &g = grads[0], &x = saved[0];
        Tensor quantised = saved[1], dx, dw;
        const bool twice = at::GradMode::is_enabled();  // a graph of the gradients is asked for
        const int64_t n = g.size(-1);
        // (a call may ask for one of them: autograd.grad of the input alone, backward(inputs=...))
        if (quantised.defined() && ctx->needs_input_grad(0)) {
            const int64_t k = quantised.size(1);
            std::vector<int64_t> shape(g.sizes().begin(), g.sizes().end());
            shape.back() = k;
            if (twice) {
                quantised = of_the_weight(quantised);
            } else if (n) {
                dx = product(g, false, quantised, true, g.numel() / n, k, n, shape);
            }
            if (!dx.defined()) dx = g.matmul(quantised);
        }
        if (x.defined() && ctx->needs_input_grad(1)) {
            const int64_t k = x.size(-1), rows = g.numel() / std::max<int64_t>(n, 1);
            // (matrices as they are: a sparse one multiplies, but does not reshape)
            const Tensor g2 = g.dim() == 2 ? g : g.reshape({rows, n}), x2 = x.dim() == 2 ? x : x.reshape({rows, k});
            if (!twice && n) dw = product(g2, true, x2, true, n, k, rows, {n, k});
            if (!dw.defined()) dw = g2.t().matmul(x2);
        }
        return {dx, dw, Tensor()};
    }
};

// bind_train(addresses): as listed in TrainApi
PyObject *bind_train(PyObject *, PyObject *seq) {
    constexpr Py_ssize_t count = sizeof(train) / sizeof(void *);
    if (!PyTuple_Check(seq) || PyTuple_GET_SIZE(seq) != count) {
        PyErr_Format(PyExc_TypeError, "bind_train() takes a tuple of %zd addresses", count);
        return nullptr;
    }
    void *at[count];
    for (Py_ssize_t i = 0; i < count; i++) {
        at[i] = PyLong_AsVoidPtr(PyTuple_GET_ITEM(seq, i));
        if (!at[i]) {
            if (!PyErr_Occurred()) PyErr_SetString(PyExc_ValueError, "null address");
            return nullptr;
        }
    }
    memcpy(&train, at, sizeof(train));
    Py_RETURN_NONE;
}

// train_linear(x, weight, cherry_indices, w_bits, group_size): linear with the straight-through fake-quantised weight; None where a tensor or
// the moment is not ordinary, and nothing launched
PyObject *train_linear(PyObject *, PyObject *const *args, Py_ssize_t nargs) {
    HANDLE_TH_ERRORS
    if (nargs != 5) {
        PyErr_SetString(PyExc_TypeError, "train_linear() takes 5 arguments");
        return nullptr;
    }
    const Tensor *x = tensor(args[0]), *weight = tensor(args[1]), *t = weight, *indices = tensor(args[2]);
    if (!x || !weight || !indices || !PyLong_CheckExact(args[3]) || !PyLong_CheckExact(args[4]) || !train.gemm) Py_RETURN_NONE;
    const long bits = PyLong_AsLong(args[3]), group = PyLong_AsLong(args[4]);
    if (PyErr_Occurred()) return nullptr;
    if (!t->is_cuda() || !plain_memory(*x) || !plain_memory(*t) || !plain_memory(*indices) || t->dim() != 2 || !t->is_contiguous())
        Py_RETURN_NONE;
    const int device = t->get_device();
    const auto type = t->scalar_type();
    const FakeQuantFn quantise = type == at::kHalf ? train.fake_quant_f16 : type == at::kBFloat16 ? train.fake_quant_bf16 : type == at::kFloat ? train.fake_quant_f32 : nullptr;
    const int64_t n = t->size(0), k = t->size(1);
    if (!quantise || x->scalar_type() != type || x->device() != t->device() || x->dim() < 2 || x->size(-1) != k || !x->numel() || n <= 0 || n > INT32_MAX ||
        k > INT32_MAX || group > INT32_MAX || !is(indices, at::kInt, 1, device) || indices->numel() > INT32_MAX ||
        c10::hip::current_device() != device || at::autocast::is_autocast_enabled(t->device().type()))
        Py_RETURN_NONE;
    Tensor quantised, out;
    {
        at::NoGradGuard plain;
        quantised = at::empty({n, k}, t->options());
    }
    const int rc = quantise((int)bits, t->const_data_ptr(), ptr(*indices), quantised.mutable_data_ptr(), (int)k, (int)n, (int)indices->numel(),
                            group > 0 ? (int)group : (int)k, 1, current_stream(device));
    if (rc != 0) Py_RETURN_NONE;  // refused before the launch: the general route words it
    {
        Unlocked<Tensor, Tensor, Tensor> free(*x, *weight, quantised);
        out = TrainLinear::apply(free.held[0], free.held[1], free.held[2]);
    }
    return THPVariable_Wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// ordinary(tensor)
PyObject *is_ordinary(PyObject *, PyObject *x) {
    HANDLE_TH_ERRORS
    const Tensor *t = tensor(x);
    return PyBool_FromLong(t && ordinary(*t));
    END_HANDLE_TH_ERRORS
}

PyMethodDef methods[] = {
    {"bind", bind, METH_O, nullptr},
    {"bind_prompt", bind_prompt, METH_O, nullptr},
    {"bind_capturing", bind_capturing, METH_O, nullptr},
    {"bind_train", bind_train, METH_O, nullptr},
    {"train_linear", (PyCFunction)(void (*)())train_linear, METH_FASTCALL, nullptr},
    {"ordinary", is_ordinary, METH_O, nullptr},
    {"vecquant", (PyCFunction)(void (*)())vecquant, METH_FASTCALL, nullptr},
    {"matvec_prepacked", (PyCFunction)(void (*)())matvec_prepacked, METH_FASTCALL, nullptr},
    {"linear", (PyCFunction)(void (*)())linear, METH_FASTCALL, nullptr},
    {"describe", (PyCFunction)(void (*)())describe, METH_FASTCALL, nullptr},
    {"plain", (PyCFunction)(void (*)())plain, METH_FASTCALL, nullptr},
    {"workspace", (PyCFunction)(void (*)())workspace, METH_FASTCALL, nullptr},
    {"scratch", (PyCFunction)(void (*)())scratch, METH_FASTCALL, nullptr},
    {nullptr, nullptr, 0, nullptr}};

PyModuleDef module = {PyModuleDef_HEAD_INIT, "cherryq_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit_cherryq_host(void) {
    const std::pair<PyObject **, const char *> all[] = {{&names.dict, "__dict__"}, {&names.buffers, "_buffers"},
        {&names.stream, "_stream"}, {&names.released, "_released"}, {&names.dequantized, "dequantized"},
        {&names.layerwise, "_layerwise_dequantize"}, {&names.prefill_rows, "prefill_rows"}, {&names.w_bits, "w_bits"},
        {&names.group_size, "group_size"}, {&names.in_features, "in_features"}, {&names.out_features, "out_features"},
        {&names.num_cherries, "num_cherries"}, {&names.qweight, "qweight"}, {&names.cherry_weight, "cherry_weight"},
        {&names.cherry_indices, "cherry_indices"}, {&names.scales, "scales"}, {&names.bias, "bias"},
        {&names.forward, "forward"}, {&names.forward_hooks, "_forward_hooks"}, {&names.forward_pre_hooks, "_forward_pre_hooks"}};
    for (auto &n : all)
        if (!(*n.first = PyUnicode_InternFromString(n.second))) return nullptr;
    PyObject *m = PyModule_Create(&module);
    if (m && PyModule_AddStringConstant(m, "built_for", CHERRYQ_BUILT_FOR)) Py_CLEAR(m);
    return m;
}
