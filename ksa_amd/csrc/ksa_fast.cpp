// The calls of the package that a serving loop makes once per layer, from Python arguments to launch in native code.
//
// Behind each of them is a kernel of 5 to 10 us at the small end of its range.  Reading some thirty arguments off tensors in
// Python, handing them to ctypes and allocating through the Python bindings took longer than that.  Host time a call before and
// now: decode of two launches 18.2 / 8.5 us, pre-attention step 17.2 / 5.9, block index (four tensors) 12.9 / 7.4, prefill 12.7 /
// under the 9.5 us that its kernel takes at 300 tokens.  What is left is the launches, 3 us each, and 1 us a tensor.
//
// Every function here takes the plain case alone - tensors of the plain type with memory, on the current GPU, nobody tracing,
// recording, transforming or profiling, arguments within the documented ranges - and returns None for anything else, before it
// has allocated or launched: the Python function that called it then goes its general way, which holds every check and every
// error.  The library's entry points come as addresses from the Python side, which has loaded it.
#include <ATen/ATen.h>
#include <ATen/core/grad_mode.h>
#include <ATen/PythonTorchFunctionTLS.h>
#include <c10/core/impl/LocalDispatchKeySet.h>
#include <c10/core/impl/TorchDispatchModeTLS.h>
#include <c10/hip/HIPFunctions.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/jit/frontend/tracer.h>
#include <torch/csrc/profiler/api.h>

#include <array>
#include <cmath>
#include <cstdint>

#include "ksa_hip.h"

namespace {

struct Library {
    decltype(&ksa_block_index) block_index;
    decltype(&ksa_decode_splits) decode_splits;
    decltype(&ksa_decode_workspace_bytes) decode_workspace_bytes;
    decltype(&ksa_decode_fwd) decode_fwd;
    decltype(&ksa_prefill_chunks_fwd) prefill_chunks_fwd;
    decltype(&ksa_pre_attention) pre_attention;
    decltype(&ksa_decode_wide_splits) decode_wide_splits;
    decltype(&ksa_decode_wide_fwd) decode_wide_fwd;
} lib{};
PyObject* lib_check = nullptr;  // `_lib.check`, which raises

// Whether a library call has launched.  If not, it was refused in front of its launch, and the general way says why; but
// an error behind a launch is raised here (an exception is set): the kernel may have run, on outputs that may be inputs.
bool launched(int rc, const char* what) {
    if (rc == KSA_ERR_LAUNCH) {
        PyObject* r = PyObject_CallFunction(lib_check, "is", rc, what);
        Py_XDECREF(r);
        if (r) PyErr_SetString(PyExc_RuntimeError, what);
    }
    return rc == KSA_OK;
}
#define KSA_UNLESS_LAUNCHED(rc, what)           \
    if (!launched(rc, what)) {                  \
        if (PyErr_Occurred()) return nullptr;   \
        Py_RETURN_NONE;                         \
    }

// Nobody records, traces, transforms or profiles (`_lib.direct`, which says why for each).  Whoever steps in front of the
// dispatcher (a mode, a torch.func transform, a tracer) includes a key of its own in this thread.
bool quiet() {
    static const c10::DispatchKeySet usual({c10::DispatchKey::BackendSelect, c10::DispatchKey::ADInplaceOrView});
    const auto keys = c10::impl::tls_local_dispatch_key_set().included_;
    return (keys & usual) == keys && c10::impl::TorchDispatchModeTLS::stack_len() == 0 && at::impl::PythonTorchFunctionTLS::stack_len() == 0 &&
           !torch::jit::tracer::isTracing() &&
           !torch::profiler::impl::profilerEnabled();
}

// A tensor with memory of its own on the GPU and nothing between it and its values: no wrapper, lazy, negative or
// functional tensor has this key set.  `param`: an nn.Parameter will do (what the kernels only read, where the general way
// does not look at requires_grad either).
const at::Tensor* plain(PyObject* o, bool param = false) {
    if (Py_TYPE(o) != reinterpret_cast<PyTypeObject*>(THPVariableClass) &&
        !(param && Py_TYPE(o) == reinterpret_cast<PyTypeObject*>(ParameterClass)))
        return nullptr;
    static const c10::DispatchKeySet allowed({c10::DispatchKey::CUDA, c10::DispatchKey::AutogradCUDA,
                                              c10::DispatchKey::ADInplaceOrView, c10::DispatchKey::AutocastCUDA});
    const at::Tensor& t = THPVariable_Unpack(o);
    const auto keys = t.key_set();
    if ((keys & allowed) != keys || !keys.has(c10::DispatchKey::CUDA) || !t.has_storage() || t.const_data_ptr() == nullptr ||
        t._fw_grad(0).defined() || (!param && t.requires_grad() && at::GradMode::is_enabled()))
        return nullptr;
    return &t;
}

int dtype_of(const at::Tensor& t) {
    const auto s = t.scalar_type();
    return s == at::kBFloat16 ? 0 : s == at::kHalf ? 1 : -1;
}

// an int of Python's own type that fits 32 bits
bool get_int(PyObject* o, int& v) {
    if (!PyLong_CheckExact(o)) return false;
    int over = 0;
    const long l = PyLong_AsLongAndOverflow(o, &over);
    if (over || l < INT32_MIN || l > INT32_MAX) return false;
    v = (int)l;
    return true;
}

// a positive scale, given or that of the head dimension
bool get_scale(PyObject* o, int64_t D, float& v) {
    const double s = o == Py_None ? std::pow((double)D, -0.5) : PyFloat_CheckExact(o) ? PyFloat_AS_DOUBLE(o) : -1.0;
    v = (float)s;
    return s > 0 && std::isfinite(s);
}

bool kernel_dim(int64_t D) { return D == 64 || D == 128 || D == 256; }
bool fits(const at::Tensor& t) {
    for (const auto s : t.sizes())
        if (s <= 0 || s > INT32_MAX) return false;
    return true;
}
// 16-byte items: what the library would refuse, behind the allocations
bool aligned(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool aligned(const at::Tensor& t) {
    const auto s = t.strides();
    return aligned(t.const_data_ptr()) && ((s[0] | s[1] | s[2]) & 7) == 0;
}
using Strides = std::array<int64_t, 3>;
Strides first3(const at::Tensor& t) { return {t.stride(0), t.stride(1), t.stride(2)}; }

struct Unlocked {  // other threads may run: an allocation can wait for the device
    PyThreadState* s = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(s); }
};
void* stream_of(int device) { return (void*)c10::hip::getCurrentHIPStream((c10::DeviceIndex)device).stream(); }
at::Tensor bytes(size_t n, const at::Tensor& like) { return at::empty({(int64_t)n}, like.options().dtype(at::kByte)); }

// decode(q, kcache, vcache, start, end, scale, nsplit)
PyObject* decode(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 7 || !quiet()) Py_RETURN_NONE;
    const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
    if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || k->sizes() != v->sizes() || !fits(*q) || !fits(*k)) Py_RETURN_NONE;
    const int dt = dtype_of(*q), dev = q->get_device();
    const int64_t b = q->size(0), Hq = q->size(1), Q = q->size(2), D = q->size(3), Hkv = k->size(1), rows = k->size(2);
    if (dt < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() || k->get_device() != dev ||
        v->get_device() != dev || dev != c10::hip::current_device() || k->size(0) != b || k->size(3) != D || Hq % Hkv != 0 ||
        !kernel_dim(D) || q->stride(3) != 1 || k->stride(3) != 1 || v->stride(3) != 1 || !aligned(*q) || !aligned(*k) || !aligned(*v))
        Py_RETURN_NONE;
    const int32_t *start = nullptr, *end = nullptr;
    int s0 = 0, e0 = (int)rows, most = (int)rows;
    const bool t0 = THPVariable_Check(a[3]), t1 = THPVariable_Check(a[4]);
    if (t0 || t1) {
        if (!t0 || !t1) Py_RETURN_NONE;
        for (int i = 0; i < 2; ++i) {
            const at::Tensor* t = plain(a[3 + i]);
            if (!t || t->scalar_type() != at::kInt || t->get_device() != dev || t->dim() != 1 || t->size(0) != b || t->stride(0) != 1)
                Py_RETURN_NONE;
            (i ? end : start) = static_cast<const int32_t*>(t->const_data_ptr());
        }
    } else {
        if ((a[3] != Py_None && !get_int(a[3], s0)) || (a[4] != Py_None && !get_int(a[4], e0))) Py_RETURN_NONE;
        if (s0 < 0 || s0 >= e0 || e0 > rows) Py_RETURN_NONE;
        most = e0 - s0;
    }
    float scale;
    int nsplit = 0;
    if (!get_scale(a[5], D, scale) || (a[6] != Py_None && (!get_int(a[6], nsplit) || nsplit < 1))) Py_RETURN_NONE;
    at::Tensor out;
    int rc;
    bool wide = false;
    {
        Unlocked u;
        if (a[6] == Py_None) {
            nsplit = lib.decode_wide_splits((int)b, (int)Hq, (int)Hkv, (int)Q, (int)D, most);
            wide = nsplit > 0;
            if (!wide) nsplit = lib.decode_splits((int)b, (int)Hq, (int)Hkv, (int)Q, (int)D, most);
        }
        const auto forward = wide ? lib.decode_wide_fwd : lib.decode_fwd;
        out = at::empty({b, Q, Hq, D}, q->options());
        at::Tensor ws;
        size_t ws_bytes = 0;
        if (nsplit > 1) {
            ws_bytes = lib.decode_workspace_bytes((int)b, (int)Hq, (int)Hkv, (int)Q, (int)D, nsplit);
            ws = bytes(ws_bytes, *q);
        }
        const Strides qs = first3(*q), ks = first3(*k), vs = first3(*v), os = first3(out);
        rc = forward(q->const_data_ptr(), k->const_data_ptr(), v->const_data_ptr(), out.mutable_data_ptr(), start, end, s0, e0,
                     (int)b, (int)Hq, (int)Hkv, (int)Q, (int)D, dt, qs.data(), ks.data(), vs.data(), os.data(), scale, nsplit,
                     ws_bytes ? ws.mutable_data_ptr() : nullptr, ws_bytes, stream_of(dev));
    }
    KSA_UNLESS_LAUNCHED(rc, wide ? "ksa_decode_wide_fwd" : "ksa_decode_fwd")
    return THPVariable_Wrap(out);
    END_HANDLE_TH_ERRORS
}

// `_chunk_tiles` of prefill.py for summary rows in line, and its `_QUEUE_ROWS`: written twice because compiled programs trace through
// the Python ones; tests/test_host.py holds them together
bool chunk_tiles(int64_t Sq, int64_t D, int64_t C, int64_t S) {
    return C > 0 && C <= 512 && C % 128 == 0 && S > 0 && (8 % S == 0 || (S == 16 && D <= 128)) && Sq >= 64 && Sq < 1 << 29 &&
           Sq % (C + S) <= C;
}
constexpr int64_t kQueueRows = 1 << 19;

// layout_rules(Sq, D, C, S) -> (whether chunk tiles take it, kQueueRows)
PyObject* layout_rules(PyObject*, PyObject* const* a, Py_ssize_t n) {
    int v[4];
    for (int i = 0; i < 4; ++i)
        if (n != 4 || !get_int(a[i], v[i])) return PyErr_Format(PyExc_TypeError, "layout_rules takes four ints");
    return Py_BuildValue("Oi", chunk_tiles(v[0], v[1], v[2], v[3]) ? Py_True : Py_False, (int)kQueueRows);
}

// prefill(q, k, v, C, S, W, skip_old_summary, scale, return_lse, summary_pos, analyse): chunk tiles only.
// analyse(summary_pos, Sq, C, S) -> (prefix rows, whether they lie in line, ...)
PyObject* prefill(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 11 || !quiet()) Py_RETURN_NONE;
    const at::Tensor *q = plain(a[0]), *k = plain(a[1]), *v = plain(a[2]);
    if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || k->sizes() != v->sizes() || !fits(*q) || !fits(*k)) Py_RETURN_NONE;
    const int dt = dtype_of(*q), dev = q->get_device();
    const int64_t b = q->size(0), Sq = q->size(1), Hq = q->size(2), D = q->size(3), Hkv = k->size(2);
    if (dt < 0 || k->scalar_type() != q->scalar_type() || v->scalar_type() != q->scalar_type() || k->get_device() != dev ||
        v->get_device() != dev || dev != c10::hip::current_device() || k->size(0) != b || k->size(1) != Sq || k->size(3) != D ||
        Hq % Hkv != 0 || !kernel_dim(D) || q->stride(3) != 1 || k->stride(3) != 1 || k->strides() != v->strides() ||
        !aligned(*q) || !aligned(*k) || !aligned(*v) || Sq * k->stride(1) * 2 >= 1ll << 32)
        Py_RETURN_NONE;
    int C, S, W;
    float scale;
    if (!get_int(a[3], C) || !get_int(a[4], S) || !get_int(a[5], W) || !PyBool_Check(a[6]) || !get_scale(a[7], D, scale) ||
        !PyBool_Check(a[8]))
        Py_RETURN_NONE;
    if (!chunk_tiles(Sq, D, C, S) || W < 0) Py_RETURN_NONE;
    if (a[9] != Py_None) {
        if (!plain(a[9])) Py_RETURN_NONE;
        PyObject* r = PyObject_CallFunction(a[10], "OLii", a[9], (long long)Sq, C, S);
        if (!r) return nullptr;
        const bool tuple = PyTuple_Check(r) && PyTuple_GET_SIZE(r) >= 2;
        const long long P = tuple ? PyLong_AsLongLong(PyTuple_GET_ITEM(r, 0)) : -1;
        const bool in_line = tuple && PyTuple_GET_ITEM(r, 1) == Py_True;
        Py_DECREF(r);
        if (PyErr_Occurred()) return nullptr;
        if (!in_line || (P != 0 && P != Sq / (C + S) * S)) Py_RETURN_NONE;
    }
    at::Tensor out, lse;
    int rc;
    {
        Unlocked u;
        out = at::empty_like(*q);
        if (a[8] == Py_True) lse = at::empty({b, Hq, Sq}, q->options().dtype(at::kFloat));
        at::Tensor sched;  // as in `_launch_chunks`
        if (b * Hq * Sq >= kQueueRows) sched = at::empty({8}, q->options().dtype(at::kInt));
        const Strides qs = first3(*q), ks = first3(*k), os = first3(out);
        rc = lib.prefill_chunks_fwd(q->const_data_ptr(), k->const_data_ptr(), v->const_data_ptr(), out.mutable_data_ptr(),
                                    lse.defined() ? lse.mutable_data_ptr<float>() : nullptr, (int)b, (int)Sq, (int)Hq, (int)Hkv,
                                    (int)D, dt, qs.data(), ks.data(), os.data(), C, S, W, a[6] == Py_True, scale, 0,
                                    sched.defined() ? sched.mutable_data_ptr<int32_t>() : nullptr, stream_of(dev));
    }
    KSA_UNLESS_LAUNCHED(rc, "ksa_prefill_chunks_fwd")
    PyObject* o = THPVariable_Wrap(out);
    PyObject* l = lse.defined() ? THPVariable_Wrap(lse) : Py_NewRef(Py_None);
    PyObject* r = o && l ? PyTuple_Pack(2, o, l) : nullptr;
    Py_XDECREF(o);
    Py_XDECREF(l);
    return r;
    END_HANDLE_TH_ERRORS
}

// pre_attention(q, k, v, q_norm_weight, k_norm_weight, cos, sin, eps, q_out, k_out, v_out, kv_out_row)
PyObject* pre_attention(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    if (n != 12 || !quiet() || !PyFloat_CheckExact(a[7])) Py_RETURN_NONE;
    const at::Tensor *q = plain(a[0], true), *k = plain(a[1], true), *v = plain(a[2], true);
    if (!q || !k || !v || q->dim() != 4 || k->dim() != 4 || k->sizes() != v->sizes() || !fits(*q) || !fits(*k)) Py_RETURN_NONE;
    const int dt = dtype_of(*q), dev = q->get_device();
    const int64_t b = q->size(0), S = q->size(1), Hq = q->size(2), D = q->size(3), Hkv = k->size(2);
    auto same = [&](const at::Tensor* t) { return t && t->scalar_type() == q->scalar_type() && t->get_device() == dev; };
    auto rows = [](const at::Tensor& t) { return aligned(t) && t.stride(2) >= 0 && t.stride(2) * 8 + 128 < 1ll << 32; };
    if (dt < 0 || !same(k) || !same(v) || dev != c10::hip::current_device() || k->size(0) != b || k->size(1) != S ||
        k->size(3) != D || (D != 64 && D != 128) || b * S >= (1ll << 31) - 64 || q->stride(3) != 1 || k->stride(3) != 1 ||
        v->stride(3) != 1 || !rows(*q) || !rows(*k) || !rows(*v) || !(PyFloat_AS_DOUBLE(a[7]) >= 0))
        Py_RETURN_NONE;
    const at::Tensor* w[2];
    const at::Tensor* rope[2];
    for (int i = 0; i < 2; ++i) {
        w[i] = plain(a[3 + i], true);
        rope[i] = plain(a[5 + i], true);
        if (!same(w[i]) || w[i]->dim() != 1 || w[i]->size(0) != D || !w[i]->is_contiguous() || !aligned(w[i]->const_data_ptr()))
            Py_RETURN_NONE;
        if (!same(rope[i]) || rope[i]->dim() != 3 || (rope[i]->size(0) != 1 && rope[i]->size(0) != b) || rope[i]->size(1) != S ||
            rope[i]->size(2) != D || !rope[i]->is_contiguous() || !aligned(rope[i]->const_data_ptr()))
            Py_RETURN_NONE;
    }
    if (rope[0]->size(0) != rope[1]->size(0)) Py_RETURN_NONE;
    const at::Tensor* given[3];
    const at::Tensor* like[3] = {q, k, v};
    for (int i = 0; i < 3; ++i) {
        given[i] = a[8 + i] == Py_None ? nullptr : plain(a[8 + i], true);
        if (a[8 + i] != Py_None &&
            (!same(given[i]) || given[i]->sizes() != like[i]->sizes() || given[i]->stride(3) != 1 || !rows(*given[i])))
            Py_RETURN_NONE;
    }
    const int32_t* kv_row = nullptr;
    int per_token = 0;
    if (a[11] != Py_None) {
        const at::Tensor* r = plain(a[11]);
        if (!r || r->scalar_type() != at::kInt || r->get_device() != dev || !r->is_contiguous() || !given[1] || !given[2] ||
            !((r->dim() == 1 && r->size(0) == b) || (r->dim() == 2 && r->size(0) == b && r->size(1) == S)))
            Py_RETURN_NONE;
        kv_row = static_cast<const int32_t*>(r->const_data_ptr());
        per_token = r->dim() == 2;
    }
    at::Tensor o[3];
    int rc;
    {
        Unlocked u;
        for (int i = 0; i < 3; ++i) o[i] = given[i] ? *given[i] : at::empty(like[i]->sizes(), like[i]->options());
        const Strides qs = first3(*q), ks = first3(*k), vs = first3(*v), qo = first3(o[0]), ko = first3(o[1]), vo = first3(o[2]);
        const Strides cs = {rope[0]->size(0) > 1 ? rope[0]->stride(0) : 0, rope[0]->stride(1), 0};
        // (unsafe access: the outputs may be views that the caller's program counts versions of, as on the general way)
        auto out = [&](int i) { return const_cast<void*>(o[i].const_data_ptr()); };
        rc = lib.pre_attention(q->const_data_ptr(), k->const_data_ptr(), v->const_data_ptr(), w[0]->const_data_ptr(),
                               w[1]->const_data_ptr(), rope[0]->const_data_ptr(), rope[1]->const_data_ptr(), out(0), out(1), out(2),
                               (int)b, (int)S, (int)Hq, (int)Hkv, (int)D, dt, qs.data(), ks.data(), vs.data(), qo.data(),
                               ko.data(), vo.data(), cs.data(), kv_row, per_token, (float)PyFloat_AS_DOUBLE(a[7]), stream_of(dev));
    }
    KSA_UNLESS_LAUNCHED(rc, "ksa_pre_attention")
    PyObject* r = PyTuple_New(3);
    for (int i = 0; r && i < 3; ++i) {
        PyObject* t = given[i] ? Py_NewRef(a[8 + i]) : THPVariable_Wrap(o[i]);
        if (!t) Py_CLEAR(r);
        else PyTuple_SET_ITEM(r, i, t);
    }
    return r;
    END_HANDLE_TH_ERRORS
}

// block_index(Sq, Sk, C, S, W, skip_old_summary, tile_m, tile_n) on the current GPU, which the caller has made ready
PyObject* block_index(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    int Sq, Sk, C, S, W, tm, tn;
    if (n != 8 || !quiet() || !get_int(a[0], Sq) || !get_int(a[1], Sk) || !get_int(a[2], C) || !get_int(a[3], S) ||
        !get_int(a[4], W) || !PyBool_Check(a[5]) || !get_int(a[6], tm) || !get_int(a[7], tn) || Sq <= 0 || Sk < Sq || tm <= 0 ||
        tn <= 0 || C <= 0 || S <= 0 || W < 0)
        Py_RETURN_NONE;
    const int64_t M = ((int64_t)Sq + tm - 1) / tm, N = ((int64_t)Sk + tn - 1) / tn;
    const int dev = c10::hip::current_device();
    at::Tensor t[4];
    int rc;
    {
        Unlocked u;
        const auto opt = at::TensorOptions().dtype(at::kInt).device(at::kCUDA, (c10::DeviceIndex)dev);
        for (int i = 0; i < 4; ++i) t[i] = i & 1 ? at::empty({1, 1, M, N}, opt) : at::empty({1, 1, M}, opt);
        int32_t* p[4];
        for (int i = 0; i < 4; ++i) p[i] = t[i].mutable_data_ptr<int32_t>();
        rc = lib.block_index(Sq, Sk, C, S, W, Sk - Sq, a[5] == Py_True, tm, tn, p[0], p[1], p[2], p[3], stream_of(dev));
    }
    KSA_UNLESS_LAUNCHED(rc, "ksa_block_index")
    PyObject* r = PyTuple_New(4);
    for (int i = 0; r && i < 4; ++i) {
        PyObject* o = THPVariable_Wrap(t[i]);
        if (!o) Py_CLEAR(r);
        else PyTuple_SET_ITEM(r, i, o);
    }
    return r;
    END_HANDLE_TH_ERRORS
}

// bind(_lib.check, addresses of ksa_block_index, ksa_decode_splits, ksa_decode_workspace_bytes, ksa_decode_fwd, ksa_prefill_chunks_fwd,
// ksa_pre_attention, ksa_decode_wide_splits, ksa_decode_wide_fwd)
PyObject* bind(PyObject*, PyObject* const* a, Py_ssize_t n) {
    void** slots[] = {(void**)&lib.block_index, (void**)&lib.decode_splits, (void**)&lib.decode_workspace_bytes,
                      (void**)&lib.decode_fwd, (void**)&lib.prefill_chunks_fwd, (void**)&lib.pre_attention,
                      (void**)&lib.decode_wide_splits, (void**)&lib.decode_wide_fwd};
    constexpr Py_ssize_t kSlots = sizeof(slots) / sizeof(slots[0]);
    if (n != 1 + kSlots) return PyErr_Format(PyExc_TypeError, "bind takes a function and %zd addresses", kSlots);
    Py_INCREF(a[0]);
    Py_XSETREF(lib_check, a[0]);
    for (Py_ssize_t i = 0; i < kSlots; ++i) {
        *slots[i] = PyLong_AsVoidPtr(a[1 + i]);
        if (PyErr_Occurred()) return nullptr;
    }
    Py_RETURN_NONE;
}

PyMethodDef methods[] = {
#define KSA_METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(name)), METH_FASTCALL, nullptr}
    KSA_METHOD(bind), KSA_METHOD(decode), KSA_METHOD(prefill), KSA_METHOD(pre_attention), KSA_METHOD(block_index),
    KSA_METHOD(layout_rules),
#undef KSA_METHOD
    {nullptr, nullptr, 0, nullptr}};
PyModuleDef module_def = {PyModuleDef_HEAD_INIT, "_fast", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__fast() { return PyModule_Create(&module_def); }
