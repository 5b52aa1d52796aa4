// CPython binding of the entry points a host calls once per layer and block.
//
// Such a call enqueues a kernel of about five microseconds, so everything around the launch counts.  Written in
// Python over ctypes (argument checks, contiguity, fresh outputs, the stream query, the conversion of some twenty
// arguments) it took longer than the kernel: 13 us for a GatedDelta forward, 26 us for a whole layer, 15 us for the
// attention.  Here the same steps run on the C++ tensor interface: the checks are field reads, outputs come from the
// caching allocator without going through the dispatcher, and the stream is a thread-local read.
//
// The argument meaning, the checks, their order and the exceptions are those of the methods in dflash_kernels.py that
// call this module; the C ABI stays the only way to the kernels.  The interpreter lock is released around the library
// call, as ctypes does.

#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <ATen/EmptyTensor.h>
#include <ATen/hip/EmptyTensor.h>
#include <c10/hip/HIPGraphsC10Utils.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/object_ptr.h>

#include <chrono>
#include <initializer_list>
#include <map>
#include <mutex>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/dflash_cache.h"
#include "../../include/dflash_hip.h"

namespace {

PyObject* g_error = nullptr;          // DFlashError, DFlashUnsupported: handed over by _lib.py
PyObject* g_unsupported = nullptr;

typedef c10::MaybeOwned<at::Tensor> Held;

[[noreturn]] void raise(PyObject* type, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    PyErr_FormatV(type ? type : PyExc_RuntimeError, fmt, ap);
    va_end(ap);
    throw python_error();
}

void need_args(Py_ssize_t got, Py_ssize_t want, const char* fn) {
    if (got != want) raise(PyExc_TypeError, "%s: %zd arguments expected, %zd given", fn, want, got);
}

const at::Tensor& tensor(PyObject* o, const char* what) {
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, "%s must be a tensor, not %.100s", what, Py_TYPE(o)->tp_name);
    const at::Tensor& t = THPVariable_Unpack(o);
    if (!t.is_cuda()) raise(g_error, "DFlash kernels run on the GPU only: got a CPU tensor (there is no CPU path)");
    return t;
}
// None -> an undefined tensor
const at::Tensor& tensor_or_none(PyObject* o, const char* what) {
    static const at::Tensor none;
    return o == Py_None ? none : tensor(o, what);
}
int64_t integer(PyObject* o) {
    const int64_t v = PyLong_AsLongLong(o);
    if (v == -1 && PyErr_Occurred()) {
        PyErr_Clear();
        PyObject* i = PyNumber_Index(o);
        if (!i) throw python_error();
        const int64_t w = PyLong_AsLongLong(i);
        Py_DECREF(i);
        if (w == -1 && PyErr_Occurred()) throw python_error();
        return w;
    }
    return v;
}
float number(PyObject* o) {
    const double v = PyFloat_AsDouble(o);
    if (v == -1.0 && PyErr_Occurred()) throw python_error();
    return (float)v;
}
bool truth(PyObject* o) {
    const int v = PyObject_IsTrue(o);
    if (v < 0) throw python_error();
    return v != 0;
}

int code_or(at::ScalarType t, int none) {
    switch (t) {
        case at::kFloat: return DFLASH_F32;
        case at::kBFloat16: return DFLASH_BF16;
        case at::kHalf: return DFLASH_F16;
        case at::kByte:
        case at::kBool: return DFLASH_U8;
        default: return none;
    }
}
int code(const at::Tensor& t) {
    const int c = code_or(t.scalar_type(), -1);
    if (c < 0) raise(g_unsupported, "dtype torch.%s is not supported", c10::toString(t.scalar_type()));
    return c;
}

void* ptr(const at::Tensor& t) { return t.defined() ? t.data_ptr() : nullptr; }
Held held(const at::Tensor& t) { return t.expect_contiguous(); }
Held held_or_none(const at::Tensor& t) { return t.defined() ? t.expect_contiguous() : Held::borrowed(t); }
// contiguous and of the given type
Held held_as(const at::Tensor& t, at::ScalarType st) {
    if (!t.defined() || (t.scalar_type() == st && t.is_contiguous())) return Held::borrowed(t);
    return Held::owned(t.to(st).contiguous());
}

at::Tensor fresh(at::IntArrayRef size, at::ScalarType st, const at::Tensor& like) {
    return at::Tensor(at::detail::empty_cuda(size, st, like.device(), std::nullopt));
}

// The outputs of one call that a program lets go of together, small ones out of one allocation: a tensor costs the host 0.6 us from the
// allocator and back, of a call that enqueues in 3 (a layer of nine outputs 9.4 us, now 8.0; a forward 5.7, now 5.2; attention with its
// logsumexp 8.8, now 8.4).  They are ordinary tensors over one storage, so that record_stream and the like act on the memory that all of
// them are in; it is free when the last of them is.  Hence what a cache keeps from block to block (the new state and conv window) is not
// among them, and larger ones (kSharedBytes together), of prompts say, have their own, as one would keep the others' memory.
class Outputs {
    static constexpr size_t kSharedBytes = 4 << 20, kAlign = 256;
    const at::Tensor& like;
    at::Tensor block;                      // undefined: one allocation each
    size_t used = 0;
    static size_t room(size_t bytes) { return (bytes + kAlign - 1) / kAlign * kAlign; }
public:
    struct Part { at::IntArrayRef size; at::ScalarType st; };
    Outputs(const at::Tensor& like, std::initializer_list<Part> parts) : like(like) {
        size_t total = 0;
        for (const Part& p : parts) total += room((size_t)c10::multiply_integers(p.size) * c10::elementSize(p.st));
        if (total <= kSharedBytes) block = fresh({(int64_t)total}, at::kByte, like);
    }
    // the next part, in the order and with the sizes that were named
    at::Tensor next(at::IntArrayRef size, at::ScalarType st) {
        if (!block.defined()) return fresh(size, st, like);
        auto impl = c10::make_intrusive<at::TensorImpl>(c10::Storage(block.storage()), block.key_set(), c10::scalarTypeToTypeMeta(st));
        impl->set_storage_offset((int64_t)(used / c10::elementSize(st)));
        impl->set_sizes_contiguous(size);
        used += room((size_t)c10::multiply_integers(size) * c10::elementSize(st));
        return at::Tensor(std::move(impl));
    }
};

void* stream() { return (void*)c10::hip::getCurrentHIPStream().stream(); }

// Runs a library call without the interpreter lock.
struct Unlocked {
    PyThreadState* ts = PyEval_SaveThread();
    ~Unlocked() { PyEval_RestoreThread(ts); }
};
template <typename F> int enqueue(F f) {
    Unlocked u;
    return f();
}
void check(int rc, const char* what) {
    if (rc == DFLASH_OK) return;
    raise(rc == DFLASH_UNSUPPORTED ? g_unsupported : g_error, "%s: %s (status %d)", what, dflash_last_error(), rc);
}

PyObject* wrap(at::Tensor&& t) {
    if (!t.defined()) Py_RETURN_NONE;
    PyObject* o = THPVariable_Wrap(std::move(t));
    if (!o) throw python_error();
    return o;
}
void put(PyObject* dict, const char* key, at::Tensor&& t) {
    PyObject* o = wrap(std::move(t));
    const int rc = PyDict_SetItemString(dict, key, o);
    Py_DECREF(o);
    if (rc) throw python_error();
}

void need_rank(const at::Tensor& t, int64_t rank, const char* fn, const char* what) {
    if (t.dim() != rank) raise(PyExc_ValueError, "%s: %s must have %d dimensions, got %d", fn, what, (int)rank, (int)t.dim());
}

// ---- recurrences -----------------------------------------------------------

// (tape, k, g, state, mask)
PyObject* tape_replay(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 5, "tape_replay");
    const at::Tensor &tape_ = tensor(a[0], "tape"), &k_ = tensor(a[1], "k"), &g_ = tensor(a[2], "g"), &state_ = tensor(a[3], "state"),
                     &mask_ = tensor_or_none(a[4], "mask");
    need_rank(k_, 4, "tape_replay_kernel", "k");
    need_rank(tape_, 4, "tape_replay_kernel", "tape");
    const Held tape = held(tape_), k = held(k_), g = held_as(g_, k_.scalar_type()), state = held(state_), mask = held_or_none(mask_);
    const int64_t B = k->size(0), T = k->size(1), Hk = k->size(2), Dk = k->size(3), Hv = tape->size(2), Dv = tape->size(3);
    at::Tensor out = fresh(state->sizes(), state->scalar_type(), *state);
    const int tc = code(*tape), kc = code(*k), sc = code(*state), mc = mask->defined() ? code(*mask) : 0;
    void* st = stream();
    check(enqueue([&] {
              return dflash_tape_replay(st, ptr(*tape), tc, ptr(*k), ptr(*g), kc, (int)g->dim(), ptr(*state), ptr(out), sc, ptr(*mask), mc,
                                        (int)B, (int)T, (int)Hk, (int)Hv, (int)Dk, (int)Dv);
          }),
          "tape_replay_kernel");
    return wrap(std::move(out));
    END_HANDLE_TH_ERRORS
}

// (q, k, v, g, beta, state, mask, want_state) -> (y, state or None, tape)
PyObject* gated_delta(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 8, "gated_delta");
    const at::Tensor &q_ = tensor(a[0], "q"), &k_ = tensor(a[1], "k"), &v_ = tensor(a[2], "v"), &g_ = tensor(a[3], "g"),
                     &beta_ = tensor(a[4], "beta"), &state_ = tensor(a[5], "state"), &mask_ = tensor_or_none(a[6], "mask");
    const bool want_state = truth(a[7]);
    const char* names[4] = {"k", "v", "g", "beta"};
    const at::Tensor* rest[4] = {&k_, &v_, &g_, &beta_};
    for (int i = 0; i < 4; ++i)
        if (rest[i]->scalar_type() != q_.scalar_type())
            raise(g_unsupported, "gated_delta_kernel_with_tape: %s dtype torch.%s differs from q's torch.%s", names[i],
                  c10::toString(rest[i]->scalar_type()), c10::toString(q_.scalar_type()));
    need_rank(k_, 4, "gated_delta_kernel_with_tape", "k");
    need_rank(v_, 4, "gated_delta_kernel_with_tape", "v");
    const Held q = held(q_), k = held(k_), v = held(v_), g = held(g_), beta = held(beta_), state = held(state_), mask = held_or_none(mask_);
    const int64_t B = k->size(0), T = k->size(1), Hk = k->size(2), Dk = k->size(3), Hv = v->size(2), Dv = v->size(3);
    const int64_t rows[4] = {B, T, Hv, Dv};
    Outputs outs(*q, {{rows, q->scalar_type()}, {rows, at::kFloat}});
    at::Tensor y = outs.next(rows, q->scalar_type()), tape = outs.next(rows, at::kFloat);
    at::Tensor out;                        // on its own: a cache keeps it when the others are gone
    if (want_state) out = fresh(state->sizes(), state->scalar_type(), *state);
    const int qc = code(*q), sc = code(*state), mc = mask->defined() ? code(*mask) : 0;
    void* st = stream();
    check(enqueue([&] {
              return dflash_gated_delta_tape(st, ptr(*q), ptr(*k), ptr(*v), ptr(*g), (int)g->dim(), ptr(*beta), qc, ptr(*state), ptr(out), sc,
                                             ptr(y), (float*)ptr(tape), ptr(*mask), mc, (int)B, (int)T, (int)Hk, (int)Hv, (int)Dk, (int)Dv);
          }),
          "gated_delta_kernel_with_tape");
    PyObject* r = PyTuple_New(3);
    if (!r) throw python_error();
    PyTuple_SET_ITEM(r, 0, wrap(std::move(y)));
    PyTuple_SET_ITEM(r, 1, wrap(std::move(out)));
    PyTuple_SET_ITEM(r, 2, wrap(std::move(tape)));
    return r;
    END_HANDLE_TH_ERRORS
}

// Arrival counters of the layer's in-launch gated norm: int32 zeros per (device, stream, B*Hv), left zero by every call.
at::Tensor kept_arrivals(const at::Tensor& like, int64_t count) {
    static std::mutex mu;
    static auto* kept = new std::map<std::tuple<int, void*, int64_t>, at::Tensor>();     // lives as long as the process
    const auto key = std::make_tuple((int)like.device().index(), stream(), count);
    {
        std::lock_guard<std::mutex> lock(mu);
        const auto it = kept->find(key);
        if (it != kept->end()) return it->second;
    }
    // zeros created inside a capture would only be RECORDED (and live in the graph's private pool): an eager call on this
    // stream before the first replay would count into uninitialised memory
    if (c10::hip::currentStreamCaptureStatusMayInitCtx() != c10::hip::CaptureStatus::None)
        raise(g_error, "gdn_layer: first use on this stream happens inside a graph capture; pass "
                       "`arrivals` (int32 zeros [B*Hv]) or call gdn_layer once on this stream beforehand");
    at::Tensor zeros = at::zeros({count}, like.options().dtype(at::kInt));
    std::lock_guard<std::mutex> lock(mu);
    return kept->emplace(key, std::move(zeros)).first->second;
}

// (mixed_qkv, conv_state, conv_weight, a_logits, b_logits, a_log, dt_bias, state, Hk, Hv, Dk, Dv, q_scale, k_scale, eps,
//  gate, norm_weight, norm_eps, silu, want_intermediates, arrivals, one_launch, out) -> dict
PyObject* gdn_layer(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 23, "gdn_layer");
    const at::Tensor &x_ = tensor(a[0], "mixed_qkv"), &cs_ = tensor_or_none(a[1], "conv_state"), &w_ = tensor(a[2], "conv_weight"),
                     &al_ = tensor(a[3], "a_logits"), &bl_ = tensor(a[4], "b_logits"), &alog_ = tensor(a[5], "a_log"),
                     &dtb_ = tensor(a[6], "dt_bias"), &state_ = tensor(a[7], "state"), &gate_ = tensor_or_none(a[15], "gate"),
                     &nw_ = tensor_or_none(a[16], "norm_weight");
    const int64_t Hk = integer(a[8]), Hv = integer(a[9]), Dk = integer(a[10]), Dv = integer(a[11]);
    const float q_scale = number(a[12]), k_scale = number(a[13]), eps = number(a[14]), norm_eps = number(a[17]);
    const int silu = (int)integer(a[18]);
    const bool want = truth(a[19]), one_launch = truth(a[21]);
    need_rank(x_, 3, "gdn_layer", "mixed_qkv");
    need_rank(w_, 2, "gdn_layer", "conv_weight");
    const int64_t B = x_.size(0), T = x_.size(1), C = x_.size(2), K = w_.size(1);
    if (C != 2 * Hk * Dk + Hv * Dv)
        raise(g_error, "gdn_layer: %d channels, expected 2*%d*%d + %d*%d", (int)C, (int)Hk, (int)Dk, (int)Hv, (int)Dv);
    if (al_.dim() != 3) raise(g_unsupported, "gdn_layer: one decay per head and step only (a_logits [B,T,Hv])");
    if (state_.scalar_type() != at::kFloat) raise(g_unsupported, "gdn_layer: float32 state only");
    const at::ScalarType dt = x_.scalar_type();
    const Held x = held(x_), w = held_as(w_, dt), cs = held_as(cs_, dt), al = held_as(al_, dt), bl = held_as(bl_, dt),
               alog = held_as(alog_, at::kFloat), dtb = held_as(dtb_, at::kFloat), state = held(state_);
    const int64_t qk_size[4] = {B, T, Hk, Dk}, g_size[3] = {B, T, Hv}, y_size[4] = {B, T, Hv, Dv}, none[1] = {0};
    const bool own_out = gate_.defined() && a[22] == Py_None;
    const auto only = [&](bool given, at::IntArrayRef size) { return given ? size : at::IntArrayRef(none); };
    Outputs outs(*x, {{qk_size, dt}, {g_size, dt}, {y_size, dt}, {y_size, at::kFloat}, {only(want, qk_size), dt}, {only(want, y_size), dt},
                      {only(want, g_size), dt}, {only(own_out, y_size), dt}});
    at::Tensor k = outs.next(qk_size, dt), g = outs.next(g_size, dt), y = outs.next(y_size, dt), tape = outs.next(y_size, at::kFloat);
    // on their own: a cache keeps them when the others are gone
    at::Tensor new_conv = fresh({B, K - 1, C}, dt, *x), new_state = fresh(state->sizes(), at::kFloat, *state), q, v, beta, out, arrivals;
    if (want) {
        q = outs.next(qk_size, dt);
        v = outs.next(y_size, dt);
        beta = outs.next(g_size, dt);
    }
    Held zg = held_as(gate_, dt), nw = held_as(nw_, dt);
    if (gate_.defined()) {
        if (!nw_.defined() || gate_.sizes() != y.sizes() || nw_.dim() != 1 || nw_.size(0) != Dv)
            raise(g_error, "gdn_layer: gate must be [B,T,Hv,Dv] and come with norm_weight [Dv]");
        if (own_out) {
            out = outs.next(y_size, dt);
        } else {
            if (!THPVariable_Check(a[22])) raise(PyExc_TypeError, "gdn_layer: out must be a tensor");
            out = THPVariable_Unpack(a[22]);
            if (out.sizes() != y.sizes() || out.scalar_type() != dt || !out.is_contiguous() || !out.is_cuda())
                raise(g_error, "gdn_layer: out must be a contiguous device tensor [B,T,Hv,Dv] of the input type");
        }
        if (one_launch) {
            if (a[20] == Py_None) {
                arrivals = kept_arrivals(*x, B * Hv);
            } else {
                if (!THPVariable_Check(a[20])) raise(PyExc_TypeError, "gdn_layer: arrivals must be a tensor");
                arrivals = THPVariable_Unpack(a[20]);
                if (arrivals.scalar_type() != at::kInt || arrivals.numel() < B * Hv || !arrivals.is_contiguous())
                    raise(g_error, "gdn_layer: arrivals must be a contiguous int32 tensor of at least B*Hv elements");
            }
        }
    }
    const int xc = code(*x);
    void* st = stream();
    check(enqueue([&] {
              return dflash_gdn_layer(st, ptr(*x), ptr(*cs), ptr(*w), ptr(*al), ptr(*bl), (const float*)ptr(*alog), (const float*)ptr(*dtb), xc,
                                      q_scale, k_scale, eps, ptr(*state), ptr(new_state), ptr(k), ptr(g), (float*)ptr(tape), ptr(new_conv),
                                      ptr(y), gate_.defined() ? ptr(*zg) : nullptr, gate_.defined() ? ptr(*nw) : nullptr, norm_eps, silu,
                                      ptr(out), (int32_t*)ptr(arrivals), ptr(q), ptr(v), ptr(beta), (int)B, (int)T, (int)Hk, (int)Hv, (int)Dk,
                                      (int)Dv, (int)K);
          }),
          "gdn_layer");
    PyObject* r = PyDict_New();
    if (!r) throw python_error();
    put(r, "out", std::move(out));
    put(r, "y", std::move(y));
    put(r, "state", std::move(new_state));
    put(r, "tape", std::move(tape));
    put(r, "k", std::move(k));
    put(r, "g", std::move(g));
    put(r, "conv_state", std::move(new_conv));
    if (want) {
        put(r, "q", std::move(q));
        put(r, "v", std::move(v));
        put(r, "beta", std::move(beta));
    }
    return r;
    END_HANDLE_TH_ERRORS
}

// ---- attention ---------------------------------------------------------------

// What the three attention calls share behind their own checks.  An output is allocated only for a call that goes out.
struct AttentionCall {
    at::Tensor workspace, out, lse;
    int dtype = 0;
    bool unused = false;                   // no workspace given, and none allocated: the call would not touch it
    // false: the shape or type is not covered (the caller returns None).  may_skip: the caller has an entry that takes no workspace.
    bool prepare(const at::Tensor& q, int64_t Hk, int64_t N, const at::Tensor& given, bool want_lse, bool may_skip = false) {
        const int B = (int)q.size(0), Hq = (int)q.size(1), M = (int)q.size(2), D = (int)q.size(3);
        const size_t need = dflash_sdpa_workspace_bytes(B, Hq, (int)Hk, M, (int)N, D);
        if (need == 0) return false;
        dtype = code_or(q.scalar_type(), -1);
        if (dtype < 0) return false;
        unused = may_skip && !given.defined() && need <= DFLASH_SDPA_STATIC_SCRATCH_BYTES && dflash_sdpa_scratch_bytes(B, Hq, (int)Hk, M, (int)N, D) == 0;
        if (!unused) workspace = given.defined() ? given : fresh({(int64_t)need}, at::kByte, q);
        if (!want_lse) {
            out = fresh(q.sizes(), q.scalar_type(), q);
            return true;
        }
        Outputs outs(q, {{q.sizes(), q.scalar_type()}, {q.sizes().slice(0, 3), at::kFloat}});
        out = outs.next(q.sizes(), q.scalar_type());
        lse = outs.next(q.sizes().slice(0, 3), at::kFloat);
        return true;
    }
    size_t workspace_bytes() const { return (size_t)workspace.numel() * workspace.element_size(); }
    PyObject* result(int rc, const char* what) {
        if (rc == DFLASH_UNSUPPORTED) Py_RETURN_NONE;
        check(rc, what);
        if (!lse.defined()) return wrap(std::move(out));
        PyObject* r = PyTuple_New(2);
        if (!r) throw python_error();
        PyTuple_SET_ITEM(r, 0, wrap(std::move(out)));
        PyTuple_SET_ITEM(r, 1, wrap(std::move(lse)));
        return r;
    }
};

bool rows_apart(const at::Tensor& k, const at::Tensor& v, int64_t D) {
    return k.stride(3) == 1 && k.stride(2) == D && k.strides() == v.strides();
}

// The additive mask as the kernels read it: of the queries' type, expanded and contiguous (DFlashKernels.swift:783-787).
Held held_mask(const at::Tensor& mask, at::ScalarType st, at::IntArrayRef size) {
    if (!mask.defined() || (mask.scalar_type() == st && mask.sizes() == size && mask.is_contiguous())) return Held::borrowed(mask);
    // what expand() takes: trailing sizes that are equal or 1
    bool fits = mask.dim() <= (int64_t)size.size();
    for (int64_t i = 0; fits && i < mask.dim(); ++i) {
        const int64_t have = mask.size(mask.dim() - 1 - i);
        fits = have == size[size.size() - 1 - i] || have == 1;
    }
    if (!fits) {
        std::string have;
        for (int64_t i = 0; i < mask.dim(); ++i) have += std::to_string(mask.size(i)) + (i + 1 < mask.dim() ? ", " : mask.dim() == 1 ? "," : "");
        raise(g_error, "batched_sdpa_2pass: mask (%s) does not broadcast to (%lld, %lld, %lld, %lld)", have.c_str(), (long long)size[0],
              (long long)size[1], (long long)size[2], (long long)size[3]);
    }
    return Held::owned(mask.to(st).expand(size).contiguous());
}

// (queries, keys, values, scale, mask, return_lse, kv_len, workspace); mask: anything that broadcasts to [B,Hq,M,N], of any type
PyObject* sdpa(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 8, "sdpa");
    for (int i = 0; i < 3; ++i)
        if (THPVariable_Check(a[i]) && THPVariable_Unpack(a[i]).dim() != 4) Py_RETURN_NONE;
    const at::Tensor &q_ = tensor(a[0], "queries"), &k_ = tensor(a[1], "keys"), &v_ = tensor(a[2], "values"),
                     &mask_ = tensor_or_none(a[4], "mask"), &len = tensor_or_none(a[6], "kv_len"), &ws = tensor_or_none(a[7], "workspace");
    const float scale = number(a[3]);
    const int64_t B = q_.size(0), Hq = q_.size(1), M = q_.size(2), D = q_.size(3), Hk = k_.size(1), N = k_.size(2);
    const int64_t mask_size[4] = {B, Hq, M, N};
    const Held mask = held_mask(mask_, q_.scalar_type(), mask_size);
    if (v_.sizes() != k_.sizes() || v_.size(3) != D || k_.scalar_type() != q_.scalar_type() || v_.scalar_type() != q_.scalar_type())
        Py_RETURN_NONE;
    const Held q = held(q_);
    const bool as_is = rows_apart(k_, v_, D);
    const Held k = as_is ? Held::borrowed(k_) : held(k_), v = as_is ? Held::borrowed(v_) : held(v_);
    AttentionCall c;
    if (!c.prepare(*q, Hk, N, ws, truth(a[5]), !mask->defined())) Py_RETURN_NONE;
    void* st = stream();
    const int64_t bs = k->stride(0), hs = k->stride(1);
    const int rc = enqueue([&] {
        // one split writes the output itself: no workspace is allocated for it (0.4 us of a call that enqueues in 5), the library's array, which
        // is as little touched, stands in
        if (c.unused)
            return dflash_sdpa_block_causal_static(st, ptr(*q), ptr(*k), ptr(*v), ptr(c.out), (float*)ptr(c.lse), c.dtype, scale, (int)B, (int)Hq,
                                                   (int)Hk, (int)M, (int)N, (int)D, bs, hs, (const int32_t*)ptr(len));
        return mask->defined() ? dflash_sdpa_block_causal_masked(st, ptr(*q), ptr(*k), ptr(*v), ptr(*mask), ptr(c.out), (float*)ptr(c.lse), c.dtype,
                                                                scale, (int)B, (int)Hq, (int)Hk, (int)M, (int)N, (int)D, bs, hs,
                                                                (const int32_t*)ptr(len), ptr(c.workspace), c.workspace_bytes())
                              : dflash_sdpa_block_causal(st, ptr(*q), ptr(*k), ptr(*v), ptr(c.out), (float*)ptr(c.lse), c.dtype, scale, (int)B,
                                                         (int)Hq, (int)Hk, (int)M, (int)N, (int)D, bs, hs, (const int32_t*)ptr(len),
                                                         ptr(c.workspace), c.workspace_bytes());
    });
    return c.result(rc, "batched_sdpa_2pass");
    END_HANDLE_TH_ERRORS
}

// (queries, k_cache, v_cache, k_new, v_new, scale, n_keys, return_lse, cache_len, workspace)
PyObject* sdpa_append(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 10, "sdpa_append");
    const at::Tensor &q_ = tensor(a[0], "queries"), &kc = tensor(a[1], "k_cache"), &vc = tensor(a[2], "v_cache"), &kn_ = tensor(a[3], "k_new"),
                     &vn_ = tensor(a[4], "v_new"), &len = tensor_or_none(a[8], "cache_len"), &ws = tensor_or_none(a[9], "workspace");
    const float scale = number(a[5]);
    const int64_t N = integer(a[6]);
    if (q_.dim() != 4 || kc.dim() != 4 || kc.sizes() != vc.sizes()) Py_RETURN_NONE;
    const int64_t B = q_.size(0), Hq = q_.size(1), M = q_.size(2), D = q_.size(3), Hk = kc.size(1), cap = kc.size(2);
    const int64_t want[4] = {B, Hk, M, D};
    const at::IntArrayRef rows(want, 4);
    if (kn_.sizes() != rows || vn_.sizes() != rows || kc.size(3) != D) Py_RETURN_NONE;
    for (const at::Tensor* t : {&kc, &vc, &kn_, &vn_})
        if (t->scalar_type() != q_.scalar_type()) Py_RETURN_NONE;
    if (!(M <= N && N <= cap))
        raise(g_error, "batched_sdpa_2pass_append: n_keys=%lld outside [%lld, capacity=%lld]", (long long)N, (long long)M, (long long)cap);
    if (!rows_apart(kc, vc, D)) raise(g_error, "batched_sdpa_2pass_append: the caches must be row-contiguous and laid out alike");
    const Held q = held(q_), kn = held(kn_), vn = held(vn_);
    AttentionCall c;
    if (!c.prepare(*q, Hk, N, ws, truth(a[7]))) Py_RETURN_NONE;
    void* st = stream();
    const int rc = enqueue([&] {
        return dflash_sdpa_block_causal_append(st, ptr(*q), ptr(kc), ptr(vc), ptr(*kn), ptr(*vn), ptr(c.out), (float*)ptr(c.lse), c.dtype, scale,
                                               (int)B, (int)Hq, (int)Hk, (int)M, (int)N, (int)D, kc.stride(0), kc.stride(1),
                                               (const int32_t*)ptr(len), ptr(c.workspace), c.workspace_bytes());
    });
    return c.result(rc, "batched_sdpa_2pass_append");
    END_HANDLE_TH_ERRORS
}

// (queries, k_pool, v_pool, page_table, scale, n_keys, k_new, v_new, lengths, return_lse, workspace)
PyObject* sdpa_paged(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 11, "sdpa_paged");
    const at::Tensor &q_ = tensor(a[0], "queries"), &kp = tensor(a[1], "k_pool"), &vp = tensor(a[2], "v_pool"),
                     &table = tensor(a[3], "page_table"), &kn_ = tensor_or_none(a[6], "k_new"), &vn_ = tensor_or_none(a[7], "v_new"),
                     &len = tensor_or_none(a[8], "lengths"), &ws = tensor_or_none(a[10], "workspace");
    const float scale = number(a[4]);
    const int64_t N = integer(a[5]);
    if (q_.dim() != 4 || kp.dim() != 4 || kp.sizes() != vp.sizes() || table.dim() != 2) Py_RETURN_NONE;
    const int64_t B = q_.size(0), Hq = q_.size(1), M = q_.size(2), D = q_.size(3);
    const int64_t num_pages = kp.size(0), Hk = kp.size(1), page_size = kp.size(2);
    const at::ScalarType dt = q_.scalar_type();
    if (kp.size(3) != D || kp.scalar_type() != dt || vp.scalar_type() != dt) Py_RETURN_NONE;
    if (kn_.defined() != vn_.defined()) raise(g_error, "batched_sdpa_2pass_paged: k_new and v_new go together");
    const int64_t want[4] = {B, Hk, M, D};
    const at::IntArrayRef rows(want, 4);
    if (kn_.defined() && (kn_.sizes() != rows || vn_.sizes() != rows || kn_.scalar_type() != dt || vn_.scalar_type() != dt)) Py_RETURN_NONE;
    if (table.scalar_type() != at::kInt || table.size(0) != B || table.stride(1) != 1)
        raise(g_error, "batched_sdpa_2pass_paged: page_table must be int32 [B, pages] with unit inner stride");
    if (!rows_apart(kp, vp, D)) raise(g_error, "batched_sdpa_2pass_paged: the pools must be row-contiguous and laid out alike");
    if (table.size(1) * page_size < N)
        raise(g_error, "batched_sdpa_2pass_paged: %lld pages of %lld keys do not cover n_keys=%lld", (long long)table.size(1),
              (long long)page_size, (long long)N);
    const int64_t pitch = B > 1 ? table.stride(0) : table.size(1);         // a single row's stride means nothing
    const Held q = held(q_), kn = held_or_none(kn_), vn = held_or_none(vn_);
    AttentionCall c;
    if (!c.prepare(*q, Hk, N, ws, truth(a[9]))) Py_RETURN_NONE;
    void* st = stream();
    const int rc = enqueue([&] {
        return dflash_sdpa_block_causal_paged(st, ptr(*q), ptr(kp), ptr(vp), (const int32_t*)ptr(table), (int)pitch, (int)page_size,
                                              (int)num_pages, kp.stride(0), kp.stride(1), ptr(*kn), ptr(*vn), ptr(c.out), (float*)ptr(c.lse),
                                              c.dtype, scale, (int)B, (int)Hq, (int)Hk, (int)M, (int)N, (int)D, (const int32_t*)ptr(len),
                                              ptr(c.workspace), c.workspace_bytes());
    });
    return c.result(rc, "batched_sdpa_2pass_paged");
    END_HANDLE_TH_ERRORS
}

// ---- acceptance ----------------------------------------------------------------

// Four words that a kernel leaves in pinned host memory, waited for by looking at them.  The device-to-host copy of 16
// bytes this replaces is a call into the copy engine's path with a wait of its own, and the 4-byte upload of `start` ahead
// of it was another; both together took longer than the kernels.  kUnset is a value that none of the words can take: they
// are counts and token ids below 2^31.
class AcceptWords {
    static constexpr int32_t kUnset = INT32_MIN;
    at::Tensor host = at::Tensor(at::detail::empty_cpu({4}, at::kInt, /*pin_memory=*/true, std::nullopt));
    bool there() const {
        for (int i = 0; i < 4; ++i)
            if (__atomic_load_n(words() + i, __ATOMIC_ACQUIRE) == kUnset) return false;
        return true;
    }
public:
    AcceptWords() { for (int i = 0; i < 4; ++i) words()[i] = kUnset; }
    int32_t* words() const { return host.mutable_data_ptr<int32_t>(); }
    // Looks for up to two milliseconds, then lets the runtime wait for the stream (a long queue ahead of the kernel, an error).
    void wait() const {
        const c10::hip::HIPStream st = c10::hip::getCurrentHIPStream();
        Unlocked u;
        const auto until = std::chrono::steady_clock::now() + std::chrono::milliseconds(2);
        for (unsigned i = 1; !there(); ++i) {
            __builtin_ia32_pause();
            if (i % 256 == 0 && std::chrono::steady_clock::now() > until) {
                st.synchronize();
                break;
            }
        }
    }
};

PyObject* accept_tuple(const AcceptWords& w, int64_t start, at::Tensor&& posterior) {
    const int32_t* v = w.words();
    PyObject* post = wrap(std::move(posterior));
    return Py_BuildValue("(iiiLN)", v[0], v[1], v[2], (long long)(start + v[1]), post);
}

// (logits, suppress mask, verify_ids, start) -> (acceptance_len, commit_count, staged_first_next, start, posterior)
PyObject* greedy_accept(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 4, "greedy_accept");
    const at::Tensor &logits_ = tensor(a[0], "logits"), &mask_ = tensor_or_none(a[1], "suppress_token_mask"), &ids_ = tensor(a[2], "verify_ids");
    const int64_t start = integer(a[3]);
    need_rank(logits_, 2, "greedy_accept_commit", "logits");
    const Held logits = held(logits_), mask = held_as(mask_, at::kByte), ids = held_as(ids_, at::kInt);
    const int64_t T = logits->size(0), V = logits->size(1);
    if (ids->dim() < 1 || ids->size(0) != T) raise(g_error, "greedy_accept_commit: one logits row per verify position");
    const int lc = code(*logits);
    at::Tensor post = fresh({T}, at::kInt, *logits);
    at::Tensor ws = fresh({(int64_t)dflash_greedy_workspace_bytes((int)T, (int)V)}, at::kByte, *logits);
    const AcceptWords out;
    void* st = stream();
    check(enqueue([&] {
              return dflash_greedy_accept_commit(st, ptr(*logits), lc, (int)T, (int)V, (const uint8_t*)ptr(*mask), (const uint32_t*)ptr(*ids),
                                                 nullptr, out.words(), (uint32_t*)ptr(post), ptr(ws), (size_t)ws.numel());
          }),
          "greedy_accept_commit");
    out.wait();
    return accept_tuple(out, start, std::move(post));
    END_HANDLE_TH_ERRORS
}

// (verify_ids, posterior, start) -> (acceptance_len, commit_count, staged_first_next, start, None)
PyObject* accept_commit(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 3, "accept_commit");
    const at::Tensor &ids_ = tensor(a[0], "verify_ids"), &post_ = tensor(a[1], "posterior");
    const int64_t start = integer(a[2]);
    const Held ids = held_as(ids_, at::kInt), post = held_as(post_, at::kInt);
    const int64_t V = ids->dim() ? ids->size(0) : 0;
    if (!post->dim() || post->size(0) < V) raise(g_error, "accept_commit: posterior must cover every verify position");
    const AcceptWords out;
    void* st = stream();
    check(enqueue([&] {
              return dflash_accept_commit(st, (const uint32_t*)ptr(*ids), (const uint32_t*)ptr(*post), (int)V, nullptr, out.words());
          }),
          "accept_commit");
    out.wait();
    return accept_tuple(out, start, at::Tensor());
    END_HANDLE_TH_ERRORS
}

// ---- rollback caches: the handle as an integer -----------------------------------

dflash_cache_t* handle(PyObject* o) {
    void* p = PyLong_AsVoidPtr(o);
    if (!p && PyErr_Occurred()) throw python_error();
    return (dflash_cache_t*)p;
}

// (handle, slot, tensor or None) -> data pointer
PyObject* cache_set_slot(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 3, "cache_set_slot");
    void* p = nullptr;
    if (a[2] != Py_None) {
        if (!THPVariable_Check(a[2])) raise(PyExc_TypeError, "cache slots hold tensors");
        const at::Tensor& t = THPVariable_Unpack(a[2]);
        if (!t.is_cuda() || !t.is_contiguous()) raise(g_error, "cache slots hold contiguous device tensors");
        p = t.data_ptr();
    }
    check(dflash_cache_set_slot(handle(a[0]), (int)integer(a[1]), p), "cache_set_slot");
    return PyLong_FromVoidPtr(p);
    END_HANDLE_TH_ERRORS
}
// (handle, slot) -> data pointer
PyObject* cache_get_slot(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 2, "cache_get_slot");
    return PyLong_FromVoidPtr(dflash_cache_get_slot(handle(a[0]), (int)integer(a[1])));
    END_HANDLE_TH_ERRORS
}
// (handle) -> whether the cache is armed
PyObject* cache_is_armed(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 1, "cache_is_armed");
    return PyBool_FromLong(dflash_cache_is_armed(handle(a[0])));
    END_HANDLE_TH_ERRORS
}
// (handle, prefix_len)
PyObject* cache_arm(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 2, "cache_arm");
    check(dflash_cache_arm_rollback(handle(a[0]), integer(a[1])), "arm_rollback");
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}
// (handle, tape, k, g, qkv or None, state) -> the contiguous tensors whose pointers the handle now holds
PyObject* cache_record_tape(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 6, "cache_record_tape");
    const at::Tensor &tape_ = tensor(a[1], "tape"), &k_ = tensor(a[2], "k"), &g_ = tensor(a[3], "g"), &qkv_ = tensor_or_none(a[4], "qkv"),
                     &state = tensor(a[5], "state");
    need_rank(k_, 4, "record_tape", "k");
    need_rank(tape_, 4, "record_tape", "tape");
    const Held tape = held(tape_), k = held(k_), g = held(g_), qkv = held_or_none(qkv_);
    const bool q = qkv->defined();
    check(dflash_cache_record_tape(handle(a[0]), ptr(*tape), code(*tape), ptr(*k), ptr(*g), code(*k), (int)g->dim(), ptr(*qkv),
                                   q ? (int)qkv->element_size() : 2, code(state), (int)k->size(0), (int)k->size(1), (int)k->size(2),
                                   (int)tape->size(2), (int)k->size(3), (int)tape->size(3), q ? (int)qkv->size(-1) : 0),
          "record_tape");
    PyObject* r = PyTuple_New(4);
    if (!r) throw python_error();
    const Held* all[4] = {&tape, &k, &g, &qkv};
    for (int i = 0; i < 4; ++i) PyTuple_SET_ITEM(r, i, wrap(at::Tensor(**all[i])));
    return r;
    END_HANDLE_TH_ERRORS
}
// A rollback cache's tensors by address, cut down to those its slots hold now.
void forget_dead(PyObject* cache, dflash_cache_t* c) {
    static PyObject* const name = PyUnicode_InternFromString("_by_ptr");
    THPObjectPtr held(PyObject_GetAttr(cache, name)), kept(PyDict_New());
    if (!held || !kept) throw python_error();
    for (int slot = 0; slot < 2; ++slot) {
        THPObjectPtr p(PyLong_FromVoidPtr(dflash_cache_get_slot(c, slot)));
        if (!p) throw python_error();
        PyObject* const t = PyDict_GetItemWithError(held.get(), p.get());
        if (t ? PyDict_SetItem(kept.get(), p.get(), t) : PyErr_Occurred() != nullptr) throw python_error();
    }
    if (PyObject_SetAttr(cache, name, kept.get())) throw python_error();
}
// (caches, target_len, acceptance_length, drafted_tokens) -> (status, nanoseconds)
PyObject* restore(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 4, "restore");
    if (!PyList_Check(a[0])) raise(PyExc_TypeError, "restore: a list of caches expected");
    static PyObject* const name = PyUnicode_InternFromString("_handle");
    std::vector<dflash_cache_t*> h((size_t)PyList_GET_SIZE(a[0]));
    for (size_t i = 0; i < h.size(); ++i) {
        THPObjectPtr o(PyObject_GetAttr(PyList_GET_ITEM(a[0], (Py_ssize_t)i), name));
        if (!o) throw python_error();
        h[i] = handle(o.get());
    }
    const int64_t target = integer(a[1]);
    const int acc = (int)integer(a[2]), drafted = (int)integer(a[3]);
    int64_t ns = 0;
    void* st = stream();
    const int rc = enqueue([&] { return dflash_restore_target_cache_after_acceptance(h.data(), (int)h.size(), st, target, acc, drafted, &ns); });
    for (size_t i = 0; i < h.size() && (Py_ssize_t)i < PyList_GET_SIZE(a[0]); ++i) {
        const int kind = dflash_cache_kind(h[i]);
        // armed: the call was refused ahead of any change, and the handle still points at the snapshot, whose tensors no slot may hold
        if ((kind == DFLASH_CACHE_TAPE || kind == DFLASH_CACHE_SNAPSHOT) && !dflash_cache_is_armed(h[i])) forget_dead(PyList_GET_ITEM(a[0], (Py_ssize_t)i), h[i]);
    }
    return Py_BuildValue("(iL)", rc, (long long)ns);
    END_HANDLE_TH_ERRORS
}

// ---- the calls of a verify step on buffers that are there already, on a given stream ---------

void* handle_of(PyObject* o) {
    void* p = PyLong_AsVoidPtr(o);
    if (!p && PyErr_Occurred()) throw python_error();
    return p;
}
// (stream, q, k, v, g, beta, state_in, state_out or None, y, tape, Hk, Hv, Dk, Dv): one sequence, one decay per head and step
PyObject* gated_delta_into(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 14, "gated_delta_into");
    void* st = handle_of(a[0]);
    const at::Tensor &q = tensor(a[1], "q"), &k = tensor(a[2], "k"), &v = tensor(a[3], "v"), &g = tensor(a[4], "g"), &beta = tensor(a[5], "beta"),
                     &in = tensor(a[6], "state_in"), &out = tensor_or_none(a[7], "state_out"), &y = tensor(a[8], "y"), &tape = tensor(a[9], "tape");
    need_rank(k, 4, "gated_delta_into", "k");
    const int qc = code(q), sc = code(in), T = (int)k.size(1), Hk = (int)integer(a[10]), Hv = (int)integer(a[11]), Dk = (int)integer(a[12]),
              Dv = (int)integer(a[13]);
    check(enqueue([&] {
              return dflash_gated_delta_tape(st, ptr(q), ptr(k), ptr(v), ptr(g), 3, ptr(beta), qc, ptr(in), ptr(out), sc, ptr(y), (float*)ptr(tape),
                                             nullptr, 0, 1, T, Hk, Hv, Dk, Dv);
          }),
          "gated_delta_tape");
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}
// (stream, q, k, v, k_new, v_new, out, lse, scale, n_keys, length, workspace, page_table or None, page_size): one sequence; k, v the caches
// [1, Hk, rows, D] or, with a page table [1, pages], the pools [pages, Hk, page_size, D]
PyObject* sdpa_append_into(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 14, "sdpa_append_into");
    void* st = handle_of(a[0]);
    const at::Tensor &q = tensor(a[1], "q"), &k = tensor(a[2], "k"), &v = tensor(a[3], "v"), &kn = tensor(a[4], "k_new"), &vn = tensor(a[5], "v_new"),
                     &out = tensor(a[6], "out"), &lse = tensor(a[7], "lse"), &len = tensor(a[10], "length"), &ws = tensor(a[11], "workspace"),
                     &table = tensor_or_none(a[12], "page_table");
    need_rank(q, 4, "sdpa_append_into", "q");
    need_rank(k, 4, "sdpa_append_into", "k");
    const float scale = number(a[8]);
    const int N = (int)integer(a[9]), page = (int)integer(a[13]), Hq = (int)q.size(1), M = (int)q.size(2), D = (int)q.size(3), Hk = (int)k.size(1);
    const int dt = code(q);
    if (table.defined()) need_rank(table, 2, "sdpa_append_into", "page_table");
    check(enqueue([&] {
              return table.defined()
                         ? dflash_sdpa_block_causal_paged(st, ptr(q), ptr(k), ptr(v), (const int32_t*)ptr(table), (int)table.size(1), page, (int)k.size(0),
                                                          k.stride(0), k.stride(1), ptr(kn), ptr(vn), ptr(out), (float*)ptr(lse), dt, scale, 1, Hq, Hk, M, N, D,
                                                          (const int32_t*)ptr(len), ptr(ws), (size_t)ws.numel())
                         : dflash_sdpa_block_causal_append(st, ptr(q), ptr(k), ptr(v), ptr(kn), ptr(vn), ptr(out), (float*)ptr(lse), dt, scale, 1, Hq, Hk, M, N,
                                                           D, k.stride(0), k.stride(1), (const int32_t*)ptr(len), ptr(ws), (size_t)ws.numel());
          }),
          table.defined() ? "sdpa_block_causal_paged" : "sdpa_block_causal");
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

// () -> the current stream's handle
PyObject* current_stream(PyObject*, PyObject* const*, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 0, "current_stream");
    return PyLong_FromVoidPtr(stream());
    END_HANDLE_TH_ERRORS
}

// (DFlashError, DFlashUnsupported)
PyObject* set_errors(PyObject*, PyObject* const* a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    need_args(n, 2, "set_errors");
    Py_INCREF(a[0]);
    Py_INCREF(a[1]);
    g_error = a[0];
    g_unsupported = a[1];
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define FAST(name, fn) {name, (PyCFunction)(void (*)(void))fn, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FAST("set_errors", set_errors), FAST("tape_replay", tape_replay), FAST("gated_delta", gated_delta),
    FAST("gdn_layer", gdn_layer),   FAST("sdpa", sdpa),               FAST("sdpa_append", sdpa_append),
    FAST("sdpa_paged", sdpa_paged), FAST("current_stream", current_stream),
    FAST("gated_delta_into", gated_delta_into), FAST("sdpa_append_into", sdpa_append_into),
    FAST("greedy_accept", greedy_accept), FAST("accept_commit", accept_commit), FAST("cache_set_slot", cache_set_slot),
    FAST("cache_get_slot", cache_get_slot), FAST("cache_record_tape", cache_record_tape), FAST("cache_is_armed", cache_is_armed), FAST("cache_arm", cache_arm), FAST("restore", restore),
    {nullptr, nullptr, 0, nullptr},
};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_native", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__native(void) { return PyModule_Create(&module); }
