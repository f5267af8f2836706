// The host side of the operators in native code: a CPython extension that takes torch tensors, allocates the results,
// calls the C ABI of the kernel library on the current stream and registers the backward passes with autograd.
//
// What bounds a small call is the host: through Python autograd Functions and ctypes one token of WKV6 took 25 us for
// 6 us of kernels.  Here a call is one C function without pybind11 (METH_FASTCALL), results come straight from the caching
// allocator, and the backward is a C++ autograd node, which the engine runs without the interpreter.
//
// The kernel library stays free of torch: its entry points are looked up by name in the file that `bind` is given.
#include <Python.h>
#include <ATen/ATen.h>
#include <ATen/TracerMode.h>
#include <ATen/autocast_mode.h>
#include <c10/hip/HIPGuard.h>
#include <c10/hip/HIPStream.h>
#include <dlfcn.h>
#include <torch/csrc/Exceptions.h>
#include <torch/csrc/autograd/custom_function.h>
#include <torch/csrc/autograd/python_variable.h>
#include <torch/csrc/utils/pybind.h>

#include "../../include/rwkv_wkv_hip.h"

using at::Tensor;
using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

namespace {

#define WKV_ABI(X)                                                                                                          \
    X(wkv_strerror) X(wkv5_forward) X(wkv6_forward) X(wkv5_forward_workspace) X(wkv6_forward_workspace) X(wkv5_backward)      \
    X(wkv6_backward) X(wkv5_backward_workspace) X(wkv6_backward_workspace) X(wkv56_forward_scratch) X(wkv6_decode) X(wkv4_forward_with) X(wkv4_forward_scratch) X(wkv4_backward) \
    X(wkv4_checkpoint_bytes) X(wkv4_backward_workspace) X(wkv_rows_products) X(wkv_lora_mix_rows) X(wkv_timemix_head)         \
    X(wkv_widen_rows) X(wkv_shift_mix_forward) X(wkv_shift_mix_backward) X(wkv_shift_mix_backward_workspace)                  \
    X(wkv_lora_mix_forward) X(wkv_lora_mix_backward) X(wkv_lora_mix_backward_workspace) X(wkv_ln_gate_forward)                \
    X(wkv_ln_gate_backward) X(wkv_ln_gate_backward_workspace) X(wkv_relu_square_forward) X(wkv_relu_square_backward)          \
    X(wkv_sigmoid_mul_forward) X(wkv_sigmoid_mul_backward)
struct {
#define X(name) decltype(&::name) name = nullptr;
    WKV_ABI(X)
#undef X
} abi;
PyObject *wkv_error = nullptr;          // rwkv_wkv_hip.WKVError

// ---- errors: Python exceptions of the kinds the Python front end raises, from any thread
[[noreturn]] void raise(PyObject *type, const std::string &what) {
    const PyGILState_STATE st = PyGILState_Ensure();
    PyErr_SetString(type, what.c_str());
    python_error e;
    e.persist();
    PyGILState_Release(st);
    throw e;
}
#define REQUIRE(cond) do { if (!(cond)) raise(PyExc_AssertionError, #cond); } while (0)
void check(int status, const char *what) {
    if (status == WKV_OK) return;
    const std::string msg = std::string(what) + ": " + abi.wkv_strerror(status);
    if (status == WKV_ERR_DIMS || status == WKV_ERR_DTYPE) raise(PyExc_ValueError, msg);
    raise(wkv_error, msg + " (status " + std::to_string(status) + ")");
}
int dtype_code(const Tensor &t) {
    switch (t.scalar_type()) {
        case at::kFloat: return WKV_F32;
        case at::kBFloat16: return WKV_BF16;
        case at::kHalf: return WKV_F16;
        default: raise(PyExc_ValueError, std::string("Unsupported dtype ") + c10::toString(t.scalar_type()) + " for WKV");
    }
}
void on_gpu(const Tensor &t) {
    if (t.defined() && !t.is_cuda()) raise(wkv_error, "rwkv_wkv_hip operators need GPU tensors (there is no CPU path)");
}

void *ptr(const Tensor &t) { return t.defined() ? t.data_ptr() : nullptr; }
float *fptr(const Tensor &t) { return static_cast<float *>(ptr(t)); }
// whether an autograd node has to see this call: a gradient is recorded, or an input carries a forward-mode tangent (which
// no node here supports: torch's own error for that comes from the node, and a call passed by it would drop the tangent)
bool seen_by_autograd(std::initializer_list<const Tensor *> inputs) {
    for (const Tensor *t : inputs)
        if (t->defined() && ((at::GradMode::is_enabled() && t->requires_grad()) || t->_fw_grad(0).defined())) return true;
    return false;
}
// torch.jit.trace is recording.  It sees what goes through torch's dispatcher or a Python autograd Function, not the calls
// made here: a graph recorded through them would hold the uninitialised results.  The entry points answer None, and the
// Python front end makes the call one node of the graph (a layer is recorded step by step).
bool traced() { return at::tracer::impl::is_dispatch_enabled(); }
// the caller's tensor: the current device is its device and the stream is that device's current one
struct OnDevice {
    c10::hip::HIPGuard guard;
    explicit OnDevice(const Tensor &t) : guard(t.device().index()) {}
    void *stream() const { return c10::hip::getCurrentHIPStream(guard.current_device().index()).stream(); }
};
Tensor as_float(const Tensor &t) { return t.scalar_type() == at::kFloat ? t : t.to(at::kFloat); }
Tensor as_type(const Tensor &t, at::ScalarType d) { return t.scalar_type() == d ? t : t.to(d); }
Tensor bytes(size_t n, const Tensor &like) { return at::empty({(int64_t)std::max<size_t>(n, 16)}, like.options().dtype(at::kByte)); }

// ---- WKV5 / WKV6
struct Dims { int B, T, C, H; };
void check_streams(const Dims &d, const Tensor &r, const Tensor &k, const Tensor &v) {
    REQUIRE(r.scalar_type() == k.scalar_type() && r.scalar_type() == v.scalar_type());
    REQUIRE(r.is_contiguous() && k.is_contiguous() && v.is_contiguous());
    const int64_t want[3] = {d.B, d.T, d.C};
    for (const Tensor *t : {&r, &k, &v}) REQUIRE(t->sizes().equals(at::IntArrayRef(want, 3)));
}
size_t forward_bytes(int version, const Dims &d, int dt, int algo) {
    return (version == 5 ? abi.wkv5_forward_workspace : abi.wkv6_forward_workspace)(d.B, d.T, d.C, d.H, dt, algo);
}
size_t backward_bytes(int version, const Dims &d, int dt, int algo) {
    return (version == 5 ? abi.wkv5_backward_workspace : abi.wkv6_backward_workspace)(d.B, d.T, d.C, d.H, dt, algo);
}
unsigned flags_of(const Dims &d, const Tensor &w) {
    return (d.T > 1 ? WKV_FLOOR_DECAY : 0u) | (w.scalar_type() == at::kBFloat16 ? WKV_W_BF16 : w.scalar_type() == at::kHalf ? WKV_W_F16 : 0u);
}

struct Forward56 { Tensor y, state, ws; };
// `w` as the kernels read it (decay_operand); out_state: written in place of a new tensor.  keep: a backward call will
// follow, so the workspace in which the kernels leave their state checkpoints (sized for that call) comes back too.
Forward56 forward56(int version, const Dims &d, int algo, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w,
                    const Tensor &u, const Tensor &s, const Tensor &out_state, bool keep) {
    const int dt = dtype_code(r);
    check_streams(d, r, k, v);
    for (const Tensor *t : {&r, &k, &v, &w, &u, &s}) on_gpu(*t);
    OnDevice dev(r);
    Forward56 o;
    o.y = at::empty_like(r);
    o.state = out_state.defined() ? out_state : at::empty_like(s);
    if (version == 6 && d.T == 1 && w.scalar_type() != at::kFloat) {
        check(abi.wkv6_decode(dev.stream(), d.B, d.C, d.H, dt, dt, ptr(r), ptr(k), ptr(v), ptr(w), fptr(u), fptr(s), ptr(o.y), fptr(o.state)), "wkv6_decode");
        return o;
    }
    size_t n = 0;
    unsigned flags = flags_of(d, w);
    Tensor scratch;
    if (keep) {
        if ((n = forward_bytes(version, d, dt, algo)) > 0) o.ws = scratch = bytes(std::max(n, backward_bytes(version, d, dt, algo)), r);
    } else if ((n = abi.wkv56_forward_scratch(d.B, d.T, d.C, d.H, dt, algo)) > 0 && !out_state.is_same(s)) {
        flags |= WKV_NO_CHECKPOINTS;          // the time split's summaries; none where no sequence is cut
        scratch = bytes(n, r);
    }
    if (version == 5)
        check(abi.wkv5_forward(dev.stream(), d.B, d.T, d.C, d.H, dt, flags, algo, ptr(r), ptr(k), ptr(v), fptr(w), fptr(u), fptr(s),
                               ptr(o.y), fptr(o.state), ptr(scratch), scratch.defined() ? scratch.numel() : 0), "wkv5_forward");
    else
        check(abi.wkv6_forward(dev.stream(), d.B, d.T, d.C, d.H, dt, flags, algo, ptr(r), ptr(k), ptr(v), ptr(w), fptr(u), fptr(s),
                               ptr(o.y), fptr(o.state), ptr(scratch), scratch.defined() ? scratch.numel() : 0), "wkv6_forward");
    return o;
}

struct Backward56 { Tensor gr, gk, gv, gw, gu, gs; };
Backward56 backward56(int version, const Dims &d, int algo, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w,
                      const Tensor &u, const Tensor &s, const Tensor &gy, const Tensor &gstate, Tensor ws, bool want_gs,
                      const Tensor &gu = Tensor()) {
    const int dt = dtype_code(r);
    OnDevice dev(r);
    Backward56 g{at::empty_like(r), at::empty_like(k), at::empty_like(v), at::empty_like(w),
                 gu.defined() ? gu : at::empty_like(u), want_gs ? at::empty_like(s) : Tensor()};
    unsigned flags = flags_of(d, w);               // (a bf16 w has its gradient in bf16 too)
    const size_t need = backward_bytes(version, d, dt, algo);
    if (ws.defined() && (size_t)ws.numel() >= need) flags |= WKV_CHECKPOINTS_VALID;
    else ws = bytes(need, r);                      // no forward workspace, or one sized for another plan (wkv_tune): rebuilt inside
    if (version == 5)
        check(abi.wkv5_backward(dev.stream(), d.B, d.T, d.C, d.H, dt, flags, algo, ptr(r), ptr(k), ptr(v), fptr(w), fptr(u), fptr(s),
                                ptr(gy), fptr(gstate), ptr(g.gr), ptr(g.gk), ptr(g.gv), fptr(g.gw), fptr(g.gu), fptr(g.gs), ptr(ws),
                                ws.numel()), "wkv5_backward");
    else
        check(abi.wkv6_backward(dev.stream(), d.B, d.T, d.C, d.H, dt, flags, algo, ptr(r), ptr(k), ptr(v), ptr(w), fptr(u), fptr(s),
                                ptr(gy), fptr(gstate), ptr(g.gr), ptr(g.gk), ptr(g.gv), ptr(g.gw), fptr(g.gu), fptr(g.gs), ptr(ws),
                                ws.numel()), "wkv6_backward");
    return g;
}

// The raw decay in the type the kernels take: WKV5's is fp32; WKV6's is read as it is, in the type of the streams, where
// the call takes a blocked algorithm (the reference widens it, RWKV-v6/src/module/TimeMix.py:50), or is one token without
// a backward, and is widened here otherwise.
Tensor decay_operand(int version, const Dims &d, int algo, const Tensor &r, const Tensor &w, bool keep) {
    if (version == 5 || w.scalar_type() == at::kFloat) return w;
    if (w.scalar_type() == r.scalar_type()) {
        if (d.T == 1 && !keep) return w;
        if (d.T > 1 && forward_bytes(6, d, dtype_code(r), algo) > 0) return w;
    }
    return w.to(at::kFloat);
}

// in_place: the new state goes into `s` (the reference's convention, RWKV-v5/src/module/TimeMix.py:60,139-140: a private
// copy of the incoming state is kept and no gradient flows through it)
struct Call56 {
    int version, algo;
    Dims d;
    bool in_place;
    Tensor r, k, v, w, u, s;

    void check_operands() const {
        REQUIRE(s.is_contiguous() && w.is_contiguous() && u.is_contiguous());
        const int64_t state[4] = {d.B, d.H, 64, 64};
        REQUIRE(s.sizes().equals(at::IntArrayRef(state, 4)) && d.H * 64 == d.C);
        if (version == 5) {
            REQUIRE(s.scalar_type() == at::kFloat && w.scalar_type() == at::kFloat && w.numel() == d.C);
        } else {
            const int64_t streams[3] = {d.B, d.T, d.C};
            REQUIRE(w.sizes().equals(at::IntArrayRef(streams, 3)));
        }
        REQUIRE(u.numel() == d.C);
    }
    bool records() const {
        return seen_by_autograd({&r, &k, &v, &w, &u}) || (!in_place && seen_by_autograd({&s}));
    }
};

class Wkv56 : public torch::autograd::Function<Wkv56> {
public:
    static variable_list forward(AutogradContext *ctx, const Call56 *c, const Tensor &r, const Tensor &k, const Tensor &v, const Tensor &w,
                                 const Tensor &u, const Tensor &s) {
        const Tensor u32 = as_float(u), s_in = c->in_place ? s.clone() : as_float(s);
        const Tensor w32 = decay_operand(c->version, c->d, c->algo, r, w, true);
        Forward56 o = forward56(c->version, c->d, c->algo, r, k, v, w32, u32, s_in, c->in_place ? s : Tensor(), true);
        ctx->set_materialize_grads(false);
        ctx->saved_data["call"] = std::vector<int64_t>{c->version, c->algo, c->d.B, c->d.T, c->d.C, c->d.H, c->in_place,
                                                       (int64_t)w.scalar_type(), (int64_t)u.scalar_type(), (int64_t)s.scalar_type()};
        ctx->save_for_backward({r, k, v, w32, u32, s_in, o.ws});
        if (c->in_place) return {o.y};
        return {o.y, as_type(o.state, s.scalar_type())};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const std::vector<int64_t> c = ctx->saved_data["call"].toIntVector();
        const Dims d{(int)c[2], (int)c[3], (int)c[4], (int)c[5]};
        const bool in_place = c[6];
        const variable_list x = ctx->get_saved_variables();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor &r = x[0], &u = x[4], &s = x[5];
        Tensor gy = grads[0].defined() ? grads[0].contiguous() : at::zeros_like(r), gstate;
        REQUIRE(gy.scalar_type() == r.scalar_type());
        if (!in_place && grads[1].defined()) gstate = as_float(grads[1]).contiguous();
        const bool want_gs = !in_place && ctx->needs_input_grad(5);      // (counted over the tensors)
        Backward56 g = backward56((int)c[0], d, (int)c[1], r, x[1], x[2], x[3], u, s, gy, gstate, x[6], want_gs);
        return {Tensor(), g.gr, g.gk, g.gv, as_type(g.gw, (at::ScalarType)c[7]), as_type(g.gu, (at::ScalarType)c[8]),
                want_gs ? as_type(g.gs, (at::ScalarType)c[9]) : Tensor()};
    }
};

// (y, new state); the state is undefined where it went into the caller's buffer
std::pair<Tensor, Tensor> call56(const Call56 &c) {
    c.check_operands();
    dtype_code(c.r);
    for (const Tensor *t : {&c.r, &c.k, &c.v, &c.w, &c.u, &c.s}) on_gpu(*t);
    if (c.records()) {
        variable_list o = Wkv56::apply(&c, c.r, c.k, c.v, c.w, c.u, c.s);
        return {o[0], c.in_place ? Tensor() : o[1]};
    }
    at::AutoDispatchBelowADInplaceOrView below;
    // one token's kernel updates the state in place by itself
    const Tensor s_in = !c.in_place ? as_float(c.s) : c.d.T == 1 ? c.s : c.s.clone();
    Forward56 o = forward56(c.version, c.d, c.algo, c.r, c.k, c.v, decay_operand(c.version, c.d, c.algo, c.r, c.w, false), as_float(c.u),
                            s_in, c.in_place ? c.s : Tensor(), false);
    return {o.y, c.in_place ? Tensor() : as_type(o.state, c.s.scalar_type())};
}

// ---- WKV4
class Wkv4 : public torch::autograd::Function<Wkv4> {
public:
    static variable_list forward(AutogradContext *ctx, const Tensor &time_decay, const Tensor &time_first, const Tensor &k_, const Tensor &v_,
                                 const Tensor &state) {
        const Tensor td = as_float(time_decay).contiguous(), tf = as_float(time_first).contiguous();
        const Tensor k = k_.contiguous(), v = v_.contiguous(), st = as_float(state).contiguous();
        const int B = k.size(0), T = k.size(1), C = k.size(2);
        Tensor ckpt = ctx ? bytes(abi.wkv4_checkpoint_bytes(B, T, C), k) : Tensor();
        Tensor y = at::empty_like(k), out = at::empty_like(st);
        OnDevice dev(k);
        const size_t n = abi.wkv4_forward_scratch(B, T, C, dtype_code(k));
        const Tensor scratch = n > 0 ? bytes(n, k) : Tensor();
        check(abi.wkv4_forward_with(dev.stream(), B, T, C, dtype_code(k), fptr(td), fptr(tf), ptr(k), ptr(v), fptr(st), ptr(y), fptr(out),
                                    ptr(ckpt), ptr(scratch), n), "wkv4_forward");
        if (ctx) {
            ctx->set_materialize_grads(false);
            ctx->saved_data["types"] = std::vector<int64_t>{(int64_t)time_decay.scalar_type(), (int64_t)time_first.scalar_type(), (int64_t)state.scalar_type()};
            ctx->save_for_backward({td, tf, k, v, st, ckpt});
        }
        return {y, out};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const std::vector<int64_t> types = ctx->saved_data["types"].toIntVector();
        const variable_list x = ctx->get_saved_variables();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor &td = x[0], &tf = x[1], &k = x[2], &v = x[3], &st = x[4], &ckpt = x[5];
        const int B = k.size(0), T = k.size(1), C = k.size(2), dt = dtype_code(k);
        const Tensor gy = grads[0].defined() ? grads[0].contiguous() : at::zeros_like(k);
        // a state gradient of zeros: its exponent is zero too, as the reference's backward is handed when autograd has none
        const Tensor gstate = grads[1].defined() ? as_float(grads[1]).contiguous() : at::zeros_like(st);
        Tensor gtd = at::empty_like(td), gtf = at::empty_like(tf), gk = at::empty_like(k), gv = at::empty_like(v), gst = at::empty_like(st);
        OnDevice dev(k);          // (before the query: the plan is the device's)
        Tensor ws = bytes(abi.wkv4_backward_workspace(B, T, C, dt), k);
        check(abi.wkv4_backward(dev.stream(), B, T, C, dt, fptr(td), fptr(tf), ptr(k), ptr(v), fptr(st), ptr(gy), fptr(gstate), fptr(gtd),
                                fptr(gtf), ptr(gk), ptr(gv), fptr(gst), ptr(ckpt), ptr(ws), ws.numel()), "wkv4_backward");
        return {as_type(gtd, (at::ScalarType)types[0]), as_type(gtf, (at::ScalarType)types[1]), gk, gv, as_type(gst, (at::ScalarType)types[2])};
    }
};

// ---- Python arguments
// The interpreter lock is given up once the arguments are in hand (the tensors' own handles are held, nothing borrowed from Python
// objects): allocations, launches and library products may wait for the GPU, and other threads run meanwhile.
typedef pybind11::gil_scoped_release NoLock;
const Tensor &tensor(PyObject *o) {
    if (!THPVariable_Check(o)) raise(PyExc_TypeError, std::string("expected a torch.Tensor, got ") + Py_TYPE(o)->tp_name);
    return THPVariable_Unpack(o);
}
Tensor maybe_tensor(PyObject *o) { return o == Py_None ? Tensor() : tensor(o); }
int integer(PyObject *o) {
    const long x = PyLong_AsLong(o);
    if (x == -1 && PyErr_Occurred()) throw python_error();
    if (x < INT_MIN || x > INT_MAX) raise(PyExc_OverflowError, "size out of range");
    return (int)x;
}
PyObject *wrapped(const Tensor &t) {
    if (!t.defined()) Py_RETURN_NONE;
    return THPVariable_Wrap(t);
}
template <class... Ts> PyObject *tuple(const Ts &...ts) {
    PyObject *o = PyTuple_New(sizeof...(ts));
    if (!o) throw python_error();
    Py_ssize_t i = 0;
    (PyTuple_SET_ITEM(o, i++, wrapped(ts)), ...);
    return o;
}
void arity(Py_ssize_t n, Py_ssize_t want) {
    if (n != want) raise(PyExc_TypeError, "wrong number of arguments");
}

// wkv56(version, algo, in_place, B, T, C, H, r, k, v, w, u, s) -> (y, new_state), or y with the new state in s; None: traced
PyObject *py_wkv56(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 13);
    if (traced()) Py_RETURN_NONE;
    const Call56 c{integer(a[0]), integer(a[1]), {integer(a[3]), integer(a[4]), integer(a[5]), integer(a[6])}, a[2] == Py_True,
                   tensor(a[7]), tensor(a[8]), tensor(a[9]), tensor(a[10]), tensor(a[11]), tensor(a[12])};
    Tensor y, state;
    {
        NoLock no_lock;
        std::tie(y, state) = call56(c);
    }
    return c.in_place ? wrapped(y) : tuple(y, state);
    END_HANDLE_TH_ERRORS
}

// forward56(version, algo, B, T, C, H, r, k, v, w, u, s, out_state or None) -> (y, new_state, workspace or None): the bare call
// with checkpoints kept, w already as the kernels read it
PyObject *py_forward56(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 13);
    const int version = integer(a[0]), algo = integer(a[1]);
    const Dims d{integer(a[2]), integer(a[3]), integer(a[4]), integer(a[5])};
    const Tensor r = tensor(a[6]), k = tensor(a[7]), v = tensor(a[8]), w = tensor(a[9]), u = tensor(a[10]), st = tensor(a[11]), out = maybe_tensor(a[12]);
    Forward56 o;
    {
        NoLock no_lock;
        at::AutoDispatchBelowADInplaceOrView below;
        o = forward56(version, d, algo, r, k, v, w, u, st, out, true);
    }
    return tuple(o.y, o.state, o.ws);
    END_HANDLE_TH_ERRORS
}

// backward56(version, algo, B, T, C, H, r, k, v, w, u, s, gy, gstate or None, workspace or None) -> gr, gk, gv, gw, gu, gs
PyObject *py_backward56(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 15);
    const int version = integer(a[0]), algo = integer(a[1]);
    const Dims d{integer(a[2]), integer(a[3]), integer(a[4]), integer(a[5])};
    const Tensor r = tensor(a[6]), k = tensor(a[7]), v = tensor(a[8]), w = tensor(a[9]), u = tensor(a[10]), st = tensor(a[11]), gy = tensor(a[12]);
    const Tensor gstate = maybe_tensor(a[13]), ws = maybe_tensor(a[14]);
    Backward56 g;
    {
        NoLock no_lock;
        at::AutoDispatchBelowADInplaceOrView below;
        g = backward56(version, d, algo, r, k, v, w, u, st, gy, gstate, ws, true);
    }
    return tuple(g.gr, g.gk, g.gv, g.gw, g.gu, g.gs);
    END_HANDLE_TH_ERRORS
}

// decay_operand(algo, B, T, C, H, r, w) -> w as the kernels of a WKV6 call with a backward read it
PyObject *py_decay_operand(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 7);
    const Dims d{integer(a[1]), integer(a[2]), integer(a[3]), integer(a[4])};
    const int algo = integer(a[0]);
    const Tensor r = tensor(a[5]), w = tensor(a[6]);
    Tensor o;
    {
        NoLock no_lock;
        o = decay_operand(6, d, algo, r, w, true);
    }
    return wrapped(o);
    END_HANDLE_TH_ERRORS
}

// wkv4(time_decay, time_first, k, v, state) -> (y, new_state); None: traced
PyObject *py_wkv4(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 5);
    if (traced()) Py_RETURN_NONE;
    const Tensor td = tensor(a[0]), tf = tensor(a[1]), k = tensor(a[2]), v = tensor(a[3]), st = tensor(a[4]);
    variable_list o;
    {
        NoLock no_lock;
        REQUIRE(k.dim() == 3 && v.sizes().equals(k.sizes()) && k.scalar_type() == v.scalar_type());
        const int64_t B = k.size(0), C = k.size(2), state[3] = {B, C, 3};
        REQUIRE(td.dim() == 1 && td.size(0) == C && tf.dim() == 1 && tf.size(0) == C && st.sizes().equals(at::IntArrayRef(state, 3)));
        dtype_code(k);
        for (const Tensor *t : {&td, &tf, &k, &v, &st}) on_gpu(*t);
        if (seen_by_autograd({&td, &tf, &k, &v, &st})) {
            o = Wkv4::apply(td, tf, k, v, st);
        } else {
            at::AutoDispatchBelowADInplaceOrView below;
            o = Wkv4::forward(nullptr, td, tf, k, v, st);
        }
    }
    return tuple(o[0], o[1]);
    END_HANDLE_TH_ERRORS
}

#include "host_layers.h"

// bind(path of the kernel library, WKVError, torch.nn.Linear, torch.nn.GroupNorm, (the dictionaries of hooks on all modules))
PyObject *py_bind(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 5);
    REQUIRE(PyTuple_Check(a[4]));
    const char *path = PyUnicode_AsUTF8(a[0]);
    if (!path) throw python_error();
    for (int i = 1; i < 5; i++) Py_INCREF(a[i]);
    wkv_error = a[1]; linear_type = a[2]; group_norm_type = a[3]; global_hooks = a[4];
    void *lib = dlopen(path, RTLD_NOW | RTLD_LOCAL);
    if (!lib) raise(wkv_error, dlerror());
#define X(name)                                                                   \
    abi.name = reinterpret_cast<decltype(&::name)>(dlsym(lib, #name));            \
    if (!abi.name) raise(wkv_error, std::string(path) + " lacks " #name);
    WKV_ABI(X)
#undef X
    Py_RETURN_NONE;
    END_HANDLE_TH_ERRORS
}

#define METHOD(name) {#name, reinterpret_cast<PyCFunction>(reinterpret_cast<void *>(py_##name)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {METHOD(bind), METHOD(wkv56), METHOD(forward56), METHOD(backward56), METHOD(decay_operand), METHOD(wkv4), METHOD(timemix),
                         METHOD(channelmix),
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "native host side of rwkv_wkv_hip", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
