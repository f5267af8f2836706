// The layers' halves in native code: `timemix` and `channelmix` take a module that holds the reference's parameters under
// the reference's names and do what its forward does (RWKV-v5/src/module/TimeMix.py:286-323, ChannelMix.py:35-49;
// RWKV-v6/src/module/TimeMix.py:253-302, ChannelMix.py:30-37), each as ONE autograd node whose backward is written out
// below.  As Python functions over a node per step a v6 layer's forward and backward took 1670 us of host time (45 nodes,
// some 130 launches), whatever its size; the projections stay library products.
//
// bf16 modules only.  Single tokens without autograd take the kernels of csrc/layer_decode.hip.
//
// A module's parameters and submodules are read from its dictionaries: nn.Module's attribute lookup costs more than a
// kernel's launch.  Whatever is not plain (hooks, biases, subclasses of Linear, other types or sizes, autocast switched
// on) gets no answer here, and the caller takes its general way.  (Part of host.cpp.)
PyObject *linear_type = nullptr, *group_norm_type = nullptr, *global_hooks = nullptr;      // global_hooks: a tuple of dicts
PyObject *dict_of(PyObject *o) {          // borrowed
    PyObject **d = _PyObject_GetDictPtr(o);
    return d ? *d : nullptr;
}
PyObject *item(PyObject *dict, const char *name) {          // borrowed, or NULL
    return dict && PyDict_Check(dict) ? PyDict_GetItemString(dict, name) : nullptr;
}
bool globally_hooked() {
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(global_hooks); i++)
        if (PyObject_Length(PyTuple_GET_ITEM(global_hooks, i)) != 0) return true;
    return false;
}
// collects the tensors of one call; `ok` falls if one of them is not what the kernels take
struct Plain {
    const Tensor &x;
    bool ok = true;
    explicit Plain(const Tensor &x_) : x(x_) {}
    bool takes(const Tensor &t, int64_t numel, at::ScalarType type = at::kBFloat16) {
        return ok = ok && t.defined() && t.device() == x.device() && t.scalar_type() == type && t.numel() == numel && t.is_contiguous() &&
                    !t.key_set().has(c10::DispatchKey::Python) && !t._fw_grad(0).defined() && (reinterpret_cast<uintptr_t>(t.data_ptr()) & 15) == 0;
    }
    // an input: its shape too (the parameters' C elements may come in any)
    bool takes(const Tensor &t, at::IntArrayRef shape, at::ScalarType type = at::kBFloat16) {
        return ok = ok && t.defined() && t.sizes().equals(shape) && takes(t, t.numel(), type);
    }
    Tensor parameter(PyObject *params, const char *name, int64_t numel) {          // (undefined where `ok` fell)
        PyObject *o = item(params, name);
        if (!o || !THPVariable_Check(o)) ok = false;
        return ok && takes(THPVariable_Unpack(o), numel) ? THPVariable_Unpack(o) : Tensor();
    }
    Tensor matrix(PyObject *params, const char *name, int64_t rows, int64_t cols) {
        Tensor t = parameter(params, name, rows * cols);
        ok = ok && t.dim() == 2 && t.size(0) == rows;
        return t;
    }
    Tensor linear(PyObject *modules, const char *name, int64_t n, int64_t k) {          // weight (n, k), no bias
        PyObject *o = item(modules, name), *d = nullptr, *p;
        ok = ok && o && (PyObject *)Py_TYPE(o) == linear_type && (d = dict_of(o)) && !item(d, "forward") && (p = item(d, "_parameters")) &&
             item(p, "bias") == Py_None && unhooked(d);
        return ok ? matrix(item(d, "_parameters"), "weight", n, k) : Tensor();
    }
    static bool unhooked(PyObject *d) {
        for (const char *name : {"_forward_hooks", "_forward_pre_hooks", "_backward_hooks", "_backward_pre_hooks"}) {
            PyObject *h = item(d, name);
            if (!h || PyObject_Length(h) != 0) return false;
        }
        return true;
    }
};

// The operands of a TimeMix: in t[] in this order (the order of the autograd node's inputs)
enum { X, SHIFT, STATE, DECAY, U, LN_W, LN_B, WR, WK, WV, WG, WO, MIX0 };          // then the mixes: v5 k, v, r, g
enum { MAA_X = MIX0, MAA_W, MAA_K, MAA_V, MAA_R, MAA_G, W1, W2, DW1, DW2, N6 };      // v6
enum { N5 = MIX0 + 4 };
struct TimeMixCall {
    int version, algo;
    Dims d;
    float eps;
    Tensor t[N6];          // (handles of their own: the interpreter lock is given up after collecting them)
    bool keep;          // a backward will follow
};
bool collect(TimeMixCall &c, PyObject *module, PyObject *px, PyObject *states) {
    PyObject *dict = dict_of(module), *prm = item(dict, "_parameters"), *mod = item(dict, "_modules"), *heads = item(dict, "n_head");
    if (!prm || !mod || !heads || !PyLong_Check(heads) || !THPVariable_Check(px) || !PyTuple_Check(states) || PyTuple_GET_SIZE(states) != 2) return false;
    PyObject *sh = PyTuple_GET_ITEM(states, 0), *st = PyTuple_GET_ITEM(states, 1);
    if (!THPVariable_Check(sh) || !THPVariable_Check(st)) return false;
    const Tensor &x = THPVariable_Unpack(px);
    if (!x.is_cuda() || x.dim() != 3 || traced() || globally_hooked() || at::autocast::is_autocast_enabled(at::kCUDA)) return false;
    const int64_t B = x.size(0), T = x.size(1), C = x.size(2), H = PyLong_AsLong(heads);
    if (H <= 0 || H * 64 != C || B <= 0 || T <= 0 || B > 65535 || T > (1 << 20) || B * T > INT_MAX) return false;
    c.d = {(int)B, (int)T, (int)C, (int)H};
    Plain p(x);
    p.takes(x, B * T * C);
    p.takes(THPVariable_Unpack(sh), {B, C});
    p.takes(THPVariable_Unpack(st), {B, H, 64, 64}, at::kFloat);
    PyObject *ln = item(mod, "ln_x"), *lnd = nullptr, *eps = nullptr;
    p.ok = p.ok && ln && (PyObject *)Py_TYPE(ln) == group_norm_type && (lnd = dict_of(ln)) && (eps = item(lnd, "eps")) && PyFloat_Check(eps);
    if (!p.ok) return false;
    c.eps = (float)PyFloat_AS_DOUBLE(eps);
    c.t[X] = x; c.t[SHIFT] = THPVariable_Unpack(sh); c.t[STATE] = THPVariable_Unpack(st);
    c.t[DECAY] = p.parameter(prm, "time_decay", C);
    c.t[U] = p.parameter(prm, "time_faaaa", C);
    c.t[LN_W] = p.parameter(item(lnd, "_parameters"), "weight", C);
    c.t[LN_B] = p.parameter(item(lnd, "_parameters"), "bias", C);
    const char *projections[5] = {"receptance", "key", "value", "gate", "output"};
    for (int j = 0; j < 5; j++) c.t[WR + j] = p.linear(mod, projections[j], C, C);
    if (c.version == 6) {
        const char *maa[6] = {"time_maa_x", "time_maa_w", "time_maa_k", "time_maa_v", "time_maa_r", "time_maa_g"};
        for (int j = 0; j < 6; j++) c.t[MAA_X + j] = p.parameter(prm, maa[j], C);
        c.t[W1] = p.matrix(prm, "time_maa_w1", C, 160);
        c.t[W2] = p.parameter(prm, "time_maa_w2", C * 160);
        p.ok = p.ok && c.t[W2].dim() == 3 && c.t[W2].size(0) == 5 && c.t[W2].size(1) == 32;
        PyObject *o = item(prm, "time_decay_w1");
        const int64_t D = o && THPVariable_Check(o) ? THPVariable_Unpack(o).numel() / C : 0;
        c.t[DW1] = p.matrix(prm, "time_decay_w1", C, D);
        c.t[DW2] = p.matrix(prm, "time_decay_w2", D, C);
    } else {
        const char *mix[4] = {"time_mix_k", "time_mix_v", "time_mix_r", "time_mix_g"};
        for (int j = 0; j < 4; j++) c.t[MIX0 + j] = p.parameter(prm, mix[j], C);
    }
    return p.ok;
}
bool any_requires_grad(const Tensor *t, int n) {
    for (int i = 0; i < n; i++)
        if (t[i].requires_grad()) return true;
    return false;
}

// ---- the steps, on tensors of one device whose stream is handed in
Tensor widen_rows(void *stream, const Tensor &like, const void *const *rows, int count, int64_t C) {      // bf16 parameters of C elements -> (count, C) fp32
    Tensor out = at::empty({count, C}, like.options().dtype(at::kFloat));
    check(abi.wkv_widen_rows(stream, count, C, rows, fptr(out)), "wkv_widen_rows");
    return out;
}
template <int N> struct Planes {          // the N planes of a tensor (N, ...)
    void *p[N];
    explicit Planes(const Tensor &t) { for (int j = 0; j < N; j++) p[j] = static_cast<char *>(t.data_ptr()) + j * (t.nbytes() / N); }
};
Tensor shift_mix(void *stream, const Dims &d, int n, bool lerp, const Tensor &x, const Tensor &shift, const float *coef) {
    Tensor out = at::empty({n, d.B * (int64_t)d.T, d.C}, x.options());
    void *outs[5];
    for (int j = 0; j < n; j++) outs[j] = static_cast<char *>(out.data_ptr()) + j * (out.nbytes() / n);
    check(abi.wkv_shift_mix_forward(stream, d.B, d.T, d.C, WKV_BF16, n, lerp, ptr(x), ptr(shift), coef, nullptr, outs), "wkv_shift_mix_forward");
    return out;
}
// gradients of the n mixed copies (n, B*T, C) -> of x, of the shift state and, in gcoef (n, C), of the coefficients
struct MixGrads { Tensor gx, gshift; };
MixGrads shift_mix_backward(void *stream, const Dims &d, int n, bool lerp, const Tensor &x, const Tensor &shift, const float *coef, const Tensor &gout,
                            float *gcoef) {
    MixGrads g{at::empty_like(x), at::empty_like(shift)};
    const void *gouts[5];
    for (int j = 0; j < n; j++) gouts[j] = static_cast<const char *>(gout.data_ptr()) + j * (gout.nbytes() / n);
    const Tensor ws = bytes(abi.wkv_shift_mix_backward_workspace(d.B, d.T, d.C, n), x);
    check(abi.wkv_shift_mix_backward(stream, d.B, d.T, d.C, WKV_BF16, n, lerp, ptr(x), ptr(shift), coef, nullptr, gouts, ptr(g.gx), ptr(g.gshift),
                                     gcoef, nullptr, ptr(ws), ws.numel()), "wkv_shift_mix_backward");
    return g;
}
Tensor plane(const Tensor &t, int64_t j) { return t.select(0, j); }
Tensor times_t(const Tensor &x, const Tensor &w) { return at::mm(x, w.t()); }          // x W^T, the projection

// What the backward needs of the forward, in the order in which it is saved after the operands
enum { COEF, XXX, ACT, W2T, MIXES, RR, KK, VV, GG, LORA, WW, YY, ZZ, WS, SAVED };
struct TimeMixOut { Tensor out, state, saved[SAVED]; };
TimeMixOut timemix_forward(const TimeMixCall &c) {
    const Dims &d = c.d;
    const Tensor *t = c.t;
    const int64_t M = d.B * (int64_t)d.T, C = d.C;
    OnDevice dev(t[X]);
    void *stream = dev.stream();
    TimeMixOut o;
    const void *rows[9] = {ptr(t[U]), ptr(t[LN_W]), ptr(t[LN_B])};
    const int mixes = c.version == 6 ? 6 : 4;
    for (int j = 0; j < mixes; j++) rows[3 + j] = ptr(t[MIX0 + j]);
    const Tensor coef = o.saved[COEF] = widen_rows(stream, t[X], rows, 3 + mixes, C);
    const float *mix = fptr(coef) + 3 * C;
    int r, k, v, g;
    if (c.version == 6) {
        o.saved[XXX] = shift_mix(stream, d, 1, false, t[X], t[SHIFT], mix).view({M, C});
        o.saved[ACT] = at::mm(o.saved[XXX], t[W1]).tanh_();
        o.saved[W2T] = t[W2].transpose(1, 2).contiguous();
        o.saved[MIXES] = at::empty({5, M, C}, t[X].options());
        check(abi.wkv_lora_mix_forward(stream, d.B, d.T, d.C, ptr(t[X]), ptr(t[SHIFT]), mix + C, ptr(o.saved[ACT]), ptr(o.saved[W2T]),
                                       Planes<5>(o.saved[MIXES]).p), "wkv_lora_mix_forward");
        r = 3; k = 1; v = 2; g = 4;
    } else {
        o.saved[MIXES] = shift_mix(stream, d, 4, true, t[X], t[SHIFT], mix);
        r = 2; k = 0; v = 1; g = 3;
    }
    const Tensor &m = o.saved[MIXES];
    o.saved[RR] = times_t(plane(m, r), t[WR]);
    o.saved[KK] = times_t(plane(m, k), t[WK]);
    o.saved[VV] = times_t(plane(m, v), t[WV]);
    o.saved[GG] = times_t(plane(m, g), t[WG]);
    const int64_t streams[3] = {d.B, d.T, d.C};
    auto seq = [&](const Tensor &x) { return x.view(at::IntArrayRef(streams, 3)); };
    if (c.version == 6) {
        o.saved[LORA] = at::mm(plane(m, 0), t[DW1]).tanh_();
        // the broadcast addition of time_decay rides on the product as its bias
        const Tensor w = at::addmm(t[DECAY].view({C}), o.saved[LORA], t[DW2]);
        o.saved[WW] = decay_operand(6, d, c.algo, seq(o.saved[RR]), seq(w), c.keep);
    } else {
        o.saved[WW] = t[DECAY].to(at::kFloat);
    }
    Forward56 f = forward56(c.version, d, c.algo, seq(o.saved[RR]), seq(o.saved[KK]), seq(o.saved[VV]), o.saved[WW], coef.select(0, 0), t[STATE],
                            Tensor(), c.keep);
    o.saved[YY] = f.y;
    o.saved[WS] = f.ws;
    o.state = f.state;
    o.saved[ZZ] = at::empty({M, C}, t[X].options());
    check(abi.wkv_ln_gate_forward(stream, M, C, WKV_BF16, c.version == 6 ? 1.f : 0.125f, c.eps, ptr(f.y), ptr(o.saved[GG]), fptr(coef) + C,
                                  fptr(coef) + 2 * C, ptr(o.saved[ZZ])), "wkv_ln_gate_forward");
    o.out = seq(times_t(o.saved[ZZ], t[WO]));
    return o;
}

template <int VERSION> class TimeMix : public torch::autograd::Function<TimeMix<VERSION>> {
    static constexpr int N = VERSION == 6 ? (int)N6 : (int)N5;
public:
    template <class... Ts> static variable_list forward(AutogradContext *ctx, const TimeMixCall *c, const Ts &...ts) {
        static_assert(sizeof...(ts) == N, "one argument per operand");
        TimeMixOut o;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            o = timemix_forward(*c);
        }
        ctx->set_materialize_grads(false);
        ctx->saved_data["call"] = std::vector<int64_t>{c->algo, c->d.B, c->d.T, c->d.C, c->d.H};
        ctx->saved_data["eps"] = (double)c->eps;
        variable_list save{ts...};
        save.insert(save.end(), o.saved, o.saved + SAVED);
        ctx->save_for_backward(std::move(save));
        return {o.out, o.state};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const std::vector<int64_t> c = ctx->saved_data["call"].toIntVector();
        const int algo = (int)c[0];
        const Dims d{(int)c[1], (int)c[2], (int)c[3], (int)c[4]};
        const int64_t M = d.B * (int64_t)d.T, C = d.C;
        const float eps = (float)ctx->saved_data["eps"].toDouble();
        const variable_list all = ctx->get_saved_variables();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor *t = all.data(), *s = all.data() + N;
        OnDevice dev(t[X]);
        void *stream = dev.stream();
        const float *coef = fptr(s[COEF]), *mix = coef + 3 * C;
        variable_list g(1 + N);
        auto out = [&](int i) -> Tensor & { return g[1 + i]; };
        auto wants = [&](int i) { return ctx->needs_input_grad(i); };
        const Tensor gout = grads[0].defined() ? grads[0].contiguous().view({M, C}) : at::zeros({M, C}, t[X].options());
        REQUIRE(gout.scalar_type() == at::kBFloat16);
        const Tensor gstate = grads[1].defined() ? as_float(grads[1]).contiguous() : Tensor();
        // output projection, ln_x and gate
        const Tensor gz = at::mm(gout, t[WO]);
        if (wants(WO)) out(WO) = at::mm(gout.t(), s[ZZ]);
        const Tensor gy = at::empty_like(s[YY]), gg = at::empty_like(s[GG]);
        // fp32 gradients of the (C) parameters, rows of one conversion: u, ln weight, ln bias, mixes
        const Tensor gsmall = at::empty({VERSION == 6 ? 9 : 7, C}, s[COEF].options());
        float *gln = fptr(gsmall) + C, *gmix = fptr(gsmall) + 3 * C;
        {
            const Tensor ws = bytes(abi.wkv_ln_gate_backward_workspace(M, C), t[X]);
            check(abi.wkv_ln_gate_backward(stream, M, C, WKV_BF16, VERSION == 6 ? 1.f : 0.125f, eps, ptr(s[YY]), ptr(s[GG]), coef + C, coef + 2 * C,
                                           ptr(gz), ptr(gy), ptr(gg), gln, ptr(ws), ws.numel()), "wkv_ln_gate_backward");
        }
        // the operator
        const int64_t streams[3] = {d.B, d.T, d.C};
        auto seq = [&](const Tensor &x) { return x.view(at::IntArrayRef(streams, 3)); };
        const Backward56 b = backward56(VERSION, d, algo, seq(s[RR]), seq(s[KK]), seq(s[VV]), s[WW], s[COEF].select(0, 0), t[STATE], gy, gstate, s[WS],
                                        wants(STATE), gsmall.select(0, 0));
        out(STATE) = b.gs;
        // gradients of the mixed copies (v6: w, k, v, r, g; v5: k, v, r, g) and of the projections
        constexpr int MIXES_N = VERSION == 6 ? 5 : 4;
        const int at_k = VERSION == 6 ? 1 : 0;
        const Tensor gm = at::empty({MIXES_N, M, C}, t[X].options());
        const Tensor gproj[4] = {b.gk.view({M, C}), b.gv.view({M, C}), b.gr.view({M, C}), gg};
        const int weight[4] = {WK, WV, WR, WG};
        for (int j = 0; j < 4; j++) {
            Tensor into = plane(gm, at_k + j);
            at::mm_out(into, gproj[j], t[weight[j]]);
            if (wants(weight[j])) out(weight[j]) = at::mm(gproj[j].t(), plane(s[MIXES], at_k + j));
        }
        if (VERSION == 6) {
            const Tensor gw = as_type(b.gw, at::kBFloat16).view({M, C});
            if (wants(DECAY)) out(DECAY) = gw.sum(0).view(t[DECAY].sizes());
            if (wants(DW2)) out(DW2) = at::mm(s[LORA].t(), gw);
            const Tensor gl = at::tanh_backward(at::mm(gw, t[DW2].t()), s[LORA]);
            if (wants(DW1)) out(DW1) = at::mm(plane(s[MIXES], 0).t(), gl);
            Tensor into = plane(gm, 0);
            at::mm_out(into, gl, t[DW1].t());
            Tensor gx = at::empty_like(t[X]), gshift = at::empty_like(t[SHIFT]), gdyn = at::empty({5, M, C}, t[X].options());
            {
                const Tensor ws = bytes(abi.wkv_lora_mix_backward_workspace(d.B, d.T, d.C), t[X]);
                check(abi.wkv_lora_mix_backward(stream, d.B, d.T, d.C, ptr(t[X]), ptr(t[SHIFT]), mix + C, ptr(s[ACT]), ptr(s[W2T]),
                                                Planes<5>(gm).p, ptr(gx), ptr(gshift), gmix + C, ptr(gdyn), ptr(ws), ws.numel()),
                      "wkv_lora_mix_backward");
            }
            // the two reductions of the second LoRA product's backward, and the first product
            Tensor ga = at::empty({M, 5, 32}, t[X].options());
            ga.copy_(at::bmm(gdyn, s[W2T]).transpose(0, 1));
            if (wants(W2)) out(W2) = at::bmm(s[ACT].view({M, 5, 32}).permute({1, 2, 0}), gdyn);
            const Tensor gpre = at::tanh_backward(ga.view({M, 160}), s[ACT]);
            if (wants(W1)) out(W1) = at::mm(s[XXX].t(), gpre);
            const MixGrads first = shift_mix_backward(stream, d, 1, false, t[X], t[SHIFT], mix, at::mm(gpre, t[W1].t()), gmix);
            out(X) = gx.add_(first.gx);
            out(SHIFT) = gshift.add_(first.gshift);
        } else {
            if (wants(DECAY)) out(DECAY) = as_type(b.gw, at::kBFloat16).view(t[DECAY].sizes());
            const MixGrads first = shift_mix_backward(stream, d, 4, true, t[X], t[SHIFT], mix, gm, gmix);
            out(X) = first.gx;
            out(SHIFT) = first.gshift;
        }
        const Tensor small = gsmall.to(at::kBFloat16);
        const int rows[3] = {U, LN_W, LN_B};
        for (int j = 0; j < 3; j++) out(rows[j]) = small.select(0, j).view(t[rows[j]].sizes());
        for (int j = 0; j < (VERSION == 6 ? 6 : 4); j++) out(MIX0 + j) = small.select(0, 3 + j).view(t[MIX0 + j].sizes());
        return g;
    }
};
template <class F, size_t... I> variable_list apply_node(const TimeMixCall &c, std::index_sequence<I...>) { return F::apply(&c, c.t[I]...); }

// ---- channel mix
enum { CM_X, CM_SHIFT, CM_MIX_K, CM_MIX_R, CM_WK, CM_WR, CM_WV, CM_N };
struct ChannelMixCall {
    bool lerp;
    Dims d;
    int64_t F;
    Tensor t[CM_N];
};
bool collect(ChannelMixCall &c, PyObject *module, PyObject *px, PyObject *sh) {
    PyObject *dict = dict_of(module), *prm = item(dict, "_parameters"), *mod = item(dict, "_modules"), *key = item(mod, "key"), *kp;
    if (!prm || !key || !THPVariable_Check(px) || !THPVariable_Check(sh) || !(kp = item(item(dict_of(key), "_parameters"), "weight")) ||
        !THPVariable_Check(kp))
        return false;
    const Tensor &x = THPVariable_Unpack(px);
    if (!x.is_cuda() || x.dim() != 3 || traced() || globally_hooked() || at::autocast::is_autocast_enabled(at::kCUDA)) return false;
    const int64_t B = x.size(0), T = x.size(1), C = x.size(2);
    if (C <= 0 || C % 64 != 0 || B <= 0 || T <= 0 || B > 65535 || T > (1 << 20) || B * T > INT_MAX) return false;
    c.F = THPVariable_Unpack(kp).numel() / C;
    if (c.F < 8 || c.F % 8 != 0 || c.F > INT_MAX / C) return false;
    c.d = {(int)B, (int)T, (int)C, (int)(C / 64)};
    Plain p(x);
    p.takes(x, B * T * C);
    p.takes(THPVariable_Unpack(sh), {B, C});
    c.t[CM_X] = x; c.t[CM_SHIFT] = THPVariable_Unpack(sh);
    c.t[CM_MIX_K] = p.parameter(prm, c.lerp ? "time_mix_k" : "time_maa_k", C);
    c.t[CM_MIX_R] = p.parameter(prm, c.lerp ? "time_mix_r" : "time_maa_r", C);
    c.t[CM_WK] = p.linear(mod, "key", c.F, C);
    c.t[CM_WR] = p.linear(mod, "receptance", C, C);
    c.t[CM_WV] = p.linear(mod, "value", C, c.F);
    return p.ok;
}
enum { CM_COEF, CM_MIXES, CM_K, CM_K2, CM_KV, CM_R, CM_SAVED };
struct ChannelMixOut { Tensor out, saved[CM_SAVED]; };
ChannelMixOut channelmix_forward(const ChannelMixCall &c) {
    const Dims &d = c.d;
    const Tensor *t = c.t;
    OnDevice dev(t[CM_X]);
    void *stream = dev.stream();
    ChannelMixOut o;
    const void *rows[2] = {ptr(t[CM_MIX_K]), ptr(t[CM_MIX_R])};
    o.saved[CM_COEF] = widen_rows(stream, t[CM_X], rows, 2, d.C);
    o.saved[CM_MIXES] = shift_mix(stream, d, 2, c.lerp, t[CM_X], t[CM_SHIFT], fptr(o.saved[CM_COEF]));
    const Tensor k = o.saved[CM_K] = times_t(plane(o.saved[CM_MIXES], 0), t[CM_WK]);
    o.saved[CM_K2] = at::empty_like(k);
    check(abi.wkv_relu_square_forward(stream, k.numel(), WKV_BF16, ptr(k), ptr(o.saved[CM_K2])), "wkv_relu_square_forward");
    o.saved[CM_KV] = times_t(o.saved[CM_K2], t[CM_WV]);
    const Tensor r = o.saved[CM_R] = times_t(plane(o.saved[CM_MIXES], 1), t[CM_WR]);
    o.out = at::empty_like(t[CM_X]);
    check(abi.wkv_sigmoid_mul_forward(stream, r.numel(), WKV_BF16, ptr(r), ptr(o.saved[CM_KV]), ptr(o.out)), "wkv_sigmoid_mul_forward");
    return o;
}
class ChannelMix : public torch::autograd::Function<ChannelMix> {
public:
    static variable_list forward(AutogradContext *ctx, const ChannelMixCall *c, const Tensor &x, const Tensor &shift, const Tensor &mix_k,
                                 const Tensor &mix_r, const Tensor &wk, const Tensor &wr, const Tensor &wv) {
        ChannelMixOut o;
        {
            at::AutoDispatchBelowADInplaceOrView below;
            o = channelmix_forward(*c);
        }
        ctx->set_materialize_grads(false);
        ctx->saved_data["call"] = std::vector<int64_t>{c->lerp, c->d.B, c->d.T, c->d.C};
        ctx->save_for_backward({x, shift, mix_k, mix_r, wk, wr, wv, o.saved[CM_COEF], o.saved[CM_MIXES], o.saved[CM_K], o.saved[CM_K2],
                                o.saved[CM_KV], o.saved[CM_R]});
        return {o.out};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        const std::vector<int64_t> c = ctx->saved_data["call"].toIntVector();
        const Dims d{(int)c[1], (int)c[2], (int)c[3], (int)(c[3] / 64)};
        const variable_list all = ctx->get_saved_variables();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor *t = all.data(), *s = all.data() + CM_N;
        if (!grads[0].defined()) return variable_list(1 + CM_N);
        OnDevice dev(t[CM_X]);
        void *stream = dev.stream();
        auto wants = [&](int i) { return ctx->needs_input_grad(i); };
        const Tensor gout = grads[0].contiguous();
        REQUIRE(gout.scalar_type() == at::kBFloat16);
        variable_list g(1 + CM_N);
        const Tensor gr = at::empty_like(s[CM_R]), gkv = at::empty_like(s[CM_KV]);
        check(abi.wkv_sigmoid_mul_backward(stream, gr.numel(), WKV_BF16, ptr(s[CM_R]), ptr(s[CM_KV]), ptr(gout), ptr(gr), ptr(gkv)), "wkv_sigmoid_mul_backward");
        const Tensor gk2 = at::mm(gkv, t[CM_WV]), gk = at::empty_like(gk2);
        if (wants(CM_WV)) g[1 + CM_WV] = at::mm(gkv.t(), s[CM_K2]);
        check(abi.wkv_relu_square_backward(stream, gk.numel(), WKV_BF16, ptr(s[CM_K]), ptr(gk2), ptr(gk)), "wkv_relu_square_backward");
        const Tensor gm = at::empty_like(s[CM_MIXES]);
        Tensor into = plane(gm, 0);
        at::mm_out(into, gk, t[CM_WK]);
        if (wants(CM_WK)) g[1 + CM_WK] = at::mm(gk.t(), plane(s[CM_MIXES], 0));
        into = plane(gm, 1);
        at::mm_out(into, gr, t[CM_WR]);
        if (wants(CM_WR)) g[1 + CM_WR] = at::mm(gr.t(), plane(s[CM_MIXES], 1));
        const Tensor gcoef = at::empty_like(s[CM_COEF]);
        const MixGrads m = shift_mix_backward(stream, d, 2, c[0], t[CM_X], t[CM_SHIFT], fptr(s[CM_COEF]), gm, fptr(gcoef));
        g[1 + CM_X] = m.gx;
        g[1 + CM_SHIFT] = m.gshift;
        const Tensor small = gcoef.to(at::kBFloat16);
        g[1 + CM_MIX_K] = small.select(0, 0).view(t[CM_MIX_K].sizes());
        g[1 + CM_MIX_R] = small.select(0, 1).view(t[CM_MIX_R].sizes());
        return g;
    }
};

// ---- one token per sequence, nothing recorded (csrc/layer_decode.hip)
bool single_tokens(const Dims &d) { return d.T == 1 && d.B <= 64; }
std::pair<Tensor, Tensor> timemix_decode(const TimeMixCall &c) {
    const Tensor *t = c.t;
    const int64_t B = c.d.B, C = c.d.C, rows = B * C;
    const Tensor &x = t[X];
    const bool v6 = c.version == 6;
    OnDevice dev(x);
    void *stream = dev.stream();
    // scratch: r, k, v, gate, the head results; v6 also the five mixes and the two LoRAs' activations
    constexpr int64_t parts = 2 * WKV_LORA_PARTS;          // (fp32 counted in bf16)
    Tensor scratch = at::empty({(v6 ? 10 : 5) * rows + (v6 ? parts * B * 224 : 0)}, x.options());
    at::BFloat16 *q = scratch.data_ptr<at::BFloat16>();
    at::BFloat16 *r = q, *k = r + rows, *v = k + rows, *g = v + rows, *z = g + rows, *mixes = z + rows, *act = mixes + 5 * rows, *lora = act + parts * B * 160;
    Tensor out = at::empty_like(x), state = at::empty_like(t[STATE]);
    const void *px = ptr(x), *ps = ptr(t[SHIFT]), *wr = ptr(t[WR]), *wk = ptr(t[WK]), *wv = ptr(t[WV]), *wg = ptr(t[WG]);
    const int n = (int)C;
    if (v6) {
        const void *maa[5];
        for (int j = 0; j < 5; j++) maa[j] = ptr(t[MAA_W + j]);
        const wkv_rows_product first{ptr(t[W1]), px, ps, ptr(t[MAA_X]), nullptr, act, 160, 1, 0, 0};
        check(abi.wkv_rows_products(stream, B, C, 1, &first), "wkv_rows_products");
        check(abi.wkv_lora_mix_rows(stream, B, C, px, ps, maa, act, ptr(t[W2]), mixes), "wkv_lora_mix_rows");
        const wkv_rows_product proj[5] = {{ptr(t[DW1]), mixes, nullptr, nullptr, nullptr, lora, 64, 1, 0, 0},
                                          {wk, mixes + rows, nullptr, nullptr, nullptr, k, n, 0, 0, 0},
                                          {wv, mixes + 2 * rows, nullptr, nullptr, nullptr, v, n, 0, 0, 0},
                                          {wr, mixes + 3 * rows, nullptr, nullptr, nullptr, r, n, 0, 0, 0},
                                          {wg, mixes + 4 * rows, nullptr, nullptr, nullptr, g, n, 0, 0, 0}};
        check(abi.wkv_rows_products(stream, B, C, 5, proj), "wkv_rows_products");
    } else {
        const wkv_rows_product proj[4] = {{wk, px, ps, ptr(t[MIX0]), nullptr, k, n, 0, 1, 0}, {wv, px, ps, ptr(t[MIX0 + 1]), nullptr, v, n, 0, 1, 0},
                                          {wr, px, ps, ptr(t[MIX0 + 2]), nullptr, r, n, 0, 1, 0}, {wg, px, ps, ptr(t[MIX0 + 3]), nullptr, g, n, 0, 1, 0}};
        check(abi.wkv_rows_products(stream, B, C, 4, proj), "wkv_rows_products");
    }
    check(abi.wkv_timemix_head(stream, B, C, c.d.H, r, k, v, g, ptr(t[DECAY]), v6 ? lora : nullptr, v6 ? ptr(t[DW2]) : nullptr, ptr(t[U]), ptr(t[LN_W]),
                               ptr(t[LN_B]), v6 ? 1.f : 0.125f, c.eps, fptr(t[STATE]), fptr(state), z), "wkv_timemix_head");
    const wkv_rows_product last{ptr(t[WO]), z, nullptr, nullptr, nullptr, ptr(out), n, 0, 0, 0};
    check(abi.wkv_rows_products(stream, B, C, 1, &last), "wkv_rows_products");
    return {out, state};
}
Tensor channelmix_decode(const ChannelMixCall &c) {
    const Tensor *t = c.t;
    const int64_t B = c.d.B, C = c.d.C, F = c.F;
    const Tensor &x = t[CM_X];
    OnDevice dev(x);
    Tensor scratch = at::empty({B * (F + C)}, x.options()), out = at::empty_like(x);
    at::BFloat16 *k = scratch.data_ptr<at::BFloat16>(), *r = k + B * F;
    const void *px = ptr(x), *ps = ptr(t[CM_SHIFT]);
    const wkv_rows_product proj[2] = {{ptr(t[CM_WK]), px, ps, ptr(t[CM_MIX_K]), nullptr, k, (int)F, 0, c.lerp, 1},
                                      {ptr(t[CM_WR]), px, ps, ptr(t[CM_MIX_R]), nullptr, r, (int)C, 0, c.lerp, 0}};
    check(abi.wkv_rows_products(dev.stream(), B, C, 2, proj), "wkv_rows_products");
    const wkv_rows_product last{ptr(t[CM_WV]), k, nullptr, nullptr, r, ptr(out), (int)C, 0, 0, 2};
    check(abi.wkv_rows_products(dev.stream(), B, F, 1, &last), "wkv_rows_products");
    return out;
}

// timemix(version, algo, module, x, (shift, state)) -> (out, (x[:, -1], new state)), or None: not a call for this way
PyObject *py_timemix(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 5);
    TimeMixCall c{};
    c.version = integer(a[0]);
    c.algo = integer(a[1]);
    if (!collect(c, a[2], a[3], a[4])) Py_RETURN_NONE;
    Tensor out, state, last;
    {
        NoLock no_lock;
        c.keep = at::GradMode::is_enabled() && any_requires_grad(c.t, c.version == 6 ? (int)N6 : (int)N5);
        if (c.keep) {
            const variable_list o = c.version == 6 ? apply_node<TimeMix<6>>(c, std::make_index_sequence<N6>()) : apply_node<TimeMix<5>>(c, std::make_index_sequence<N5>());
            out = o[0]; state = o[1];
        } else {
            at::AutoDispatchBelowADInplaceOrView below;
            if (single_tokens(c.d) && (c.version == 5 || c.t[DW1].size(1) == 64)) {
                std::tie(out, state) = timemix_decode(c);
            } else {
                TimeMixOut o = timemix_forward(c);
                out = o.out; state = o.state;
            }
        }
        last = c.t[X].select(1, c.d.T - 1);
    }
    PyObject *states = tuple(last, state);
    return Py_BuildValue("(NN)", wrapped(out), states);
    END_HANDLE_TH_ERRORS
}

// channelmix(version, module, x, shift) -> (out, x[:, -1]), or None
PyObject *py_channelmix(PyObject *, PyObject *const *a, Py_ssize_t n) {
    HANDLE_TH_ERRORS
    arity(n, 4);
    ChannelMixCall c{};
    c.lerp = integer(a[0]) == 5;
    if (!collect(c, a[1], a[2], a[3])) Py_RETURN_NONE;
    Tensor out, last;
    {
        NoLock no_lock;
        if (at::GradMode::is_enabled() && any_requires_grad(c.t, CM_N)) {
            out = ChannelMix::apply(&c, c.t[0], c.t[1], c.t[2], c.t[3], c.t[4], c.t[5], c.t[6])[0];
        } else {
            at::AutoDispatchBelowADInplaceOrView below;
            out = single_tokens(c.d) && c.F % 64 == 0 ? channelmix_decode(c) : channelmix_forward(c).out;
        }
        last = c.t[CM_X].select(1, c.d.T - 1);
    }
    return tuple(out, last);
    END_HANDLE_TH_ERRORS
}
