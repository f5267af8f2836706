// The layers' halves in native code: `timemix` and `channelmix` take a module that holds the reference's parameters under
// the reference's names and do what its forward does (RWKV-v5/src/module/TimeMix.py:286-323, ChannelMix.py:35-49;
// RWKV-v6/src/module/TimeMix.py:253-302, ChannelMix.py:30-37), each as two autograd nodes whose backwards are written
// out below.  As Python functions over a node per step a v6 layer's forward and backward took 1670 us of host time (45 nodes,
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

// The operands of a TimeMix, in the order of the inputs of its two autograd nodes: the front (token shift and mixes) and the back
// (from the mixed copies to the result)
enum { X, SHIFT, MIX0 };                                                                     // then the mixes: v5 k, v, r, g
enum { FRONT5 = MIX0 + 4, MAA_X = MIX0, MAA_W, MAA_K, MAA_V, MAA_R, MAA_G, W1, W2, FRONT6 };      // v6
enum { STATE, DECAY, U, LN_W, LN_B, WR, WK, WV, WG, WO, BACK5, DW1 = BACK5, DW2, BACK6 };
struct TimeMixCall {
    int version, algo;
    Dims d;
    float eps;
    Tensor f[FRONT6], b[BACK6];          // (handles of their own: the interpreter lock is given up after collecting them)
    Tensor coef;                         // fp32 rows: u, ln weight, ln bias, mixes
    bool keep;                           // a backward will follow
    int mixes() const { return version == 6 ? 6 : 4; }
    int front() const { return version == 6 ? (int)FRONT6 : (int)FRONT5; }
    int back() const { return version == 6 ? (int)BACK6 : (int)BACK5; }
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
    c.f[X] = x; c.f[SHIFT] = THPVariable_Unpack(sh); c.b[STATE] = THPVariable_Unpack(st);
    c.b[DECAY] = p.parameter(prm, "time_decay", C);
    c.b[U] = p.parameter(prm, "time_faaaa", C);
    c.b[LN_W] = p.parameter(item(lnd, "_parameters"), "weight", C);
    c.b[LN_B] = p.parameter(item(lnd, "_parameters"), "bias", C);
    const char *projections[5] = {"receptance", "key", "value", "gate", "output"};
    for (int j = 0; j < 5; j++) c.b[WR + j] = p.linear(mod, projections[j], C, C);
    if (c.version == 6) {
        const char *maa[6] = {"time_maa_x", "time_maa_w", "time_maa_k", "time_maa_v", "time_maa_r", "time_maa_g"};
        for (int j = 0; j < 6; j++) c.f[MAA_X + j] = p.parameter(prm, maa[j], C);
        c.f[W1] = p.matrix(prm, "time_maa_w1", C, 160);
        c.f[W2] = p.parameter(prm, "time_maa_w2", C * 160);
        p.ok = p.ok && c.f[W2].dim() == 3 && c.f[W2].size(0) == 5 && c.f[W2].size(1) == 32;
        PyObject *o = item(prm, "time_decay_w1");
        const int64_t D = o && THPVariable_Check(o) ? THPVariable_Unpack(o).numel() / C : 0;
        c.b[DW1] = p.matrix(prm, "time_decay_w1", C, D);
        c.b[DW2] = p.matrix(prm, "time_decay_w2", D, C);
    } else {
        const char *mix[4] = {"time_mix_k", "time_mix_v", "time_mix_r", "time_mix_g"};
        for (int j = 0; j < 4; j++) c.f[MIX0 + j] = p.parameter(prm, mix[j], C);
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

// Each half of a layer is two autograd nodes, not one: a node's saved tensors live until its backward is over, and with one node
// the front's buffers of gradients came on top of all that the back had saved (v6 layer, T 4096 H64: 1663 MB at the peak, with
// two 1238; as a node per step 1142).  In the forward, and in either backward, a tensor is let go as soon as the last reader
// has it (a prompt of that size: 452 MB when all were kept to the end, 323 now).

// ---- front: the mixed copies (n, B*T, C), v6 w, k, v, r, g; v5 k, v, r, g
enum { XXX, ACT, W2T, FRONT_SAVED };
struct FrontOut { Tensor mixes, saved[FRONT_SAVED]; };
FrontOut front_forward(const TimeMixCall &c) {
    const Dims &d = c.d;
    const Tensor *t = c.f;
    const int64_t M = d.B * (int64_t)d.T, C = d.C;
    OnDevice dev(t[X]);
    void *stream = dev.stream();
    const float *mix = fptr(c.coef) + 3 * C;
    FrontOut o;
    if (c.version == 5) {
        o.mixes = shift_mix(stream, d, 4, true, t[X], t[SHIFT], mix);
        return o;
    }
    Tensor xxx = shift_mix(stream, d, 1, false, t[X], t[SHIFT], mix).view({M, C});
    o.saved[ACT] = at::mm(xxx, t[W1]).tanh_();
    if (c.keep) o.saved[XXX] = xxx;
    xxx.reset();
    o.saved[W2T] = t[W2].transpose(1, 2).contiguous();
    o.mixes = at::empty({5, M, C}, t[X].options());
    check(abi.wkv_lora_mix_forward(stream, d.B, d.T, d.C, ptr(t[X]), ptr(t[SHIFT]), mix + C, ptr(o.saved[ACT]), ptr(o.saved[W2T]),
                                   Planes<5>(o.mixes).p), "wkv_lora_mix_forward");
    return o;
}
template <int VERSION> class Front : public torch::autograd::Function<Front<VERSION>> {
    static constexpr int N = VERSION == 6 ? (int)FRONT6 : (int)FRONT5;
public:
    template <class... Ts> static variable_list forward(AutogradContext *ctx, const TimeMixCall *c, const Ts &...ts) {
        static_assert(sizeof...(ts) == N, "one argument per operand");
        at::AutoDispatchBelowADInplaceOrView below;
        FrontOut o = front_forward(*c);
        ctx->set_materialize_grads(false);
        ctx->saved_data["call"] = std::vector<int64_t>{c->d.B, c->d.T, c->d.C, c->d.H};
        variable_list save{ts..., c->coef};
        save.insert(save.end(), o.saved, o.saved + FRONT_SAVED);
        ctx->save_for_backward(std::move(save));
        return {o.mixes};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list g(1 + N);
        if (!grads[0].defined()) return g;
        const std::vector<int64_t> c = ctx->saved_data["call"].toIntVector();
        const Dims d{(int)c[0], (int)c[1], (int)c[2], (int)c[3]};
        const int64_t M = d.B * (int64_t)d.T, C = d.C;
        const variable_list all = ctx->get_saved_variables();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor *t = all.data(), *s = all.data() + N + 1;
        OnDevice dev(t[X]);
        void *stream = dev.stream();
        const float *mix = fptr(all[N]) + 3 * C;
        auto out = [&](int i) -> Tensor & { return g[1 + i]; };
        auto wants = [&](int i) { return ctx->needs_input_grad(i); };
        Tensor gm = grads[0].contiguous();
        grads.clear();
        REQUIRE(gm.scalar_type() == at::kBFloat16);
        constexpr int MIXES = VERSION == 6 ? 6 : 4;
        const Tensor gcoef = at::empty({MIXES, C}, all[N].options());
        if (VERSION == 6) {
            Tensor gx = at::empty_like(t[X]), gshift = at::empty_like(t[SHIFT]), gdyn = at::empty({5, M, C}, t[X].options());
            {
                const Tensor ws = bytes(abi.wkv_lora_mix_backward_workspace(d.B, d.T, d.C), t[X]);
                check(abi.wkv_lora_mix_backward(stream, d.B, d.T, d.C, ptr(t[X]), ptr(t[SHIFT]), mix + C, ptr(s[ACT]), ptr(s[W2T]),
                                                Planes<5>(gm).p, ptr(gx), ptr(gshift), fptr(gcoef) + C, ptr(gdyn), ptr(ws), ws.numel()),
                      "wkv_lora_mix_backward");
            }
            gm.reset();
            // the two reductions of the second LoRA product's backward, and the first product
            Tensor ga = at::empty({M, 5, 32}, t[X].options());
            ga.copy_(at::bmm(gdyn, s[W2T]).transpose(0, 1));
            if (wants(W2)) out(W2) = at::bmm(s[ACT].view({M, 5, 32}).permute({1, 2, 0}), gdyn);
            gdyn.reset();
            const Tensor gpre = at::tanh_backward(ga.view({M, 160}), s[ACT]);
            if (wants(W1)) out(W1) = at::mm(s[XXX].t(), gpre);
            const MixGrads first = shift_mix_backward(stream, d, 1, false, t[X], t[SHIFT], mix, at::mm(gpre, t[W1].t()), fptr(gcoef));
            out(X) = gx.add_(first.gx);
            out(SHIFT) = gshift.add_(first.gshift);
        } else {
            const MixGrads first = shift_mix_backward(stream, d, 4, true, t[X], t[SHIFT], mix, gm, fptr(gcoef));
            out(X) = first.gx;
            out(SHIFT) = first.gshift;
        }
        const Tensor small = gcoef.to(at::kBFloat16);
        for (int j = 0; j < MIXES; j++) out(MIX0 + j) = small.select(0, j).view(t[MIX0 + j].sizes());
        return g;
    }
};

// ---- back: projections, operator, ln_x and gate, output.  What its backward needs, in the order in which it is saved after
// the operands
enum { COEF, MIXED, RR, KK, VV, GG, LORA, WW, YY, ZZ, WS, BACK_SAVED };
struct BackOut { Tensor out, state, saved[BACK_SAVED]; };
BackOut back_forward(const TimeMixCall &c, Tensor mixed) {
    const Dims &d = c.d;
    const Tensor *t = c.b;
    const int64_t M = d.B * (int64_t)d.T, C = d.C;
    const bool v6 = c.version == 6;
    OnDevice dev(mixed);
    void *stream = dev.stream();
    BackOut o;
    auto kept = [&](int i, const Tensor &x) -> const Tensor & { if (c.keep) o.saved[i] = x; return x; };
    const int64_t streams[3] = {d.B, d.T, d.C};
    auto seq = [&](const Tensor &x) { return x.view(at::IntArrayRef(streams, 3)); };
    const int at_k = v6 ? 1 : 0;
    Tensor r = kept(RR, times_t(plane(mixed, at_k + 2), t[WR])), k = kept(KK, times_t(plane(mixed, at_k), t[WK]));
    Tensor v = kept(VV, times_t(plane(mixed, at_k + 1), t[WV])), g = kept(GG, times_t(plane(mixed, at_k + 3), t[WG])), w;
    if (v6) {
        const Tensor lora = kept(LORA, at::mm(plane(mixed, 0), t[DW1]).tanh_());
        // the broadcast addition of time_decay rides on the product as its bias
        w = decay_operand(6, d, c.algo, seq(r), seq(at::addmm(t[DECAY].view({C}), lora, t[DW2])), c.keep);
    } else {
        w = t[DECAY].to(at::kFloat);
    }
    kept(WW, w);
    kept(COEF, c.coef);
    kept(MIXED, mixed);
    mixed.reset();
    Forward56 f = forward56(c.version, d, c.algo, seq(r), seq(k), seq(v), w, c.coef.select(0, 0), t[STATE], Tensor(), c.keep);
    for (Tensor *x : {&r, &k, &v, &w}) x->reset();
    kept(YY, f.y);
    kept(WS, f.ws);
    o.state = f.state;
    Tensor z = kept(ZZ, at::empty({M, C}, f.y.options()));
    check(abi.wkv_ln_gate_forward(stream, M, C, WKV_BF16, v6 ? 1.f : 0.125f, c.eps, ptr(f.y), ptr(g), fptr(c.coef) + C, fptr(c.coef) + 2 * C, ptr(z)),
          "wkv_ln_gate_forward");
    f.y.reset();
    g.reset();
    o.out = seq(times_t(z, t[WO]));
    return o;
}
template <int VERSION> class Back : public torch::autograd::Function<Back<VERSION>> {
    static constexpr int N = VERSION == 6 ? (int)BACK6 : (int)BACK5;          // operands; the mixed copies come after them
public:
    template <class... Ts> static variable_list forward(AutogradContext *ctx, const TimeMixCall *c, const Tensor &mixed, const Ts &...ts) {
        static_assert(sizeof...(ts) == N, "one argument per operand");
        at::AutoDispatchBelowADInplaceOrView below;
        BackOut o = back_forward(*c, mixed);
        ctx->set_materialize_grads(false);
        ctx->saved_data["call"] = std::vector<int64_t>{c->algo, c->d.B, c->d.T, c->d.C, c->d.H};
        ctx->saved_data["eps"] = (double)c->eps;
        variable_list save{ts...};
        save.insert(save.end(), o.saved, o.saved + BACK_SAVED);
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
        OnDevice dev(s[MIXED]);
        void *stream = dev.stream();
        const float *coef = fptr(s[COEF]);
        variable_list g(2 + N);
        auto out = [&](int i) -> Tensor & { return g[2 + i]; };
        auto wants = [&](int i) { return ctx->needs_input_grad(1 + i); };
        Tensor gout = grads[0].defined() ? grads[0].contiguous().view({M, C}) : at::zeros({M, C}, s[MIXED].options());
        REQUIRE(gout.scalar_type() == at::kBFloat16);
        const Tensor gstate = grads[1].defined() ? as_float(grads[1]).contiguous() : Tensor();
        grads.clear();
        // output projection, ln_x and gate
        Tensor gz = at::mm(gout, t[WO]);
        if (wants(WO)) out(WO) = at::mm(gout.t(), s[ZZ]);
        gout.reset();
        Tensor gy = at::empty_like(s[YY]), gg = at::empty_like(s[GG]);
        // fp32 gradients of the (C) parameters, rows of one conversion: u, ln weight, ln bias
        const Tensor gsmall = at::empty({3, C}, s[COEF].options());
        {
            const Tensor ws = bytes(abi.wkv_ln_gate_backward_workspace(M, C), gz);
            check(abi.wkv_ln_gate_backward(stream, M, C, WKV_BF16, VERSION == 6 ? 1.f : 0.125f, eps, ptr(s[YY]), ptr(s[GG]), coef + C, coef + 2 * C,
                                           ptr(gz), ptr(gy), ptr(gg), fptr(gsmall) + C, ptr(ws), ws.numel()), "wkv_ln_gate_backward");
        }
        gz.reset();
        // the operator
        const int64_t streams[3] = {d.B, d.T, d.C};
        auto seq = [&](const Tensor &x) { return x.view(at::IntArrayRef(streams, 3)); };
        Backward56 b = backward56(VERSION, d, algo, seq(s[RR]), seq(s[KK]), seq(s[VV]), s[WW], s[COEF].select(0, 0), t[STATE], gy, gstate, s[WS],
                                  wants(STATE), gsmall.select(0, 0));
        gy.reset();
        out(STATE) = b.gs;
        // gradients of the mixed copies (v6: w, k, v, r, g; v5: k, v, r, g) and of the projections
        constexpr int at_k = VERSION == 6 ? 1 : 0;
        const bool mixes = ctx->needs_input_grad(0);
        const Tensor gm = mixes ? at::empty_like(s[MIXED]) : Tensor();
        Tensor gproj[4] = {std::move(b.gk), std::move(b.gv), std::move(b.gr), std::move(gg)};
        const int weight[4] = {WK, WV, WR, WG};
        for (int j = 0; j < 4; j++) {
            const Tensor gp = gproj[j].view({M, C});
            gproj[j].reset();
            if (mixes) {
                Tensor into = plane(gm, at_k + j);
                at::mm_out(into, gp, t[weight[j]]);
            }
            if (wants(weight[j])) out(weight[j]) = at::mm(gp.t(), plane(s[MIXED], at_k + j));
        }
        if (VERSION == 6) {
            const Tensor gw = as_type(b.gw, at::kBFloat16).view({M, C});
            b.gw.reset();
            // (a product with ones: torch's sum over the rows takes scratch memory of sixteen times what it sums)
            if (wants(DECAY)) out(DECAY) = at::mm(at::ones({1, M}, gw.options()), gw).view(t[DECAY].sizes());
            if (wants(DW2)) out(DW2) = at::mm(s[LORA].t(), gw);
            const Tensor gl = at::tanh_backward(at::mm(gw, t[DW2].t()), s[LORA]);
            if (wants(DW1)) out(DW1) = at::mm(plane(s[MIXED], 0).t(), gl);
            if (mixes) {
                Tensor into = plane(gm, 0);
                at::mm_out(into, gl, t[DW1].t());
            }
        } else if (wants(DECAY)) {
            out(DECAY) = as_type(b.gw, at::kBFloat16).view(t[DECAY].sizes());
        }
        const Tensor small = gsmall.to(at::kBFloat16);
        const int rows[3] = {U, LN_W, LN_B};
        for (int j = 0; j < 3; j++) out(rows[j]) = small.select(0, j).view(t[rows[j]].sizes());
        g[1] = gm;
        return g;
    }
};
void widen(TimeMixCall &c) {
    const void *rows[9] = {ptr(c.b[U]), ptr(c.b[LN_W]), ptr(c.b[LN_B])};
    for (int j = 0; j < c.mixes(); j++) rows[3 + j] = ptr(c.f[MIX0 + j]);
    OnDevice dev(c.f[X]);
    c.coef = widen_rows(dev.stream(), c.f[X], rows, 3 + c.mixes(), c.d.C);
}
template <int VERSION, size_t... F, size_t... R> variable_list apply_nodes(const TimeMixCall &c, std::index_sequence<F...>, std::index_sequence<R...>) {
    const Tensor mixed = Front<VERSION>::apply(&c, c.f[F]...)[0];
    return Back<VERSION>::apply(&c, mixed, c.b[R]...);
}

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
// front: the two mixed copies and their projections k (B*T, F), r (B*T, C)
struct ChannelFront { Tensor k, r, coef, mixed; };
ChannelFront channel_front(const ChannelMixCall &c) {
    const Dims &d = c.d;
    const Tensor *t = c.t;
    OnDevice dev(t[CM_X]);
    void *stream = dev.stream();
    ChannelFront o;
    const void *rows[2] = {ptr(t[CM_MIX_K]), ptr(t[CM_MIX_R])};
    o.coef = widen_rows(stream, t[CM_X], rows, 2, d.C);
    o.mixed = shift_mix(stream, d, 2, c.lerp, t[CM_X], t[CM_SHIFT], fptr(o.coef));
    o.k = times_t(plane(o.mixed, 0), t[CM_WK]);
    o.r = times_t(plane(o.mixed, 1), t[CM_WR]);
    return o;
}
class ChannelFrontNode : public torch::autograd::Function<ChannelFrontNode> {
    enum { N = CM_WR + 1 };
public:
    static variable_list forward(AutogradContext *ctx, const ChannelMixCall *c, const Tensor &x, const Tensor &shift, const Tensor &mix_k,
                                 const Tensor &mix_r, const Tensor &wk, const Tensor &wr) {
        at::AutoDispatchBelowADInplaceOrView below;
        const ChannelFront o = channel_front(*c);
        ctx->set_materialize_grads(false);
        ctx->saved_data["call"] = std::vector<int64_t>{c->lerp, c->d.B, c->d.T, c->d.C};
        ctx->save_for_backward({x, shift, mix_k, mix_r, wk, wr, o.coef, o.mixed});
        return {o.k, o.r};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list g(1 + N);
        if (!grads[0].defined() && !grads[1].defined()) return g;
        const std::vector<int64_t> c = ctx->saved_data["call"].toIntVector();
        const Dims d{(int)c[1], (int)c[2], (int)c[3], (int)(c[3] / 64)};
        const variable_list t = ctx->get_saved_variables();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor &coef = t[N], &mixed = t[N + 1];
        OnDevice dev(t[CM_X]);
        auto wants = [&](int i) { return ctx->needs_input_grad(i); };
        const Tensor gm = at::empty_like(mixed);
        for (int j = 0; j < 2; j++) {          // k, r
            Tensor into = plane(gm, j);
            if (!grads[j].defined()) { into.zero_(); continue; }
            const Tensor gp = grads[j].contiguous();
            grads[j].reset();
            REQUIRE(gp.scalar_type() == at::kBFloat16);
            at::mm_out(into, gp, t[CM_WK + j]);
            if (wants(CM_WK + j)) g[1 + CM_WK + j] = at::mm(gp.t(), plane(mixed, j));
        }
        const Tensor gcoef = at::empty_like(coef);
        const MixGrads m = shift_mix_backward(dev.stream(), d, 2, c[0], t[CM_X], t[CM_SHIFT], fptr(coef), gm, fptr(gcoef));
        g[1 + CM_X] = m.gx;
        g[1 + CM_SHIFT] = m.gshift;
        const Tensor small = gcoef.to(at::kBFloat16);
        g[1 + CM_MIX_K] = small.select(0, 0).view(t[CM_MIX_K].sizes());
        g[1 + CM_MIX_R] = small.select(0, 1).view(t[CM_MIX_R].sizes());
        return g;
    }
};
// back: out = sigmoid(r) * (relu(k)^2 W^T).  k is let go with the caller's handle
struct ChannelBack { Tensor out, k2, kv; };
ChannelBack channel_back(const Tensor &x, Tensor k, const Tensor &r, const Tensor &wv) {
    OnDevice dev(x);
    ChannelBack o;
    o.k2 = at::empty_like(k);
    check(abi.wkv_relu_square_forward(dev.stream(), k.numel(), WKV_BF16, ptr(k), ptr(o.k2)), "wkv_relu_square_forward");
    k.reset();
    o.kv = times_t(o.k2, wv);
    o.out = at::empty_like(x);
    check(abi.wkv_sigmoid_mul_forward(dev.stream(), r.numel(), WKV_BF16, ptr(r), ptr(o.kv), ptr(o.out)), "wkv_sigmoid_mul_forward");
    return o;
}
class ChannelBackNode : public torch::autograd::Function<ChannelBackNode> {
public:
    static variable_list forward(AutogradContext *ctx, const ChannelMixCall *c, const Tensor &k, const Tensor &r, const Tensor &wv) {
        at::AutoDispatchBelowADInplaceOrView below;
        const ChannelBack o = channel_back(c->t[CM_X], k, r, wv);
        ctx->set_materialize_grads(false);
        ctx->save_for_backward({k, r, wv, o.k2, o.kv});
        return {o.out};
    }
    static variable_list backward(AutogradContext *ctx, variable_list grads) {
        variable_list g(4);
        if (!grads[0].defined()) return g;
        const variable_list x = ctx->get_saved_variables();
        at::AutoDispatchBelowADInplaceOrView below;
        const Tensor &k = x[0], &r = x[1], &wv = x[2], &k2 = x[3], &kv = x[4];
        OnDevice dev(k);
        void *stream = dev.stream();
        Tensor gout = grads[0].contiguous(), gkv = at::empty_like(kv);
        grads.clear();
        REQUIRE(gout.scalar_type() == at::kBFloat16);
        g[2] = at::empty_like(r);
        check(abi.wkv_sigmoid_mul_backward(stream, r.numel(), WKV_BF16, ptr(r), ptr(kv), ptr(gout), ptr(g[2]), ptr(gkv)), "wkv_sigmoid_mul_backward");
        gout.reset();
        {
            const Tensor gk2 = at::mm(gkv, wv);
            g[1] = at::empty_like(gk2);
            check(abi.wkv_relu_square_backward(stream, k.numel(), WKV_BF16, ptr(k), ptr(gk2), ptr(g[1])), "wkv_relu_square_backward");
        }
        if (ctx->needs_input_grad(2)) g[3] = at::mm(gkv.t(), k2);
        return g;
    }
};
Tensor channelmix_forward(const ChannelMixCall &c) {          // nothing recorded
    ChannelFront f = channel_front(c);
    f.mixed.reset();
    return channel_back(c.t[CM_X], std::move(f.k), f.r, c.t[CM_WV]).out;
}

// ---- one token per sequence, nothing recorded (csrc/layer_decode.hip)
bool single_tokens(const Dims &d) { return d.T == 1 && d.B <= 64; }
std::pair<Tensor, Tensor> timemix_decode(const TimeMixCall &c) {
    const Tensor *f = c.f, *t = c.b;
    const int64_t B = c.d.B, C = c.d.C, rows = B * C;
    const Tensor &x = f[X];
    const bool v6 = c.version == 6;
    OnDevice dev(x);
    void *stream = dev.stream();
    // scratch: r, k, v, gate, the head results; v6 also the five mixes and the two LoRAs' activations
    constexpr int64_t parts = 2 * WKV_LORA_PARTS;          // (fp32 counted in bf16)
    Tensor scratch = at::empty({(v6 ? 10 : 5) * rows + (v6 ? parts * B * 224 : 0)}, x.options());
    at::BFloat16 *q = scratch.data_ptr<at::BFloat16>();
    at::BFloat16 *r = q, *k = r + rows, *v = k + rows, *g = v + rows, *z = g + rows, *mixes = z + rows, *act = mixes + 5 * rows, *lora = act + parts * B * 160;
    Tensor out = at::empty_like(x), state = at::empty_like(t[STATE]);
    const void *px = ptr(x), *ps = ptr(f[SHIFT]), *wr = ptr(t[WR]), *wk = ptr(t[WK]), *wv = ptr(t[WV]), *wg = ptr(t[WG]);
    const int n = (int)C;
    if (v6) {
        const void *maa[5];
        for (int j = 0; j < 5; j++) maa[j] = ptr(f[MAA_W + j]);
        const wkv_rows_product first{ptr(f[W1]), px, ps, ptr(f[MAA_X]), nullptr, act, 160, 1, 0, 0};
        check(abi.wkv_rows_products(stream, B, C, 1, &first), "wkv_rows_products");
        check(abi.wkv_lora_mix_rows(stream, B, C, px, ps, maa, act, ptr(f[W2]), mixes), "wkv_lora_mix_rows");
        const wkv_rows_product proj[5] = {{ptr(t[DW1]), mixes, nullptr, nullptr, nullptr, lora, 64, 1, 0, 0},
                                          {wk, mixes + rows, nullptr, nullptr, nullptr, k, n, 0, 0, 0},
                                          {wv, mixes + 2 * rows, nullptr, nullptr, nullptr, v, n, 0, 0, 0},
                                          {wr, mixes + 3 * rows, nullptr, nullptr, nullptr, r, n, 0, 0, 0},
                                          {wg, mixes + 4 * rows, nullptr, nullptr, nullptr, g, n, 0, 0, 0}};
        check(abi.wkv_rows_products(stream, B, C, 5, proj), "wkv_rows_products");
    } else {
        const wkv_rows_product proj[4] = {{wk, px, ps, ptr(f[MIX0]), nullptr, k, n, 0, 1, 0}, {wv, px, ps, ptr(f[MIX0 + 1]), nullptr, v, n, 0, 1, 0},
                                          {wr, px, ps, ptr(f[MIX0 + 2]), nullptr, r, n, 0, 1, 0}, {wg, px, ps, ptr(f[MIX0 + 3]), nullptr, g, n, 0, 1, 0}};
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
        c.keep = at::GradMode::is_enabled() && (any_requires_grad(c.f, c.front()) || any_requires_grad(c.b, c.back()));
        if (c.keep) {
            widen(c);
            const variable_list o = c.version == 6 ? apply_nodes<6>(c, std::make_index_sequence<FRONT6>(), std::make_index_sequence<BACK6>())
                                                   : apply_nodes<5>(c, std::make_index_sequence<FRONT5>(), std::make_index_sequence<BACK5>());
            out = o[0]; state = o[1];
        } else {
            at::AutoDispatchBelowADInplaceOrView below;
            if (single_tokens(c.d) && (c.version == 5 || c.b[DW1].size(1) == 64)) {
                std::tie(out, state) = timemix_decode(c);
            } else {
                widen(c);
                const BackOut o = back_forward(c, front_forward(c).mixes);
                out = o.out; state = o.state;
            }
        }
        last = c.f[X].select(1, c.d.T - 1);
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
            const variable_list kr = ChannelFrontNode::apply(&c, c.t[CM_X], c.t[CM_SHIFT], c.t[CM_MIX_K], c.t[CM_MIX_R], c.t[CM_WK], c.t[CM_WR]);
            out = ChannelBackNode::apply(&c, kr[0], kr[1], c.t[CM_WV])[0];
        } else {
            at::AutoDispatchBelowADInplaceOrView below;
            out = single_tokens(c.d) && c.F % 64 == 0 ? channelmix_decode(c) : channelmix_forward(c);
        }
        last = c.t[CM_X].select(1, c.d.T - 1);
    }
    return tuple(out, last);
    END_HANDLE_TH_ERRORS
}
