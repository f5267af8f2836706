"""The element-wise passes around the operator (token shift + mixing, ln_x * gate, channel-mix activations, L2Wrap)
on the HIP kernels, through the C ABI, against the CPU oracle (oracle/blocks.py: the reference's lines in plain torch,
gradients by autograd).  Tolerances: rtol 1e-3 for fp32 tensors, 2e-2 for bf16 / fp16 (of |ref| + rms(ref))."""
import copy

import pytest
import torch

from oracle import blocks as OB
from oracle import wkv56 as O
from oracle.timemix_restated import ChannelMix5, ChannelMix6, TimeMix5, TimeMix6
from tests.util import assert_close

pytestmark = pytest.mark.gpu
RTOL = {torch.float32: 1e-3, torch.bfloat16: 2e-2, torch.float16: 2e-2}


def _g(seed):
    return torch.Generator().manual_seed(seed)


def _leaf(t):
    return t.clone().requires_grad_(True)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("B,T,C", [(1, 1, 64), (2, 7, 264), (3, 130, 64), (2, 64, 2560), (1, 200, 320)])
@pytest.mark.parametrize("n,lerp,dyn", [(1, False, False), (2, True, False), (4, True, False), (2, False, False),
                                        (5, False, True), (3, False, True)])
def test_token_shift_mix(dtype, B, T, C, n, lerp, dyn):
    from rwkv_wkv_hip import blocks as K
    g = _g(B * 1000 + T + C + n)
    x = torch.randn(B, T, C, generator=g).to(dtype)
    shift = torch.randn(B, C, generator=g).to(dtype)
    coefs = [torch.rand(1, 1, C, generator=g) for _ in range(n)]
    d = (torch.randn(n, B, T, C, generator=g) * 0.3).to(dtype) if dyn else None
    gouts = [torch.randn(B, T, C, generator=g).to(dtype) for _ in range(n)]

    def run(fn, dev):
        xs, ss = _leaf(x.to(dev)), _leaf(shift.to(dev))
        cs = [_leaf(c.to(dev)) for c in coefs]
        ds = _leaf(d.to(dev)) if dyn else None
        outs = fn(xs, ss, cs, ds)
        torch.autograd.backward(list(outs), [go.to(dev) for go in gouts])
        return outs, xs.grad, ss.grad, [c.grad for c in cs], (ds.grad if dyn else None)

    # the oracle computes in fp32 from the same (already rounded) inputs
    def ref_fn(xs, ss, cs, ds):
        xf, sf = xs.float(), ss.float()
        return OB.mix_v5(xf, sf, cs) if lerp else OB.mix_v6(xf, sf, cs, None if ds is None else ds.float())
    ref = run(ref_fn, "cpu")
    got = run(lambda xs, ss, cs, ds: K.token_shift_mix(xs, ss, cs, dyn=ds, lerp=lerp), "cuda")
    torch.cuda.synchronize()
    rt = RTOL[dtype]
    for j in range(n):
        assert got[0][j].dtype == dtype
        assert_close(got[0][j], ref[0][j], rt, f"out[{j}]")
        assert_close(got[3][j], ref[3][j], max(rt, 2e-3) if dtype == torch.float32 else rt, f"gcoef[{j}]")
    assert_close(got[1], ref[1], rt, "gx")
    assert_close(got[2], ref[2], rt, "gshift")
    if dyn:
        assert_close(got[4], ref[4], rt, "gdyn")


@pytest.mark.parametrize("B,T,C", [(1, 1, 32), (2, 7, 96), (3, 130, 64), (2, 128, 2560), (1, 200, 320), (2, 129, 32),
                                   (1, 257, 128), (2, 16, 4096), (3, 300, 72), (1, 65, 8), (2, 1, 200), (1, 513, 136)])
def test_lora_shift_mix(B, T, C):
    """The five data-dependent mixes with the second LoRA product inside the kernel (bf16) against the oracle in fp32
    on the same rounded inputs: the five outputs and the gradients of x, the shift state, the five time_maa
    parameters, the activations and time_maa_w2."""
    from rwkv_wkv_hip import blocks as K
    bf = torch.bfloat16
    g = _g(B * 1000 + T + C)
    x = torch.randn(B, T, C, generator=g).to(bf)
    shift = torch.randn(B, C, generator=g).to(bf)
    coefs = [torch.rand(1, 1, C, generator=g) for _ in range(5)]
    act = torch.tanh(torch.randn(B * T, 5, 32, generator=g)).to(bf)
    w2 = (torch.randn(5, 32, C, generator=g) * 0.1).to(bf)
    gouts = [torch.randn(B, T, C, generator=g).to(bf) for _ in range(5)]

    def run(fn, dev):
        xs, ss, as_, ws = (_leaf(t.to(dev)) for t in (x, shift, act, w2))
        cs = [_leaf(c.to(dev)) for c in coefs]
        outs = fn(xs, ss, cs, as_, ws)
        torch.autograd.backward(list(outs), [go.to(dev).to(outs[0].dtype) for go in gouts])
        return outs, xs.grad, ss.grad, [c.grad for c in cs], as_.grad, ws.grad

    ref = run(lambda xs, ss, cs, as_, ws: OB.lora_mix_v6(xs.float(), ss.float(), cs, as_.float(), ws.float()), "cpu")
    assert K.lora_mix_available(x, act, w2)
    got = run(lambda xs, ss, cs, as_, ws: K.lora_shift_mix(xs, ss, cs, as_, ws), "cuda")
    torch.cuda.synchronize()
    for j in range(5):
        assert got[0][j].dtype == bf
        assert_close(got[0][j], ref[0][j], 2e-2, f"out[{j}]")
        assert_close(got[3][j], ref[3][j], 2e-2, f"gmaa[{j}]")
    assert_close(got[1], ref[1], 2e-2, "gx")
    assert_close(got[2], ref[2], 2e-2, "gshift")
    assert_close(got[4], ref[4], 2e-2, "gact")
    assert_close(got[5], ref[5], 2e-2, "gw2")


def test_lora_shift_mix_matches_the_unfused_passes():
    """the fused pass against bmm + token_shift_mix on the same device: the same mathematics with dyn rounded to bf16
    on its way through memory in the one and kept in fp32 in the other"""
    from rwkv_wkv_hip import blocks as K
    bf = torch.bfloat16
    B, T, C = 2, 200, 256
    g = _g(5)
    x, shift = torch.randn(B, T, C, generator=g).to(bf).cuda(), torch.randn(B, C, generator=g).to(bf).cuda()
    coefs = [torch.rand(1, 1, C, generator=g).cuda() for _ in range(5)]
    act = torch.tanh(torch.randn(B * T, 5, 32, generator=g)).to(bf).cuda()
    w2 = (torch.randn(5, 32, C, generator=g) * 0.1).to(bf).cuda()
    with torch.no_grad():
        fused = K.lora_shift_mix(x, shift, coefs, act, w2)
        dyn = torch.bmm(act.transpose(0, 1), w2).view(5, B, T, C)
        plain = K.token_shift_mix(x, shift, coefs, dyn=dyn)
    for j in range(5):
        assert_close(fused[j], plain[j].float().cpu(), 2e-2, f"out[{j}]")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,C", [(1, 64), (9, 320), (130, 128), (64, 2560), (257, 4096)])
@pytest.mark.parametrize("divisor,eps,gated", [(8.0, 1e-5, True), (1.0, 64e-5, True), (1.0, 1e-5, False)])
def test_ln_x_gate(dtype, rows, C, divisor, eps, gated):
    from rwkv_wkv_hip import blocks as K
    g = _g(rows + C)
    y = (torch.randn(rows, C, generator=g) * 3 + 0.5).to(dtype)
    gate = torch.randn(rows, C, generator=g).to(dtype) if gated else None
    w, b = torch.randn(C, generator=g), torch.randn(C, generator=g)
    go = torch.randn(rows, C, generator=g).to(dtype)

    def run(fn, dev):
        ys, ws, bs = _leaf(y.to(dev)), _leaf(w.to(dev)), _leaf(b.to(dev))
        gs = _leaf(gate.to(dev)) if gated else None
        out = fn(ys, gs, ws, bs)
        out.backward(go.to(dev).to(out.dtype))
        return out, ys.grad, (gs.grad if gated else None), ws.grad, bs.grad
    ref = run(lambda ys, gs, ws, bs: OB.ln_x_gate(ys.float(), None if gs is None else gs.float(), ws, bs, C // 64, eps, divisor), "cpu")
    got = run(lambda ys, gs, ws, bs: K.ln_x_gate(ys, gs, ws, bs, eps, scale=1.0 / divisor), "cuda")
    torch.cuda.synchronize()
    rt = RTOL[dtype]
    assert got[0].dtype == dtype
    assert_close(got[0], ref[0], rt, "out")
    assert_close(got[1], ref[1], rt, "gy")
    if gated:
        assert_close(got[2], ref[2], rt, "ggate")
    assert_close(got[3], ref[3], max(rt, 2e-3), "gweight")
    assert_close(got[4], ref[4], max(rt, 2e-3), "gbias")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("shape", [(1, 1, 8), (2, 7, 264), (2, 128, 8960)])
def test_channel_mix_activations(dtype, shape):
    from rwkv_wkv_hip import blocks as K
    g = _g(sum(shape))
    k, kv, go = (torch.randn(*shape, generator=g).to(dtype) for _ in range(3))

    def run(mod, dev, f32):
        cast = (lambda t: t.float()) if f32 else (lambda t: t)
        ks, rs, kvs = _leaf(k.to(dev)), _leaf(k.to(dev)), _leaf(kv.to(dev))
        a = mod.relu_square(cast(ks))
        b = mod.sigmoid_mul(cast(rs), cast(kvs))
        torch.autograd.backward([a, b], [go.to(dev).to(a.dtype), go.to(dev).to(b.dtype)])
        return a, b, ks.grad, rs.grad, kvs.grad
    ref, got = run(OB, "cpu", True), run(K, "cuda", False)
    torch.cuda.synchronize()
    for name, a, b in zip(("relu^2", "sigmoid*kv", "gk", "gr", "gkv"), got, ref):
        assert a.dtype == dtype
        assert_close(a, b, RTOL[dtype], name)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("B,T,V", [(1, 1, 8), (2, 5, 50277), (2, 3, 65536)])
def test_l2wrap(dtype, B, T, V):
    """bf16 logits tie often: the kernel, like torch on the CPU, takes the first position of the maximum."""
    from rwkv_wkv_hip import blocks as K
    g = _g(V)
    y = torch.randn(B, T, V, generator=g).to(dtype)
    y[0, 0, V // 2] = y[0, 0, V - 1] = 9.0                        # a forced tie
    mask = (torch.rand(B, T, generator=g) > 0.3).float()
    factor = 1e-4 / (B * T)

    def run(mod, dev):
        ys = _leaf(y.to(dev))
        loss = ys.float().sum() * 0 + 2.0
        mod.L2Wrap.apply(loss, ys, factor, mask.to(dev)).backward()
        return ys.grad
    ref, got = run(OB, "cpu"), run(K, "cuda")
    torch.cuda.synchronize()
    assert got.dtype == dtype
    assert torch.equal((got != 0).cpu(), ref != 0), "position of the maximum"
    assert_close(got, ref, RTOL[dtype], "gy")


def _run_module(fwd, mod, x, state, gy, extra_grads=()):
    mod.zero_grad()
    x = x.clone().requires_grad_(True)
    state = tuple(s.clone().requires_grad_(True) for s in state) if isinstance(state, tuple) else state.clone().requires_grad_(True)
    y, new = fwd(mod, x, state)
    outs, gs = [y], [gy]
    if isinstance(new, tuple):
        outs.append(new[1]); gs.append(torch.ones_like(new[1]) * 0.1)
    torch.autograd.backward(outs, gs)
    grads = {n: p.grad.detach().float().cpu() for n, p in mod.named_parameters() if p.grad is not None}
    sg = state[0].grad if isinstance(state, tuple) else state.grad
    return y.detach(), x.grad.detach(), sg.detach(), grads


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("T", [128, 72])
def test_timemix_forward_on_the_kernels(version, T):
    """timemix5_forward / timemix6_forward (every element-wise pass and the operator on HIP kernels) against the
    restated reference module on the CPU oracle: output, input / shift-state gradients and every parameter gradient."""
    from rwkv_wkv_hip import blocks as K
    B, C, H = 2, 128, 2
    g = _g(11)
    x, shift, gy = torch.randn(B, T, C, generator=g), torch.randn(B, C, generator=g), torch.randn(B, T, C, generator=g)
    state = torch.randn(B, H, 64, 64, generator=g) * 0.1
    cpu = (TimeMix5 if version == 5 else TimeMix6)(C, H, seed=5)
    with torch.no_grad():
        cpu.ln_x.weight.copy_(torch.randn(C, generator=g)); cpu.ln_x.bias.copy_(torch.randn(C, generator=g))
    gpu = copy.deepcopy(cpu).cuda()
    if version == 5:
        ref_fwd = lambda m, xs, st: m(xs, st, lambda B, T, C, H, s, r, k, v, w, u: O.wkv5_op(B, T, C, H, s, r, k, v, w, u))
        our_fwd = K.timemix5_forward
    else:
        ref_fwd = lambda m, xs, st: m(xs, st, lambda B, T, C, H, r, k, v, w, u, s: O.wkv6_op(B, T, C, H, r, k, v, w, u, s))
        our_fwd = K.timemix6_forward
    ref = _run_module(ref_fwd, cpu, x, (shift, state), gy)
    got = _run_module(our_fwd, gpu, x.cuda(), (shift.cuda(), state.cuda()), gy.cuda())
    torch.cuda.synchronize()
    for name, a, b in zip(("y", "gx", "gshift"), got[:3], ref[:3]):
        assert_close(a, b, 2e-3, f"timemix v{version} {name}")
    assert set(got[3]) == set(ref[3])
    for n in ref[3]:
        assert_close(got[3][n], ref[3][n], 3e-3, f"timemix v{version} grad {n}")


@pytest.mark.parametrize("version", [5, 6])
def test_timemix_forward_on_the_kernels_bf16_module(version):
    """The whole module in bf16 (weights, matmuls, every element-wise pass), as mixed-precision training runs it, against
    the fp32 CPU module: compared in norm (the matmuls round too); the carried state, which only the operator touches and
    which stays fp32, element-wise."""
    from rwkv_wkv_hip import blocks as K
    B, T, C, H = 2, 128, 128, 2
    g = _g(13)
    x, shift = torch.randn(B, T, C, generator=g), torch.randn(B, C, generator=g)
    state = torch.randn(B, H, 64, 64, generator=g) * 0.1
    gy = torch.randn(B, T, C, generator=g)
    cpu = (TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8)
    gpu = copy.deepcopy(cpu).cuda().bfloat16()
    if version == 5:
        ref_fwd = lambda m, xs, st: m(xs, st, lambda B, T, C, H, s, r, k, v, w, u: O.wkv5_op(B, T, C, H, s, r, k, v, w, u))
        our_fwd = K.timemix5_forward
    else:
        ref_fwd = lambda m, xs, st: m(xs, st, lambda B, T, C, H, r, k, v, w, u, s: O.wkv6_op(B, T, C, H, r, k, v, w, u, s))
        our_fwd = K.timemix6_forward
    ref = _run_module(ref_fwd, cpu, x, (shift, state), gy)
    got = _run_module(our_fwd, gpu, x.cuda().bfloat16(), (shift.cuda().bfloat16(), state.cuda()), gy.cuda().bfloat16())
    torch.cuda.synchronize()
    assert got[0].dtype == torch.bfloat16
    for name, a, b in zip(("y", "gx", "gshift"), got[:3], ref[:3]):
        rel = ((a.float().cpu() - b).norm() / b.norm()).item()
        assert rel < 4e-2, f"timemix bf16 v{version} {name}: relative error {rel}"
    for n in ref[3]:
        a, b = got[3][n], ref[3][n]
        rel = ((a - b).norm() / (b.norm() + 1e-6)).item()
        assert rel < 8e-2, f"timemix bf16 v{version} grad {n}: relative error {rel}"
    with torch.no_grad():
        _, (_, s_ref) = ref_fwd(cpu, x, (shift, state))
        _, (_, s_got) = our_fwd(gpu, x.cuda().bfloat16(), (shift.cuda().bfloat16(), state.cuda()))
    assert s_got.dtype == torch.float32
    assert_close(s_got, s_ref, 6e-2, f"timemix bf16 v{version} state")


@pytest.mark.parametrize("rows", [1, 2, 3, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,K", [(256, 64), (1024, 192), (2080, 320), (4128, 192), (8224, 2112), (16416, 64)])
def test_products_of_a_few_rows(rows, n, K):
    """Each shape of the kernel: 8, 16 and 32 columns, four and eight wavefronts, one to four tiles of rows, contractions that
    end inside a segment; two products in one launch, one mixed and squared, one (n + 32 columns) as it is.  Against 64 bits:
    the mixed row and the result round to bf16 (2^-9 each, the square doubles it), the sums to 32 bits."""
    import ctypes
    from rwkv_wkv_hip import _lib

    class Product(ctypes.Structure):
        _fields_ = [(f, ctypes.c_void_p) for f in ("w", "x", "shift", "mix", "mul", "out")] + [(f, ctypes.c_int) for f in ("n", "k_major", "lerp", "act")]
    g = torch.Generator().manual_seed(rows + n)
    r = lambda *shape: torch.randn(*shape, generator=g).bfloat16().cuda()
    x, shift, mix, w1, w2 = r(rows, K), r(rows, K), torch.rand(K, generator=g).bfloat16().cuda(), r(n, K), r(n + 32, K)
    o1, o2 = torch.full((rows, n), 9.0, dtype=torch.bfloat16, device="cuda"), torch.full((rows, n + 32), 9.0, dtype=torch.bfloat16, device="cuda")
    p = lambda t: t.data_ptr()
    jobs = (Product * 2)(Product(p(w1), p(x), p(shift), p(mix), None, p(o1), n, 0, 0, 1), Product(p(w2), p(x), None, None, None, p(o2), n + 32, 0, 0, 0))
    assert _lib.lib().wkv_rows_products(torch.cuda.current_stream().cuda_stream, rows, K, 2, jobs) == 0
    torch.cuda.synchronize()
    d = lambda t: t.double()
    mixed = (d(x) + (d(shift) - d(x)) * d(mix)).bfloat16()
    e1, e2 = torch.relu(d(mixed) @ d(w1).t()) ** 2, d(x) @ d(w2).t()
    for got, want, tol in ((o1, e1, 3 * 2 ** -8), (o2, e2, 2 ** -8)):
        err = (d(got) - want).abs()
        assert bool((err <= tol * want.abs() + 2 ** -9 * want.pow(2).mean().sqrt()).all()), err.max().item()


@pytest.mark.parametrize("rows", [1, 2, 3, 16, 17, 32, 33, 64])
@pytest.mark.parametrize("n,K", [(1024, 192), (4096, 2048), (8192, 64)])
def test_products_of_a_few_rows_of_every_kind(rows, n, K):
    """Every kind of job in one launch, in the shapes that each number of workgroups gives it: weights kept [k][n] (mixed and
    not; the sum of their parts), a mix with 1 - mix, and a product behind its gate.  Against 64 bits: an fp32 sum of K terms is
    off by at most K 2^-24 of the sum of their sizes, one element of the mixed row may round to the neighbouring bf16 (2^-7), the result
    rounds to bf16 before and after the gate (eight significant bits: 2^-8 each; the gate's own error, 2^-20, is lost in them)."""
    import ctypes
    from rwkv_wkv_hip import _lib

    class Product(ctypes.Structure):
        _fields_ = [(f, ctypes.c_void_p) for f in ("w", "x", "shift", "mix", "mul", "out")] + [(f, ctypes.c_int) for f in ("n", "k_major", "lerp", "act")]
    g = torch.Generator().manual_seed(rows + n)
    r = lambda *shape: torch.randn(*shape, generator=g).bfloat16().cuda()
    x, shift, mix, mul = r(rows, K), r(rows, K), torch.rand(K, generator=g).bfloat16().cuda(), r(rows, n)
    wa, wb, wc, wd = r(K, 160), r(K, 64), r(n, K), r(n, K)
    oa, ob = (torch.full((8, rows, m), 9.0, device="cuda") for m in (160, 64))
    oc, od = (torch.full((rows, n), 9.0, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    p = lambda t: t.data_ptr()
    jobs = (Product * 4)(Product(p(wa), p(x), p(shift), p(mix), None, p(oa), 160, 1, 0, 0), Product(p(wb), p(x), None, None, None, p(ob), 64, 1, 0, 0),
                         Product(p(wc), p(x), p(shift), p(mix), None, p(oc), n, 0, 1, 0), Product(p(wd), p(x), None, None, p(mul), p(od), n, 0, 0, 2))
    assert _lib.lib().wkv_rows_products(torch.cuda.current_stream().cuda_stream, rows, K, 4, jobs) == 0
    torch.cuda.synchronize()
    d = lambda t: t.double()
    mixed = (d(x) + (d(shift) - d(x)) * d(mix)).bfloat16()
    lerped = (d(x) + (d(shift) - d(x)) * (1 - d(mix))).bfloat16()
    for name, got, a, w, rounding in (("k major, mixed", d(oa).sum(0), mixed, wa, 0), ("k major", d(ob).sum(0), x, wb, 0), ("lerp", d(oc), lerped, wc.t(), 2 ** -8),
                                      ("gated", d(od), x, wd.t(), 2 * 2 ** -8)):
        want, sizes = d(a) @ d(w), d(a).abs() @ d(w).abs()
        bound = K * 2 ** -24 * sizes + (2 ** -7 * d(a).abs().amax(1, keepdim=True) * d(w).abs().amax(0) if a is not x else 0)
        if name == "gated":
            want, bound = torch.sigmoid(d(mul)) * want, torch.sigmoid(d(mul)) * bound
        err = (got - want).abs() - bound - 1.01 * rounding * want.abs()
        assert bool((err <= 0).all()), (name, err.max().item())


@pytest.mark.parametrize("rows", [1, 5, 20, 40])
@pytest.mark.parametrize("count", [1, 7, 8])
def test_products_of_a_few_rows_find_their_job(rows, count):
    """As many jobs as a launch takes, down to a single workgroup each (16 columns; a [k][n] one among them): every workgroup
    finds its own.  Against 64 bits: the result rounds to bf16 (2^-8 of eight significant bits), fp32 sums of K terms."""
    import ctypes
    from rwkv_wkv_hip import _lib

    class Product(ctypes.Structure):
        _fields_ = [(f, ctypes.c_void_p) for f in ("w", "x", "shift", "mix", "mul", "out")] + [(f, ctypes.c_int) for f in ("n", "k_major", "lerp", "act")]
    K, g = 256, torch.Generator().manual_seed(rows + count)
    x = torch.randn(rows, K, generator=g).bfloat16().cuda()
    ns, k_major = [16, 48, 16, 32, 160, 16, 64, 16][:count], [int(i == 4) for i in range(count)]
    ws = [torch.randn(*((K, n) if kk else (n, K)), generator=g).bfloat16().cuda() for n, kk in zip(ns, k_major)]
    outs = [torch.full((8, rows, n), 9.0, device="cuda") if kk else torch.full((rows, n), 9.0, dtype=torch.bfloat16, device="cuda") for n, kk in zip(ns, k_major)]
    jobs = (Product * count)(*(Product(w.data_ptr(), x.data_ptr(), None, None, None, o.data_ptr(), n, kk, 0, 0) for w, o, n, kk in zip(ws, outs, ns, k_major)))
    assert _lib.lib().wkv_rows_products(torch.cuda.current_stream().cuda_stream, rows, K, count, jobs) == 0
    torch.cuda.synchronize()
    for i, (w, o, kk) in enumerate(zip(ws, outs, k_major)):
        w, got = (w if kk else w.t()).double(), o.double().sum(0) if kk else o.double()
        want, sizes = x.double() @ w, x.double().abs() @ w.abs()
        assert bool(((got - want).abs() <= 2 ** -8 * want.abs() + K * 2 ** -24 * sizes).all()), i


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("B,H,ffn", [(1, 1, 64), (3, 2, 448), (16, 1, 192), (17, 3, 640), (33, 2, 256), (64, 9, 2016), (65, 1, 128),
                                     (1, 32, 7168), (20, 40, 8960)])
def test_layer_of_single_tokens(version, B, H, ffn):
    """A serving loop's layer (one token per sequence, no autograd, bf16): row counts at the edges of the 16-row tiles, widths
    of fewer and of more 64-deep chunks than a workgroup has wavefronts, and the widths of models in use, whose products take other
    shapes; 65 rows and ffn = 2016 take the general way.
    Against the fp32 modules on the same rounded parameters.  Six bf16 roundings (2^-9 each, added in squares: 4.8e-3) lie
    between input and output: 1e-2 in norm over all rows.  In one row the operator's sum over 64 keys and ln_x's mean can
    cancel, which divides by what is left: among 64 rows some lose a digit, 4.8e-2 (the general way's worst row: 2.1e-2)."""
    from rwkv_wkv_hip import blocks as K
    C = 64 * H
    g = _g(B + 10 * H)
    bf = lambda t: t.bfloat16().float()
    x, shift, shift2 = (bf(torch.randn(B, *n, generator=g)) for n in ((1, C), (C,), (C,)))
    state = torch.randn(B, H, 64, 64, generator=g) * 0.1
    tm, cm = (TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8), (ChannelMix5 if version == 5 else ChannelMix6)(C, ffn, seed=9)
    for m in (tm, cm):
        for p in m.parameters():
            p.data = bf(p.data)
    if version == 5:
        wkv = lambda B, T, C, H, s, r, k, v, w, u: O.wkv5_op(B, T, C, H, s, r, k, v, w, u)
    else:
        wkv = lambda B, T, C, H, r, k, v, w, u, s: O.wkv6_op(B, T, C, H, r, k, v, w, u, s)
    gtm, gcm = copy.deepcopy(tm).cuda().bfloat16(), copy.deepcopy(cm).cuda().bfloat16()
    with torch.no_grad():
        a_ref, (sh_ref, s_ref) = tm(x, (shift, state), wkv)
        y_ref, sh2_ref = cm(a_ref, shift2)
        timemix, channelmix = (K.timemix5_forward, K.channelmix5_forward) if version == 5 else (K.timemix6_forward, K.channelmix6_forward)
        xg, states = x.cuda().bfloat16(), (shift.cuda().bfloat16(), state.cuda())
        a, (sh, s) = timemix(gtm, xg, states)
        y, sh2 = channelmix(gcm, a, shift2.cuda().bfloat16())
    assert a.dtype == y.dtype == torch.bfloat16 and a.shape == y.shape == x.shape
    assert torch.equal(sh.float().cpu(), sh_ref) and torch.equal(sh2, a[:, -1]) and s.dtype == torch.float32
    for name, got, ref in (("timemix", a, a_ref), ("state", s, s_ref), ("layer", y, y_ref)):
        got, ref = got.float().cpu().reshape(B, -1), ref.reshape(B, -1)
        rel = (got - ref).norm(dim=1) / ref.norm(dim=1)
        assert rel.max() < 4.8e-2, f"{name}: row {int(rel.argmax())} off by {rel.max():.2e}"
        assert (got - ref).norm() < 1e-2 * ref.norm(), f"{name}: off by {((got - ref).norm() / ref.norm()).item():.2e}"


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("B,H", [(1, 2), (3, 5), (17, 12), (64, 4)])
def test_single_token_layer_rounds_where_the_steps_round(version, B, H):
    """The TimeMix of one token per sequence without autograd (kernels of its own) against the same call with autograd on
    (the steps, with a bf16 tensor between any two).  Both round at the same places, so they differ only where sums in another order
    land on the other side of a rounding: of the state's two factors and decay some percent of the elements by 2^-8,
    1e-3 in norm; of the output, behind four roundings, 2.5e-3.  (Kept in fp32 in between they differ by 1.2e-3 to 1.6e-3 and by 4e-3.)"""
    from rwkv_wkv_hip import blocks as K
    C = 64 * H
    g = _g(B + H)
    m = (TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8).cuda().bfloat16()
    x, shift = torch.randn(B, 1, C, generator=g).cuda().bfloat16(), torch.randn(B, C, generator=g).cuda().bfloat16()
    state = (torch.randn(B, H, 64, 64, generator=g) * 0.1).cuda()
    timemix = K.timemix5_forward if version == 5 else K.timemix6_forward
    ref, (_, s_ref) = timemix(m, x, (shift, state))
    assert ref.requires_grad
    with torch.no_grad():
        got, (_, s) = timemix(m, x, (shift, state))
    rel = lambda a, b: ((a - b).double().norm() / b.double().norm()).item()
    assert rel(s, s_ref) < 1e-3 and rel(got, ref) < 2.5e-3, (rel(s, s_ref), rel(got, ref))


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("T,grad", [(1, False), (1, True), (5, False), (5, True)])
def test_layer_refuses_states_of_another_shape(version, T, grad):
    """A shift state that is not (B, C) and a WKV state that is not (B, H, 64, 64) are refused, also where they have as many
    elements as the right ones."""
    from rwkv_wkv_hip import blocks as K
    B, H = 3, 2
    C = 64 * H
    tm, cm = ((TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8).cuda().bfloat16(),
              (ChannelMix5 if version == 5 else ChannelMix6)(C, 4 * C, seed=9).cuda().bfloat16())
    timemix, channelmix = (K.timemix5_forward, K.channelmix5_forward) if version == 5 else (K.timemix6_forward, K.channelmix6_forward)
    x, shift, state = torch.randn(B, T, C).cuda().bfloat16(), torch.randn(B, C).cuda().bfloat16(), torch.randn(B, H, 64, 64).cuda()
    with torch.set_grad_enabled(grad):
        timemix(tm, x, (shift, state)), channelmix(cm, x, shift)
        for wrong in (shift.view(C, B), shift.view(B, 1, C), shift.view(-1)):
            with pytest.raises(Exception):
                timemix(tm, x, (wrong, state))
            with pytest.raises(Exception):
                channelmix(cm, x, wrong)
        for wrong in (state.view(H, B, 64, 64), state.view(B, H, 4096), state.view(B * H, 64, 64)):
            with pytest.raises(Exception):
                timemix(tm, x, (shift, wrong))


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("grad", [True, False])
def test_layer_native_holds_no_more_memory_than_the_steps(version, grad):
    """The most memory a layer's pass (with its backward) holds at once, against the same layer as a node per step, which lets go of every
    saved tensor on the way: within a tenth."""
    from rwkv_wkv_hip import blocks as K
    B, T, H = 1, 2048, 32
    C = 64 * H
    timemix, channelmix = (K.timemix5_forward, K.channelmix5_forward) if version == 5 else (K.timemix6_forward, K.channelmix6_forward)
    x, gy = torch.randn(B, T, C).cuda().bfloat16(), torch.randn(B, T, C).cuda().bfloat16()
    shift, state = torch.randn(B, C).cuda().bfloat16(), torch.randn(B, H, 64, 64).cuda()

    def peak(hooked):
        tm, cm = ((TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8).cuda().bfloat16(),
                  (ChannelMix5 if version == 5 else ChannelMix6)(C, C * 7 // 2, seed=9).cuda().bfloat16())
        if hooked:
            tm.key.register_forward_hook(lambda *a: None)
            cm.key.register_forward_hook(lambda *a: None)
        leaves = [x.clone().requires_grad_(grad), *tm.parameters(), *cm.parameters()]

        def run():
            with torch.set_grad_enabled(grad):
                y, _ = channelmix(cm, timemix(tm, leaves[0], (shift, state))[0], shift)
            return torch.autograd.grad(y, leaves, gy) if grad else y
        run()
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        run()
        return torch.cuda.max_memory_allocated() - before
    native, steps = peak(False), peak(True)
    assert native <= 1.1 * steps, (native / 2**20, steps / 2**20)


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("T,frozen", [(1, ()), (2, ("key",)), (65, ()), (130, ("ln_x", "output", "value", "time"))])
def test_layer_native_matches_the_steps(version, T, frozen):
    """A layer's halves as the native host side runs them against the same kernels step by step (which a hook on one of the
    submodules asks for), with and without autograd and with some parameters frozen.  The two do the same operations in the
    same order; a matrix product may still be given another library kernel, whose sums round differently: one bf16 rounding
    (2^-8) per element of each result, in norm, carried through at most six products in a row."""
    from rwkv_wkv_hip import blocks as K
    B, C, H = 2, 128, 2
    g = _g(17)
    x, gy = torch.randn(B, T, C, generator=g), torch.randn(B, T, C, generator=g)
    tm, cm = (TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8), (ChannelMix5 if version == 5 else ChannelMix6)(C, 4 * C, seed=9)
    for m in (tm, cm):
        for n, p in m.named_parameters():
            p.requires_grad_(not n.startswith(frozen))
    timemix, channelmix = (K.timemix5_forward, K.channelmix5_forward) if version == 5 else (K.timemix6_forward, K.channelmix6_forward)

    def layer(hooked, grad):
        mods = [copy.deepcopy(m).cuda().bfloat16() for m in (tm, cm)]
        if hooked:
            for m in mods:
                m.key.register_forward_hook(lambda *a: None)
        rows = [t.cuda().bfloat16().requires_grad_(grad) for t in (x, x[:, 0] * 0.5, x[:, 0] * 0.25)]
        wkv = torch.randn(B, H, 64, 64, generator=_g(18)).cuda().requires_grad_(grad)
        with torch.set_grad_enabled(grad):
            a, (sh, s) = timemix(mods[0], rows[0], (rows[1], wkv))
            y, sh2 = channelmix(mods[1], a, rows[2])
        assert torch.equal(sh, rows[0][:, -1]) and torch.equal(sh2, a[:, -1])
        if not grad:
            return {"a": a, "s": s, "y": y}
        torch.autograd.backward([y, s, sh2], [gy.cuda().bfloat16(), torch.ones_like(s) * 0.1, torch.ones_like(sh2) * 0.1])
        named = {f"{i}.{n}": p.grad for i, m in enumerate(mods) for n, p in m.named_parameters()}
        return {"a": a, "s": s, "y": y, "gwkv": wkv.grad, **{f"grow{i}": t.grad for i, t in enumerate(rows)}, **named}

    for grad in (True, False):
        got, ref = layer(False, grad), layer(True, grad)
        for n in ref:
            assert (got[n] is None) == (ref[n] is None), n
            if ref[n] is not None:
                assert got[n].dtype == ref[n].dtype and got[n].shape == ref[n].shape, n
                assert (got[n] - ref[n]).float().norm() <= 6 * 2 ** -8 * ref[n].float().norm(), n


def _layer(version, C, H):
    from rwkv_wkv_hip import blocks as K
    tm, cm = ((TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8).cuda().bfloat16(),
              (ChannelMix5 if version == 5 else ChannelMix6)(C, 4 * C, seed=9).cuda().bfloat16())
    return tm, cm, *((K.timemix5_forward, K.channelmix5_forward) if version == 5 else (K.timemix6_forward, K.channelmix6_forward))


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("T", [1, 5])
@pytest.mark.parametrize("grad", [False, True])
def test_which_calls_the_native_layer_answers(version, T, grad):
    """A plain bf16 module is answered by the native host side; whatever is not plain gets None from it (and so goes the
    general way)."""
    from rwkv_wkv_hip import _lib, ops
    B, H = 2, 2
    C = 64 * H
    x, shift, state = torch.randn(B, T, C).cuda().bfloat16(), torch.randn(B, C).cuda().bfloat16(), torch.randn(B, H, 64, 64).cuda()

    def answered(change=lambda tm, cm: None, x=x, shift=shift, state=state):
        tm, cm, _, _ = _layer(version, C, H)
        undo = change(tm, cm)
        with torch.set_grad_enabled(grad):
            got = _lib.host().timemix(version, ops._algo, tm, x, (shift, state)), _lib.host().channelmix(version, cm, x, shift)
        if undo is not None:
            undo.remove()
        assert (got[0] is None) == (got[1] is None)
        return got[0] is not None

    def replace(make):
        def change(tm, cm):
            for m in (tm, cm):
                new = make(m.key)
                new.weight = m.key.weight
                m.key = new.cuda().bfloat16()
        return change

    class Own(torch.nn.Linear):
        pass
    hook = lambda *a: None
    assert answered()
    assert not answered(lambda tm, cm: [m.key.register_forward_hook(hook) for m in (tm, cm)] and None)
    assert not answered(lambda tm, cm: [m.value.register_forward_pre_hook(hook) for m in (tm, cm)] and None)
    assert not answered(lambda tm, cm: [m.receptance.register_full_backward_hook(hook) for m in (tm, cm)] and None)
    assert not answered(lambda tm, cm: torch.nn.modules.module.register_module_forward_hook(hook))
    assert not answered(lambda tm, cm: [setattr(m.key, "forward", hook) for m in (tm, cm)] and None)
    assert not answered(replace(lambda l: torch.nn.Linear(l.in_features, l.out_features, bias=True)))
    assert not answered(replace(lambda l: Own(l.in_features, l.out_features, bias=False)))
    assert not answered(lambda tm, cm: [m.float() for m in (tm, cm)] and None)
    assert not answered(x=x.float())
    assert not answered(x=torch.empty(B, C, T, device="cuda", dtype=x.dtype).transpose(1, 2)) or T == 1
    assert not answered(x=torch.empty(B * T * C + 1, device="cuda", dtype=x.dtype)[1:].view(B, T, C))
    assert not answered(shift=shift.float())
    assert not answered(shift=shift.view(1, B, C))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        assert not answered()


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("way", ["saved on the host", "recomputed", "autocast"])
def test_layer_native_under_hooks_and_autocast(version, way):
    """What a layer saves for its backward may be taken away in between (packed by saved-tensor hooks, dropped and recomputed by
    activation checkpointing): the same bits.  Under autocast a layer goes step by step: as the same steps without."""
    from torch.utils.checkpoint import checkpoint
    B, T, H = 2, 70, 2
    C = 64 * H
    tm, cm, timemix, channelmix = _layer(version, C, H)
    g = _g(21)
    n = lambda *shape: torch.randn(*shape, generator=g).cuda()
    x, shift, shift2, state, gy, gs = n(B, T, C).bfloat16(), n(B, C).bfloat16(), n(B, C).bfloat16(), n(B, H, 64, 64), n(B, T, C).bfloat16(), n(B, H, 64, 64)

    def run(how):
        leaves = [t.clone().requires_grad_(True) for t in (x, shift, shift2, state)]
        wrt = [*leaves, *tm.parameters(), *cm.parameters()]

        def layer(x, shift, shift2, state):
            a, (_, s) = timemix(tm, x, (shift, state))
            return channelmix(cm, a, shift2)[0], s
        if how == "recomputed":
            out = checkpoint(layer, *leaves, use_reentrant=False)
        elif how == "saved on the host":
            with torch.autograd.graph.save_on_cpu():
                out = layer(*leaves)
        elif how == "autocast":
            with torch.autocast("cuda", dtype=torch.bfloat16):
                out = layer(*leaves)
        else:
            out = layer(*leaves)
        return [*out, *torch.autograd.grad(out, wrt, [gy, gs])]
    if way == "autocast":
        got = run(way)
        for m in (tm, cm):
            m.key.register_forward_hook(lambda *a: None)
    else:
        got = run(way)
    for a, b in zip(got, run("plain")):
        assert a.dtype == b.dtype and torch.equal(a, b)


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_channelmix_forward_on_the_kernels(version, dtype):
    from rwkv_wkv_hip import blocks as K
    B, T, C = 2, 70, 128
    g = _g(12)
    x, shift, gy = torch.randn(B, T, C, generator=g), torch.randn(B, C, generator=g), torch.randn(B, T, C, generator=g)
    cpu = (ChannelMix5 if version == 5 else ChannelMix6)(C, 4 * C, seed=6)
    gpu = copy.deepcopy(cpu).cuda().to(dtype)
    ref = _run_module(lambda m, xs, st: m(xs, st), cpu, x, shift, gy)
    fwd = K.channelmix5_forward if version == 5 else K.channelmix6_forward
    got = _run_module(fwd, gpu, x.cuda().to(dtype), shift.cuda().to(dtype), gy.cuda().to(dtype))
    torch.cuda.synchronize()
    if dtype == torch.float32:
        for name, a, b in zip(("y", "gx", "gshift"), got[:3], ref[:3]):
            assert_close(a, b, 2e-3, f"channelmix v{version} {name}")
        for n in ref[3]:
            assert_close(got[3][n], ref[3][n], 3e-3, f"channelmix v{version} grad {n}")
    else:       # the whole module (weights, matmuls) is bf16 here, the reference fp32: compare in norm
        for name, a, b in zip(("y", "gx"), got[:2], ref[:2]):
            rel = ((a.float().cpu() - b).norm() / b.norm()).item()
            assert rel < 3e-2, f"channelmix bf16 v{version} {name}: relative error {rel}"


def test_full_shape_7b_edges():
    """The 7B shape of one segment (B1 T4096 C4096, bf16): every pass against the CPU oracle on the whole tensor."""
    from rwkv_wkv_hip import blocks as K
    B, T, C = 1, 4096, 4096
    g = _g(77)
    bf = torch.bfloat16
    x, shift = torch.randn(B, T, C, generator=g).to(bf), torch.randn(B, C, generator=g).to(bf)
    coefs = [torch.rand(C, generator=g) for _ in range(5)]
    dyn = (torch.randn(5, B, T, C, generator=g) * 0.3).to(bf)
    with torch.no_grad():
        ref = OB.mix_v6(x.float(), shift.float(), coefs, dyn.float())
        got = K.token_shift_mix(x.cuda(), shift.cuda(), [c.cuda() for c in coefs], dyn=dyn.cuda())
        for j in range(5):
            assert_close(got[j], ref[j], 2e-2, f"7B mix out[{j}]")
        y, gate = (torch.randn(B, T, C, generator=g) * 2).to(bf), torch.randn(B, T, C, generator=g).to(bf)
        w, b = torch.randn(C, generator=g), torch.randn(C, generator=g)
        ref = OB.ln_x_gate(y.float(), gate.float(), w, b, C // 64, 64e-5)
        got = K.ln_x_gate(y.cuda(), gate.cuda(), w.cuda(), b.cuda(), 64e-5)
        assert_close(got, ref, 2e-2, "7B ln_x*gate")
