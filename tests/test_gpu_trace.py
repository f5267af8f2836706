"""torch.jit.trace over the operators and the layers: a graph recorded on one set of inputs gives, on another, what the
direct call gives."""
import pytest
import torch

from oracle.timemix_restated import ChannelMix5, ChannelMix6, TimeMix5, TimeMix6

pytestmark = [pytest.mark.gpu, pytest.mark.filterwarnings("ignore::torch.jit.TracerWarning"), pytest.mark.filterwarnings("ignore::DeprecationWarning")]


def _inputs(version, T, io, seed):
    g = torch.Generator().manual_seed(seed)
    n = lambda *shape: torch.randn(*shape, generator=g) * 0.5
    B, H = 2, 2
    C = 64 * H
    if version == 4:
        return [n(C) - 1, n(C), n(B, T, C).to(io), n(B, T, C).to(io), torch.stack([n(B, C), n(B, C).abs() + 1, n(B, C)], 2)]
    r, k, v = (n(B, T, C).to(io) for _ in range(3))
    u, s = n(H, 64), n(B, H, 64, 64)
    return [s, r, k, v, n(H, 64) - 1, u] if version == 5 else [r, k, v, n(B, T, C).to(io) - 1, u, s]


def _call(version, T):
    import rwkv_wkv_hip as W
    if version == 4:
        return lambda *a: W.wkv_op(*a)
    return lambda *a: (W.WKV_5 if version == 5 else W.WKV_6).apply(2, T, 128, 2, *a)


@pytest.mark.parametrize("version", [4, 5, 6])
@pytest.mark.parametrize("T,io", [(1, torch.bfloat16), (20, torch.float32), (70, torch.bfloat16)])
def test_traced_operator(version, T, io):
    call = _call(version, T)
    first, other = ([x.cuda() for x in _inputs(version, T, io, seed)] for seed in (1, 2))
    graph = torch.jit.trace(call, tuple(first), check_trace=False)
    for a, b in zip(graph(*other), call(*other)):
        assert torch.equal(a, b)
    # recorded and run with autograd on
    leaves = lambda xs: [x.clone().requires_grad_(True) for x in xs]
    graph = torch.jit.trace(call, tuple(leaves(first)), check_trace=False)
    got, want = leaves(other), leaves(other)
    (y, s), (y2, s2) = graph(*got), call(*want)
    gy, gs = torch.randn_like(y), torch.randn_like(s)
    for a, b in zip((y, s, *torch.autograd.grad([y, s], got, [gy, gs])), (y2, s2, *torch.autograd.grad([y2, s2], want, [gy, gs]))):
        assert torch.equal(a, b)


@pytest.mark.parametrize("version", [5, 6])
def test_traced_operator_with_the_state_in_place(version):
    import rwkv_wkv_hip as W
    T = 20
    run = W.RUN_WKV5_CUDA if version == 5 else W.RUN_WKV6STATE_CUDA
    call = lambda *a: run(2, T, 128, 2, *a)
    first, other = ([x.cuda() for x in _inputs(version, T, torch.bfloat16, seed)] for seed in (1, 2))
    graph = torch.jit.trace(call, tuple(x.clone() for x in first), check_trace=False)
    a, b = [x.clone() for x in other], [x.clone() for x in other]
    assert torch.equal(graph(*a), call(*b)) and all(torch.equal(x, y) for x, y in zip(a, b))
    s = 0 if version == 5 else 5
    assert not torch.equal(a[s], other[s])


@pytest.mark.parametrize("version", [5, 6])
@pytest.mark.parametrize("T", [1, 33])
def test_traced_layer(version, T):
    """The graph holds the layer's steps, whose results differ from the native halves' by roundings (six in a row at most)."""
    from rwkv_wkv_hip import blocks as K
    B, H = 2, 2
    C = 64 * H
    tm = (TimeMix5 if version == 5 else TimeMix6)(C, H, seed=8).cuda().bfloat16()
    cm = (ChannelMix5 if version == 5 else ChannelMix6)(C, 4 * C, seed=9).cuda().bfloat16()
    timemix, channelmix = (K.timemix5_forward, K.channelmix5_forward) if version == 5 else (K.timemix6_forward, K.channelmix6_forward)

    def layer(x, shift, state, shift2):
        a, (sh, s) = timemix(tm, x, (shift, state))
        y, sh2 = channelmix(cm, a, shift2)
        return y, sh, s, sh2

    def rows(seed):
        g = torch.Generator().manual_seed(seed)
        n = lambda *shape: torch.randn(*shape, generator=g).cuda()
        return n(B, T, C).bfloat16(), n(B, C).bfloat16(), n(B, H, 64, 64) * 0.1, n(B, C).bfloat16()
    for p in [*tm.parameters(), *cm.parameters()]:          # (the tracer takes no constants that require a gradient)
        p.requires_grad_(False)
    with torch.no_grad():
        graph = torch.jit.trace(layer, rows(1), check_trace=False)
        for a, b in zip(graph(*rows(2)), layer(*rows(2))):
            assert (a - b).float().norm() <= 6 * 2 ** -8 * b.float().norm()
