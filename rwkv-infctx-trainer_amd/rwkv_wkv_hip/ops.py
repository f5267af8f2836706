"""torch.autograd front ends with the reference trainer's call signatures.

WKV_5.apply(B, T, C, H, state, r, k, v, w, u)  -> (y, new_state)
WKV_6.apply(B, T, C, H, r, k, v, w, u, s)      -> (y, new_state)
wkv_op(time_decay, time_first, k, v, wkv_state) -> (y, new_state)

Argument order and meaning are those of WKV5_CUDA / WKV6STATE_CUDA
(RWKV-v5/src/module/TimeMix.py:20-31, RWKV-v6/src/module/TimeMix.py:19-26) and
of torch.ops.rwkv.wkv (RWKV-v4neo/src/model.py:130-132): ``w`` is the RAW decay
parameter and the gradient returned for it is with respect to that raw
parameter.  Unlike the reference's kernels the functions are functional (the
new state is returned, and is differentiable); RUN_WKV5_CUDA /
RUN_WKV6STATE_CUDA keep the reference's in-place convention on top of them.

All tensors must live on the GPU; the work is done by librwkv_wkv_hip.so on the
current HIP stream.  The operators' host side (checks, allocation, autograd) is
native: csrc/host.cpp.
"""
from __future__ import annotations

import contextlib
import os

import torch

from . import _lib
from ._lib import WKVError, check

HEAD = 64
_DT = {torch.float32: _lib.WKV_F32, torch.bfloat16: _lib.WKV_BF16, torch.float16: _lib.WKV_F16}
_ALGO = {"auto": _lib.ALGO_AUTO, "recurrent": _lib.ALGO_RECURRENT, "chunked": _lib.ALGO_CHUNKED}
_algo = _ALGO[os.environ.get("RWKV_WKV_ALGO", "auto")]


def set_algo(name: str):
    """'auto' | 'recurrent' | 'chunked' for the WKV5/WKV6 operators."""
    global _algo
    _algo = _ALGO[name]


def _ptr(t):
    return None if t is None else t.data_ptr()


def _stream():
    return torch.cuda.current_stream().cuda_stream


def _on_gpu(*ts):
    for t in ts:
        if t is not None and not t.is_cuda:
            raise WKVError("rwkv_wkv_hip operators need GPU tensors (there is no CPU path)")


def _workspace(nbytes, device):
    return torch.empty(max(int(nbytes), 16), dtype=torch.uint8, device=device)


stats = {"forward_launches": 0, "forward_reused": 0}      # counters for tests and diagnostics


class RecomputeCache:
    """Opt-in reuse of a forward pass by the recomputation that activation checkpointing runs later.

    Under activation checkpointing (the reference wraps every block in ``deepspeed.checkpointing.checkpoint``,
    RWKV-v5/src/model.py:674-683) the operator's forward runs twice per layer and segment: once without autograd
    while the model runs forward, once more when backward recomputes the block.  With a cache installed
    (``with recompute_cache(): ...`` around the training step) the first run keeps its outputs and its state
    checkpoints, and the recomputation takes them over instead of running the kernels again: one forward pass of the
    operator less per layer and segment, paid for with y, the new state and the checkpoints (about 6 bytes per token
    and channel) held from forward to backward.

    Which kept run a call with autograd on may take over:

    * keyed (recommended): the caller names each call, ``with call_key((layer, segment)): ...`` around the block's
      forward.  A kept run is taken over only by a call with the same key and signature (operator, shape, dtypes);
      any other call runs the kernels.  This is safe for every pattern, including the reference's outer per-segment
      checkpoint (RWKV-v5/src/model.py:1248: segments 0..S-2 run without autograd, the last one with) and nested
      checkpoints.
    * unkeyed: last kept, first taken over, by signature.  This is what plain activation checkpointing of a stack of
      equal layers does (the recomputation replays the blocks in reverse order) and nothing else: a call with
      autograd on that is not a recomputation would take over another call's results.  That is why every take-over
      is verified: 1024 elements spread over r, kept on the device from the first run, are compared with the
      recomputation's r by a few asynchronous device operations, and ``check()`` (called on leaving the ``with`` block;
      one synchronisation per step) raises if any take-over met different inputs.  The step's gradients are then
      wrong and must be discarded; switch to keys.

    Kept runs that are never taken over (forward-only work inside the block, segments outside the BPTT range) stay
    until the ``with`` block is left; ``max_bytes`` bounds what they hold (oldest dropped first).  Under nested
    checkpoints an inner recomputation runs without autograd again and keeps its run a second time: harmless, the
    copy is dropped on leaving."""

    SAMPLE = 1024

    def __init__(self, max_entries: int = 4096, max_bytes: int = 16 << 30, verify: bool = True):
        self.entries, self.max_entries, self.max_bytes, self.verify = [], max_entries, max_bytes, verify
        self.bytes, self.bad = 0, None

    @classmethod
    def _sample(cls, r):
        flat = r.reshape(-1)
        step = max(flat.numel() // cls.SAMPLE, 1)
        return flat[::step][:cls.SAMPLE].clone()

    @staticmethod
    def _nbytes(payload):
        return sum(t.numel() * t.element_size() for t in payload if torch.is_tensor(t))

    def push(self, key, sig, r, payload):
        n = self._nbytes(payload)
        while self.entries and (len(self.entries) >= self.max_entries or self.bytes + n > self.max_bytes):
            self.bytes -= self.entries.pop(0)[4]
        self.entries.append((key, sig, self._sample(r) if self.verify else None, payload, n))
        self.bytes += n

    def pop(self, key, sig, r):
        hit = None
        if key is None:         # unkeyed: the most recent kept run, if it is unkeyed too and has this signature
            if self.entries and self.entries[-1][0] is None and self.entries[-1][1] == sig:
                hit = self.entries.pop()
        else:
            for i in range(len(self.entries) - 1, -1, -1):
                if self.entries[i][0] == key and self.entries[i][1] == sig:
                    hit = self.entries.pop(i)
                    break
        if hit is None:
            return None
        self.bytes -= hit[4]
        if hit[2] is not None:      # asynchronous: no host synchronisation here
            differs = (hit[2] != self._sample(r)).any()
            self.bad = differs if self.bad is None else (self.bad | differs)
        return hit[3]

    def check(self):
        """Raises if a take-over since the last check met inputs that differ from the kept run's (synchronises)."""
        bad, self.bad = self.bad, None
        if bad is not None and bool(bad.item()):
            raise WKVError("recompute cache: a kept forward run was taken over by a call with different inputs (a call "
                           "with autograd on that was not the recomputation of that run); the gradients of this step "
                           "are wrong.  Name the calls with call_key() or keep such calls outside recompute_cache()")

    def clear(self):
        self.entries.clear()
        self.bytes = 0


_cache = None
_key = None


class recompute_cache:
    """Context manager that installs a ``RecomputeCache`` for the operators called inside it; on leaving, the
    take-overs are verified (``RecomputeCache.check``) and what is still kept is dropped."""

    def __init__(self, cache: RecomputeCache = None):
        self.cache = cache or RecomputeCache()

    def __enter__(self):
        global _cache
        self.prev, _cache = _cache, self.cache
        return self.cache

    def __exit__(self, exc_type, *exc):
        global _cache
        _cache = self.prev
        self.cache.clear()
        if exc_type is None:
            self.cache.check()
        else:
            self.cache.bad = None
        return False


class call_key:
    """Names the operator calls made inside it for the recompute cache (any hashable: e.g. (layer, segment)).  The
    same key must be in force when the block's forward is recomputed, which it is when the ``with`` sits inside the
    checkpointed function."""

    def __init__(self, key):
        self.key = key

    def __enter__(self):
        global _key
        self.prev, _key = _key, self.key
        return self

    def __exit__(self, *exc):
        global _key
        _key = self.prev
        return False


def _forward56_cached(version, B, T, C, H, r, k, v, w, u, s, need_grad, out_state):
    """The operator's forward behind the recompute cache: y, the new state, the workspace with the state checkpoints and
    the algorithm in force."""
    cache = _cache
    sig = (version, B, T, C, H, r.dtype, w.dtype, tuple(w.shape), out_state is not None)
    if need_grad:
        hit = cache.pop(_key, sig, r)
        if hit is not None:          # the recomputation of a forward run that kept its results
            y, new_state, ws, algo = hit
            if out_state is not None:
                out_state.copy_(new_state)
                new_state = out_state
            stats["forward_reused"] += 1
            return y, new_state, ws, algo
    algo = _algo
    y, new_state, ws = _lib.host().forward56(version, algo, B, T, C, H, r, k, v, w, u, s, out_state)
    stats["forward_launches"] += 1
    if not need_grad:
        cache.push(_key, sig, r, (y, new_state.clone() if out_state is not None else new_state, ws, algo))
    return y, new_state, ws, algo


class _Cached56(torch.autograd.Function):
    """WKV5 / WKV6 while a recompute cache is installed (otherwise the native front, csrc/host.cpp, is called directly).
    ``in_place``: the new state goes into ``s`` and no gradient flows through it, as in the reference
    (RWKV-v5/src/module/TimeMix.py:60,139-140)."""

    @staticmethod
    def forward(ctx, version, in_place, grad_mode, B, T, C, H, r, k, v, w, u, s):
        assert s.is_contiguous() and w.is_contiguous() and u.is_contiguous()
        assert s.shape == (B, H, HEAD, HEAD) and H * HEAD == C and u.numel() == C
        assert (s.dtype == w.dtype == torch.float32 and w.numel() == C) if version == 5 else w.shape == (B, T, C)
        need_grad = grad_mode and any(ctx.needs_input_grad)      # no checkpoints kept under torch.no_grad()
        with torch.no_grad():
            u32, s32 = u.float(), s.clone() if in_place else s.float()
            w32 = w if version == 5 else _lib.host().decay_operand(_algo, B, T, C, H, r, w)
            y, new_state, ws, algo = _forward56_cached(version, B, T, C, H, r, k, v, w32, u32, s32, need_grad, s if in_place else None)
        ctx.set_materialize_grads(False)
        ctx.call = (version, in_place, algo, B, T, C, H, w.dtype, u.dtype, s.dtype)
        ctx.ws = ws
        ctx.save_for_backward(r, k, v, w32, u32, s32)
        return y if in_place else (y, new_state.to(s.dtype))

    @staticmethod
    def backward(ctx, gy, gstate=None):
        version, in_place, algo, B, T, C, H, wdtype, udtype, sdtype = ctx.call
        r, k, v, w32, u32, s32 = ctx.saved_tensors
        gy = torch.zeros_like(r) if gy is None else gy.contiguous()
        assert gy.dtype == r.dtype
        gstate = None if gstate is None else gstate.float().contiguous()
        gr, gk, gv, gw, gu, gs = _lib.host().backward56(version, algo, B, T, C, H, r, k, v, w32, u32, s32, gy, gstate, ctx.ws)
        return (None,) * 7 + (gr, gk, gv, gw.to(wdtype), gu.to(udtype), None if in_place else gs.to(sdtype))


@contextlib.contextmanager
def _untraced():
    recording = torch._C._get_tracing_state()
    torch._C._set_tracing_state(None)
    try:
        yield recording
    finally:
        torch._C._set_tracing_state(recording)


class _Traced(torch.autograd.Function):
    """An operator's call while ``torch.jit.trace`` records: one node of the graph, which makes the call again on the inputs
    the graph is run with.  (The tracer does not see the native front end, csrc/host.cpp.)  ``written``: the tensor the call
    writes its new state into."""

    @staticmethod
    def forward(ctx, call, written, *args):
        ctx.call, ctx.args = call, [None if torch.is_tensor(a) else a for a in args]
        ctx.save_for_backward(*[a.detach().clone() if a is written else a for a in args if torch.is_tensor(a)])
        ctx.set_materialize_grads(False)
        with _untraced() as recording:
            outs = call(*args)
        if recording is None:
            return outs
        outs, many = outs if isinstance(outs, tuple) else (outs,), isinstance(outs, tuple)
        known = [torch.empty(o.shape, dtype=o.dtype, device=o.device) for o in outs]      # seen by the tracer, as results that
        with _untraced():                                                                 # require a gradient have to be
            for a, o in zip(known, outs):
                a.copy_(o)
        return tuple(known) if many else known[0]

    @staticmethod
    def backward(ctx, *gouts):
        saved = iter(ctx.saved_tensors)
        args = [next(saved).detach().requires_grad_(need) if a is None else a for a, need in zip(ctx.args, ctx.needs_input_grad[2:])]
        with torch.enable_grad():
            outs = ctx.call(*args)
        outs = outs if isinstance(outs, tuple) else (outs,)
        leaves = [a for a, need in zip(args, ctx.needs_input_grad[2:]) if need]
        pairs = [(o, g) for o, g in zip(outs, gouts) if g is not None]
        grads = iter(torch.autograd.grad([o for o, _ in pairs], leaves, [g for _, g in pairs], allow_unused=True))
        return (None, None, *(next(grads) if need else None for need in ctx.needs_input_grad[2:]))


def _op56(version, in_place, B, T, C, H, r, k, v, w, u, s):
    if _cache is not None:
        return _Cached56.apply(version, in_place, torch.is_grad_enabled(), B, T, C, H, r, k, v, w, u, s)
    out = _lib.host().wkv56(version, _algo, in_place, B, T, C, H, r, k, v, w, u, s)
    if out is None:
        return _Traced.apply(_op56, s if in_place else None, version, in_place, B, T, C, H, r, k, v, w, u, s)
    stats["forward_launches"] += 1
    return out


class WKV_5:
    """WKV5: per-channel decay.  ``WKV_5.apply(B, T, C, H, state, r, k, v, w, u) -> (y, new_state)`` with state
    (B,H,64,64) fp32 [key][value]; r,k,v (B,T,C) in one dtype; w (H,64) fp32 raw; u (H,64).  Differentiable in
    everything, the state included; a call under torch.no_grad() keeps no checkpoints."""

    @staticmethod
    def apply(B, T, C, H, state, r, k, v, w, u):
        return _op56(5, False, B, T, C, H, r, k, v, w, u, state)


class WKV_6:
    """WKV6: per-token decay.  ``WKV_6.apply(B, T, C, H, r, k, v, w, u, s) -> (y, new_state)`` with r,k,v (B,T,C);
    w (B,T,C) raw (any float dtype, used in fp32; a bf16 or fp16 w of the streams' type is read as it is by the blocked
    algorithms and by a single token without a backward; its gradient comes back in its type, as in the reference,
    RWKV-v6/src/module/TimeMix.py:50,90); u (H,64);
    s (B,H,64,64) [key][value]."""

    @staticmethod
    def apply(B, T, C, H, r, k, v, w, u, s):
        return _op56(6, False, B, T, C, H, r, k, v, w, u, s)


def _direct_state(state, B, H):
    return state.dtype == torch.float32 and state.is_contiguous() and state.shape == (B, H, HEAD, HEAD) and not state.requires_grad


def RUN_WKV5_CUDA(B, T, C, H, state, r, k, v, w, u):
    """The reference's calling convention (RWKV-v5/src/module/TimeMix.py:145-154): returns y and leaves the new
    state in ``state``.  An fp32 contiguous state buffer (e.g. one layer's slice of the trainer's (N_layer,B,H,64,64)
    tensor, RWKV-v5/src/model.py:53-61) is written by the kernel directly, the incoming state surviving in a private copy
    for backward; anything else goes through the functional operator and a copy."""
    if _direct_state(state, B, H) and w.dtype == torch.float32 and w.is_contiguous() and u.is_contiguous():
        return _op56(5, True, B, T, C, H, r, k, v, w, u, state)
    y, new_state = WKV_5.apply(B, T, C, H, state.clone(), r, k, v, w, u)
    with torch.no_grad():
        state.copy_(new_state)
    return y


def RUN_WKV6STATE_CUDA(B, T, C, H, r, k, v, w, u, s):
    """The reference's calling convention (RWKV-v6/src/module/TimeMix.py:111-118): returns y and leaves the new
    state in ``s`` (written by the kernel directly when ``s`` is an fp32 contiguous buffer)."""
    if _direct_state(s, B, H) and w.is_contiguous() and u.is_contiguous() and w.shape == (B, T, C):
        return _op56(6, True, B, T, C, H, r, k, v, w, u, s)
    y, new_state = WKV_6.apply(B, T, C, H, r, k, v, w, u, s.clone())
    with torch.no_grad():
        s.copy_(new_state)
    return y


def wkv_op(time_decay, time_first, k, v, wkv_state):
    """RWKV-v4 WKV with the signature of torch.ops.rwkv.wkv
    (RWKV-v4neo/src/model.py:130-132): time_decay, time_first (C); k, v (B,T,C);
    wkv_state (B,C,3) = (aa, bb, pp).  Returns (y, new_state)."""
    out = _lib.host().wkv4(time_decay, time_first, k, v, wkv_state)
    return _Traced.apply(wkv_op, None, time_decay, time_first, k, v, wkv_state) if out is None else out


def cumsum_decay(w, chunk_len=128, per_token=True, factors=False, precision=64):
    """Decay tables of the chunked formulation from the raw decay parameter w (B,T,C) fp32, or (C,) expanded over
    T tokens when ``per_token`` is an int T.  Returns dict(log_w, incl, inter, intra, chunk_sum), all in log space;
    with ``factors=True`` also the exponentiated tables ws_exp, inter_exp, intra_exp (fp32) and the two re-centred
    factors r_decay, k_inv_decay of the intra-chunk product (fp64 for ``precision=64``, fp32 for 32), i.e.
    everything RWKV-v5/src/module/rwkv_inner.py:43-93 derives from w."""
    L = _lib.lib()
    _on_gpu(w)
    w = w.float().contiguous()
    if w.dim() == 3:
        Bw, T, C = w.shape
        pt = 1
    else:
        (C,), Bw, T, pt = w.shape, 1, int(per_token), 0
    new = lambda dt=torch.float32: torch.empty(Bw, T, C, dtype=dt, device=w.device)
    out = {n: new() for n in ("log_w", "incl", "inter", "intra")}
    out["chunk_sum"] = torch.empty(Bw, T // chunk_len, C, dtype=torch.float32, device=w.device)
    if not factors:
        check(L.wkv_cumsum_decay(_stream(), Bw, T, C, chunk_len, pt, _ptr(w), _ptr(out["log_w"]), _ptr(out["incl"]),
                                 _ptr(out["inter"]), _ptr(out["intra"]), _ptr(out["chunk_sum"])), "wkv_cumsum_decay")
        return out
    pdt = torch.float64 if precision == 64 else torch.float32
    out["ws_exp"] = torch.empty_like(out["chunk_sum"])
    out["inter_exp"], out["intra_exp"] = new(), new()
    out["r_decay"], out["k_inv_decay"] = new(pdt), new(pdt)
    check(L.wkv_cumsum_decay_factors(_stream(), Bw, T, C, chunk_len, pt, precision, _ptr(w), _ptr(out["log_w"]),
                                     _ptr(out["incl"]), _ptr(out["inter"]), _ptr(out["intra"]), _ptr(out["chunk_sum"]),
                                     _ptr(out["ws_exp"]), _ptr(out["inter_exp"]), _ptr(out["intra_exp"]),
                                     _ptr(out["r_decay"]), _ptr(out["k_inv_decay"])), "wkv_cumsum_decay_factors")
    return out
