"""GPU tests of the native host path (csrc/fox_torch.cpp) against the general Python path, which the same inputs take through the
autograd nodes directly: the two launch the same kernels, so every output and gradient must agree bit for bit, in both
layouts, with every optional argument, and for inputs the native path hands back (tensors that need a copy first)."""
import time
import warnings
from importlib import import_module

import numpy as np
import pytest
import torch

from conftest import make_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ft():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    import forgetting_transformer
    return forgetting_transformer


def _grads(out, leaves, do):
    return (out.detach(),) + torch.autograd.grad(out, leaves, do)


def _equal(a, b):
    for x, y in zip(a, b):
        assert x.shape == y.shape and x.dtype == y.dtype and torch.equal(x, y)


@pytest.mark.parametrize("head_first", [True, False])
@pytest.mark.parametrize("logit", [False, True])
@pytest.mark.parametrize("thr,seq,M", [(None, None, 130), ("auto", [3, 60], 130), (-5.0, None, 200), ("per_head", [0, 7], 1), ("table", None, 77)])
def test_attention(ft, head_first, logit, thr, seq, M):
    from forgetting_transformer.ops import _native
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    B, H, N, D = 2, 3, 200, 64
    q, k, v, g, do, ss = make_inputs(B, H, M, N, D, device="cuda", head_first=head_first, seq_start=seq, seed=M, gate_mean=1.0)
    if logit:
        g = (g * 3 + 2).bfloat16()
    t = {"per_head": torch.linspace(-9, -3, H, device="cuda"), "table": torch.full((B, H), -4.0, device="cuda")}.get(thr, thr)
    leaves = [x.requires_grad_() for x in (q, k, v, g)]
    assert _native.load().attention(q, k, v, g, head_first, ss, None, F._native_threshold(t, q, head_first), logit) is not None
    fn = ft.forgetting_attention_from_logits if logit else ft.forgetting_attention
    out = fn(q, k, v, g, head_first=head_first, seq_start=ss, adaptive_threshold=t)
    a = [x if head_first else x.transpose(1, 2) for x in (q, k, v, g)]
    node = F.ForgettingAttentionFromLogits if logit else F.ForgettingAttention
    ref = node.apply(*a, ss, None, t) if logit else node.apply(*a, ss, True, None, t)
    back = lambda x: x if head_first else x.transpose(1, 2)
    if logit:
        assert torch.equal(out[1], back(ref[1])) and not out[1].requires_grad
        out, ref = out[0], ref[0]
    _equal(_grads(out, leaves, do), _grads(back(ref), leaves, do))
    with torch.no_grad():
        plain = fn(q, k, v, g, head_first=head_first, seq_start=ss, adaptive_threshold=t)
    assert torch.equal(plain[0] if logit else plain, out) and not (plain[0] if logit else plain).requires_grad


@pytest.mark.parametrize("head_first", [True, False])
@pytest.mark.parametrize("gated,M", [(True, 130), (False, 130), (True, 1)])
def test_attention_norm_gate(ft, head_first, gated, M):
    from forgetting_transformer.ops import _lib
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    B, H, N, D = 2, 3, 200, 64
    q, k, v, g, do, ss = make_inputs(B, H, M, N, D, device="cuda", head_first=False, seed=M)
    gate = torch.randn(B, M, H, D, device="cuda").bfloat16() if gated else None
    swap = (lambda x: x.transpose(1, 2)) if head_first else (lambda x: x)   # head-first views of (B, T, H * D) memory, as the layer has them
    w = torch.rand(H * D, device="cuda", requires_grad=True)
    leaves = [x.requires_grad_() for x in (q, k, v, g) + ((gate,) if gated else ())] + [w]
    args = [swap(x) for x in (q, k, v, g)]
    y = ft.forgetting_attention_norm_gate(*args, swap(gate) if gated else None, w, head_first=head_first)
    hf = [x.transpose(1, 2) for x in (q, k, v, g)] + [gate.transpose(1, 2) if gated else None]
    ref = F.ForgettingAttentionNormGate.apply(*hf, w, None, None, None, _lib.ACT_SIGMOID if gated else _lib.ACT_NONE, 1e-6, False)
    _equal(_grads(swap(y), leaves, do), _grads(ref.transpose(1, 2), leaves, do))


def test_norms_and_shift(ft):
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.norm_gate import GroupNormGated, GroupNormPlain
    from forgetting_transformer.ops.token_shift import TokenShift
    x, g = (torch.randn(2, 50, 192, device="cuda").bfloat16().requires_grad_() for _ in range(2))
    w = torch.rand(192, device="cuda").bfloat16().requires_grad_()
    do = torch.randn_like(x)
    _equal(_grads(ft.group_norm(x, w, is_rms_norm=True, num_groups=3), [x, w], do),
           _grads(GroupNormPlain.apply(x, w, None, None, 1e-5, False, False, True, 3), [x, w], do))
    _equal(_grads(ft.group_norm_gated(x, g, w, is_rms_norm=True, num_groups=3), [x, g, w], do),
           _grads(GroupNormGated.apply(x, g, w, None, "swish", None, 1e-6, False, False, True, 3), [x, g, w], do))
    x4 = x.detach().view(2, 50, 3, 64).requires_grad_()
    p, c = (torch.rand(2, 50, 3, device="cuda").requires_grad_() for _ in range(2))
    _equal(_grads(ft.token_shift(x4, p, c), [x4, p, c], do.view_as(x4)), _grads(TokenShift.apply(x4, p, c), [x4, p, c], do.view_as(x4)))


def test_calls_the_native_path_hands_back(ft):
    """Misaligned and non-unit-stride inputs are copied by the general path, other streams and a second backward behave as before."""
    q, k, v, g, do, _ = make_inputs(1, 2, 90, 90, 32, device="cuda", seed=1)
    want = ft.forgetting_attention(q, k, v, g, head_first=True)
    odd = torch.empty(1, 2, 90, 33, device="cuda", dtype=q.dtype)[..., :32].copy_(q)
    assert torch.equal(ft.forgetting_attention(odd, k, v, g, head_first=True), want)
    assert torch.equal(ft.forgetting_attention(q, k, v, g, head_first=True, seq_start=torch.zeros(1, dtype=torch.int32, device="cuda")), want)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        other = ft.forgetting_attention(q, k, v, g, head_first=True)
    torch.cuda.current_stream().wait_stream(s)
    assert torch.equal(other, want)
    leaves = [x.requires_grad_() for x in (q, k, v, g)]
    out = ft.forgetting_attention(q, k, v, g, head_first=True)
    _equal(torch.autograd.grad(out, leaves, do, retain_graph=True), torch.autograd.grad(out, leaves, do))
    with pytest.raises(RuntimeError, match="backward through the graph a second time"):
        torch.autograd.grad(out, leaves, do)


@pytest.mark.parametrize("H,D,shared", [(1, 16, False), (5, 64, False), (12, 128, False), (3, 32, True)])
def test_qk_norm_threshold(ft, H, D, shared):
    """The kernel against the tensor expression it replaces, rounding for rounding."""
    general = import_module("forgetting_transformer.ops.forgetting_attention")._qk_norm_threshold_general
    n = D if shared else H * D
    wq, wk = (torch.randn(n, device="cuda", requires_grad=True) for _ in range(2))
    got = ft.qk_norm_threshold(wq, wk, H, D, 1777, -10.0, shared)
    want = general(wq, wk, H, D, 1777, -10.0, shared)
    assert torch.equal(got, want) and got.shape == want.shape and not got.requires_grad
    with torch.no_grad():
        wk[n - 1] = float("nan")
    assert torch.equal(ft.qk_norm_threshold(wq, wk, H, D, 1777, -10.0, shared).isnan(), general(wq, wk, H, D, 1777, -10.0, shared).isnan())


@pytest.mark.parametrize("rows,G,D", [(1, 1, 16), (3, 3, 64), (700, 12, 64), (5000, 5, 32), (4097, 33, 64), (40000, 2, 16), (33001, 1, 128)])
@pytest.mark.parametrize("gated", [False, True])
def test_norm_backward_plans(ft, rows, G, D, gated):
    """Backward of the norms over the ways it is cut: one or several column blocks, row lanes, rows per lane, one or two passes over the
    partial weight gradients.  dweight sums `rows` products of O(1) 16-bit values: fp32 rounding of the partial sums gives
    about sqrt(rows) * 2^-24 of its scale, well below the 1e-4 asked; dx and dg are one rounding to bf16 (2^-8 of their own scale)."""
    from oracle import fox_oracle as O
    gen = torch.Generator(device="cuda").manual_seed(rows + G)
    rnd = lambda: torch.randn(rows, G * D, generator=gen, device="cuda").bfloat16()
    x, g, do = rnd().requires_grad_(), rnd().requires_grad_() if gated else None, rnd()
    w = (torch.rand(G * D, generator=gen, device="cuda") + 0.5).requires_grad_()
    leaves = [x, w] + ([g] if gated else [])
    y = ft.group_norm_gated(x, g, w, None, "sigmoid", is_rms_norm=True, num_groups=G) if gated else ft.group_norm(x, w, is_rms_norm=True, num_groups=G)
    got = torch.autograd.grad(y, leaves, do)
    ref = [t.detach().double().requires_grad_() for t in leaves]
    yr = O.group_norm_gated_ref(ref[0], ref[2], ref[1], G, 1e-6, "sigmoid") if gated else O.group_norm_ref(ref[0], ref[1], G, 1e-5)
    want = torch.autograd.grad(yr, ref, do.double())
    for name, a, b, tol in zip(("dx", "dw", "dg"), got, want, (2 ** -8, 1e-4, 2 ** -8)):
        assert (a.double() - b).abs().max() <= tol * b.abs().max(), name


@pytest.mark.parametrize("B,T,H,D", [(1, 1, 1, 16), (2, 3, 5, 64), (1, 257, 3, 128), (2, 4001, 12, 64), (1, 20000, 16, 64)])
def test_token_shift_strips(ft, B, T, H, D):
    """Token shift over the strip lengths a size selects, last strips of one step included (fp32 reference, one rounding to bf16)."""
    from oracle import fox_oracle as O
    gen = torch.Generator(device="cuda").manual_seed(T)
    x = torch.randn(B, T, H, D, generator=gen, device="cuda").bfloat16().requires_grad_()
    p, c = (torch.rand(B, T, H, generator=gen, device="cuda").requires_grad_() for _ in range(2))
    do = torch.randn(B, T, H, D, generator=gen, device="cuda").bfloat16()
    out = ft.token_shift(x, p, c)
    ref = [t.detach().float().requires_grad_() for t in (x, p, c)]
    out_ref = O.token_shift_ref(*ref)
    for a, b in zip((out,) + torch.autograd.grad(out, [x, p, c], do), (out_ref,) + torch.autograd.grad(out_ref, ref, do.float())):
        assert (a.float() - b).abs().max() <= 2 ** -8 * b.abs().max()


def test_forward_mode_is_refused(ft):
    """The operators have no forward-mode rule: a dual tensor raises, its tangent is not dropped."""
    import torch.autograd.forward_ad as fwd
    q, k, v, g, _, _ = make_inputs(1, 2, 70, 70, 64, device="cuda", head_first=True, seed=3)
    with fwd.dual_level(), pytest.raises((RuntimeError, NotImplementedError)):
        ft.forgetting_attention(fwd.make_dual(q, torch.ones_like(q)), k, v, g, head_first=True)


@pytest.mark.parametrize("true,false", [(1, 0), (np.True_, np.False_)])
def test_flags_count_by_their_truth_value(ft, true, false):
    """Configurations hold switches as 0/1 or numpy.bool_: they mean what `if flag` means, also with fp32 logits, where nothing in the
    types tells logits from log gates."""
    q, k, v, _, _, _ = make_inputs(1, 2, 70, 70, 64, device="cuda", head_first=False, seed=11)
    logits, w = torch.randn(1, 70, 2, device="cuda") + 1, torch.rand(128, device="cuda") + 0.5
    call = lambda **kw: ft.forgetting_attention_norm_gate(q, k, v, kw.pop("g", logits), None, w, **kw)
    want, got = call(fgate_is_logit=True), call(fgate_is_logit=true, head_first=false)
    assert isinstance(got, tuple) and len(got) == 2
    _equal(got, want)
    log_gates = torch.nn.functional.logsigmoid(logits)
    _equal([call(g=log_gates, fgate_is_logit=false)], [call(g=log_gates)])
    hf = [x.transpose(1, 2) for x in (q, k, v, log_gates)]
    _equal([ft.forgetting_attention(*hf, head_first=true)], [ft.forgetting_attention(*hf, head_first=True)])
    wq, wk = torch.rand(64, device="cuda"), torch.rand(64, device="cuda")
    for H in (1, 5):
        got, want = ft.qk_norm_threshold(wq, wk, H, 64, 99, -10.0, true), ft.qk_norm_threshold(wq, wk, H, 64, 99, -10.0, True)
        assert got.shape == want.shape == () and torch.equal(got, want)
    assert ft.qk_norm_threshold(wq, wk, 1, 64, 99, -10.0, false).shape == (1,)


def test_flags_without_a_truth_value_raise(ft):
    q, k, v, g, _, _ = make_inputs(1, 2, 70, 70, 64, device="cuda", head_first=False, seed=11)
    w, both = torch.rand(128, device="cuda"), np.array([True, False])
    with pytest.raises(ValueError, match="ambiguous"):
        ft.forgetting_attention(q, k, v, g, head_first=both)
    with pytest.raises(ValueError, match="ambiguous"):
        ft.forgetting_attention_norm_gate(q, k, v, g, None, w, fgate_is_logit=both)
    with pytest.raises(ValueError, match="ambiguous"):
        ft.qk_norm_threshold(w, w, 2, 64, 99, -10.0, both)


@pytest.mark.parametrize("thr", [-7.125, -7])   # values no other test uses: the first call with each is the one under inference mode
def test_a_number_as_threshold_in_inference_mode_then_training(ft, thr):
    """The (B, H) tensor made of a number serves later calls too: evaluating first must not leave a tensor training cannot save."""
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    q, k, v, g, do, _ = make_inputs(1, 3, 150, 150, 64, device="cuda", head_first=True, seed=4, gate_mean=1.0)
    with torch.inference_mode():
        first = ft.forgetting_attention(q, k, v, g, head_first=True, adaptive_threshold=thr)
    leaves = [x.requires_grad_() for x in (q, k, v, g)]
    out = ft.forgetting_attention(*leaves, head_first=True, adaptive_threshold=thr)
    assert torch.equal(out, first)
    ref = F.ForgettingAttention.apply(*leaves, None, True, None, thr)
    _equal(_grads(out, leaves, do), _grads(ref, leaves, do))


def test_other_threads_run_while_an_operator_is_called(ft):
    """The interpreter lock is free during allocation and launches.  With a switch interval that never expires, another thread gets
    its turn only when the calling thread gives the lock up by itself; nothing else in the loops below does."""
    import sys
    import threading
    q, k, v, g, _, _ = make_inputs(1, 2, 64, 64, 64, device="cuda", head_first=True, seed=2)
    x, w, p = torch.randn(1, 64, 2, 64, device="cuda").bfloat16(), torch.rand(128, device="cuda"), torch.rand(1, 64, 2, device="cuda")
    cache = [torch.zeros(1, 2, 128, 64, device="cuda").bfloat16(), torch.zeros(1, 2, 128, 64, device="cuda").bfloat16(),
             torch.zeros(1, 2, 128, device="cuda")]
    from forgetting_transformer.ops import _native
    ext = _native.load()
    x2 = x.view(1, 64, 128)
    calls = {"attention": (ext.attention, (q, k, v, g, True, None, None, None, False)),
             "decode": (ext.attention, (q[:, :, :1], k, v, g, True, None, None, None, False)),
             "attention_norm_gate": (ext.attention_norm_gate, (q, k, v, g, None, w, 2, 1e-6, True, None, None, None, False)),
             "norm": (ext.norm, (x2, None, w, 2, 1e-6, 2)), "token_shift": (ext.token_shift, (x, p, p)),
             "qk_norm_threshold": (ext.qk_norm_threshold, (w, w, 2, 64, 99, -10.0, False)),
             "cache_append": (ext.cache_append, (*cache, k, v, g, 0))}
    interval, ready = sys.getswitchinterval(), threading.Event()
    stuck = []
    with torch.no_grad():
        for name, (fn, args) in calls.items():
            assert fn(*args) is not None, name
            torch.cuda.synchronize()
            turns, stop = [0], [False]
            ready.clear()

            def other():
                ready.set()
                while not stop[0]:
                    turns[0] += 1
                    time.sleep(0)       # gives the lock back after every turn

            thread = threading.Thread(target=other)
            try:
                sys.setswitchinterval(1000.0)
                thread.start()
                ready.wait()
                time.sleep(0.05)        # it waits for the lock by now, with the interval above
                before = turns[0]
                for _ in range(3000):
                    fn(*args)
                    if turns[0] > before:
                        break
                else:
                    stuck.append(name)
            finally:
                stop[0] = True
                sys.setswitchinterval(interval)
                thread.join()
            torch.cuda.synchronize()
    assert not stuck, stuck


def test_function_transforms_are_refused(ft):
    """No operator has rules for functorch's transforms: a call under one raises, whether its tensors are the transformed ones or
    are only closed over."""
    q, k, v, g, _, _ = make_inputs(1, 2, 70, 70, 64, device="cuda", head_first=True, seed=3)
    x, w, p = torch.randn(2, 30, 128, device="cuda").bfloat16(), torch.rand(128, device="cuda"), torch.rand(2, 30, 2, device="cuda")
    x4 = x.view(2, 30, 2, 64)
    calls = [lambda t: ft.forgetting_attention(q + t.to(q.dtype) if t is not None else q, k, v, g, head_first=True),
             lambda t: ft.forgetting_attention_norm_gate(q + t.to(q.dtype) if t is not None else q, k, v, g, None, w, head_first=True),
             lambda t: ft.group_norm(x + t.to(x.dtype) if t is not None else x, w, is_rms_norm=True, num_groups=2),
             lambda t: ft.token_shift(x4 + t.to(x.dtype) if t is not None else x4, p, p)]
    ts = torch.zeros(3, device="cuda")
    for call in calls:
        for used in (True, False):
            with pytest.raises(RuntimeError, match="setup_context"):
                torch.func.vmap(lambda t: call(t if used else None).sum() + t)(ts)
            with pytest.raises(RuntimeError, match="setup_context"):
                torch.func.grad(lambda t: call(t if used else None).float().sum() + t)(ts[0])


class _Tagged(torch.Tensor):
    """A subclass without a dispatch of its own: what torch calls __torch_function__ keeps the type."""


def test_tensor_subclasses_keep_their_type(ft):
    """As the general path does, a result laid out like a subclass instance is one."""
    from forgetting_transformer.ops.token_shift import TokenShift
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    q, k, v, g, _, _ = make_inputs(1, 2, 70, 70, 64, device="cuda", head_first=True, seed=3)
    tagged = q.as_subclass(_Tagged)
    out, ref = ft.forgetting_attention(tagged, k, v, g, head_first=True), F.ForgettingAttention.apply(tagged, k, v, g, None, True, None, None)
    assert type(out) is type(ref) is _Tagged and torch.equal(out, ref)
    x, p = q.transpose(1, 2).contiguous().as_subclass(_Tagged), torch.rand(1, 70, 2, device="cuda")
    out, ref = ft.token_shift(x, p, p), TokenShift.apply(x, p, p)
    assert type(out) is type(ref) is _Tagged and torch.equal(out, ref)
    par = torch.nn.Parameter(q)
    assert type(ft.forgetting_attention(par, k, v, g, head_first=True)) is torch.Tensor


def test_dispatch_modes_see_the_calls_operations(ft):
    """Under a dispatch mode the general path runs, whose allocations and copies the mode can see, refuse or replace."""
    from torch.utils._python_dispatch import TorchDispatchMode

    class Names(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            names.append(str(func))
            return func(*args, **(kwargs or {}))

    cache, names = ft.FgateDynamicCache(max_length=8), []
    new = [torch.randn(1, 2, 3, 64, device="cuda").bfloat16() for _ in range(2)] + [torch.randn(1, 2, 3, device="cuda")]
    cache.update(*new, 0)
    with Names():
        got = cache.update(*new, 0)
    assert sum("copy_" in n for n in names) == 3
    for a, b in zip(got, new):
        assert torch.equal(a, torch.cat([b, b], dim=2))


def _repacked(t):   # as a copy to pinned host memory and back leaves it: the values, in a plain contiguous tensor
    return torch.empty(t.shape, dtype=t.dtype, device=t.device).copy_(t)


@pytest.mark.parametrize("head_first", [True, False])
@pytest.mark.parametrize("gated", [True, False])
@pytest.mark.parametrize("general", [True, False])
def test_saved_tensors_that_come_back_in_another_layout(ft, head_first, gated, general):
    """Saved-tensor hooks may hand back tensors with other strides: the gradients are the same."""
    from forgetting_transformer.ops import _lib
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    B, H, T, D = 2, 3, 90, 32
    swap = (lambda x: x.transpose(1, 2)) if head_first else (lambda x: x)
    q, k, v, gate, do = (swap(torch.randn(B, T, H, D, device="cuda").bfloat16()) for _ in range(5))
    logits, w = swap(torch.randn(B, T, H, device="cuda") + 2), torch.rand(H * D, device="cuda") + 0.5
    leaves = [x.requires_grad_() for x in (q, k, v, logits, w) + ((gate,) if gated else ())]

    def grads():
        if general:
            hf = [x if head_first else x.transpose(1, 2) for x in (q, k, v, logits, gate)]
            y = F.ForgettingAttentionNormGate.apply(*hf[:4], hf[4] if gated else None, w, None, None, None,
                                                    _lib.ACT_SIGMOID if gated else _lib.ACT_NONE, 1e-6, True)[0]
            y = y if head_first else y.transpose(1, 2)
        else:
            y = ft.forgetting_attention_norm_gate(q, k, v, logits, gate if gated else None, w, head_first=head_first, fgate_is_logit=True)[0]
        return lambda: torch.autograd.grad(y, leaves, do)

    want = grads()()
    with torch.autograd.graph.saved_tensors_hooks(_repacked, lambda t: t):
        later = grads()
    _equal(later(), want)


def _padded(t):       # the values, with gaps behind every row
    if t.dim() < 2:
        return t
    return torch.empty((*t.shape[:-1], t.shape[-1] + 8), dtype=t.dtype, device=t.device)[..., :t.shape[-1]].copy_(t)


def _turned(t):       # the values, with the last axis outermost in memory
    return torch.empty((t.shape[-1], *t.shape[:-1]), dtype=t.dtype, device=t.device).movedim(0, -1).copy_(t) if t.dim() > 1 else t


def _some_turned(t):  # of tensors with the same shape only every second one
    _some_turned.calls = getattr(_some_turned, "calls", 0) + 1
    return _turned(t) if _some_turned.calls % 2 else t


@pytest.mark.parametrize("pack", [_repacked, _padded, _turned, _some_turned])
@pytest.mark.parametrize("head_first", [True, False])
def test_every_backward_with_saved_tensors_in_other_layouts(ft, pack, head_first):
    B, T, H, D = 2, 45, 3, 32
    rnd = lambda *s: torch.randn(*s, device="cuda").bfloat16().requires_grad_()
    x, gate, k, v = rnd(B, T, H * D), rnd(B, T, H * D), rnd(B, T, H, D), rnd(B, T, H, D)
    w, p, c = torch.rand(H * D, device="cuda", requires_grad=True), *(torch.rand(B, T, H, device="cuda", requires_grad=True) for _ in range(2))
    logits, do = torch.randn(B, T, H, device="cuda", requires_grad=True), torch.randn(B, T, H, D, device="cuda").bfloat16()
    thr, ss = torch.full((B, H), -9.0, device="cuda"), torch.tensor([0, 7], device="cuda")
    leaves = [x, gate, k, v, w, p, c, logits]

    def grads():
        q = ft.group_norm_gated(x, gate, w, is_rms_norm=True, num_groups=H).view(B, T, H, D)
        ks = ft.token_shift(k, p, c)
        if head_first:
            out, _ = ft.forgetting_attention_from_logits(q.transpose(1, 2), ks.transpose(1, 2), v.transpose(1, 2), logits.transpose(1, 2),
                                                         head_first=True, seq_start=ss, adaptive_threshold=thr)
            out = out.transpose(1, 2)
        else:
            out = ft.forgetting_attention(q, ks, v, torch.nn.functional.logsigmoid(logits), seq_start=ss, adaptive_threshold=thr)
        return lambda: torch.autograd.grad(out, leaves, do)

    want = grads()()
    with torch.autograd.graph.saved_tensors_hooks(pack, lambda t: t):
        later = grads()
    _equal(later(), want)


@pytest.mark.parametrize("head_first", [True, False])
def test_bounds_of_a_backward_whose_forward_ran_before_the_recording(ft, head_first):
    """record_pruning_bounds collects every backward made inside the block, whichever path its forward took."""
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    B, H, T, D = 1, 2, 700, 64
    q, k, v, g, do, _ = make_inputs(B, H, T, T, D, device="cuda", head_first=head_first, seed=6, gate_mean=-1.0)
    leaves = [x.requires_grad_() for x in (q, k, v, g)]
    call = lambda: ft.forgetting_attention(*leaves, head_first=head_first, adaptive_threshold=-12.0)
    with F.record_pruning_bounds() as want:
        torch.autograd.grad(call(), leaves, do)
    out = call()
    with F.record_pruning_bounds() as got:
        torch.autograd.grad(out, leaves, do, retain_graph=True)
    torch.autograd.grad(out, leaves, do)          # after the block: nothing is recorded
    assert len(want) == 2 and len(got) == 1 and set(got[0]) == {"dq_first_block", "kv_end_row"}
    for name, t in got[0].items():
        assert t.dtype == torch.int32 and torch.equal(t, want[1][name])
    plain = ft.forgetting_attention(*leaves, head_first=head_first)
    with F.record_pruning_bounds() as got:       # no threshold, no bounds
        torch.autograd.grad(plain, leaves, do)
    assert got == []


def test_qk_norm_threshold_with_a_tensor_tolerance(ft):
    """A tolerance that is a tensor is added as one: per head, without waiting for the device, and under stream capture."""
    H, D = 4, 64
    wq, wk = torch.randn(H * D, device="cuda"), torch.randn(H * D, device="cuda")
    base = ft.qk_norm_threshold(wq, wk, H, D, 512, 0.0)
    tol = torch.tensor(-10.0, device="cuda")
    rows = torch.linspace(-12, -9, H, device="cuda")
    assert torch.equal(ft.qk_norm_threshold(wq, wk, H, D, 512, rows), base + rows)
    mode = torch.cuda.get_sync_debug_mode()
    torch.cuda.set_sync_debug_mode("warn")
    try:
        with warnings.catch_warnings(record=True) as seen:
            warnings.simplefilter("always")
            got = ft.qk_norm_threshold(wq, wk, H, D, 512, tol)
    finally:
        torch.cuda.set_sync_debug_mode(mode)
    assert torch.equal(got, base + tol) and not [w for w in seen if "synchroniz" in str(w.message)]
    assert torch.equal(ft.qk_norm_threshold(wq, wk, H, D, 512, np.float32(-10.0)), base + tol)


@pytest.mark.parametrize("M", [1, 70])
def test_a_threshold_that_requires_grad(ft, M):
    """A trainable threshold has no gradient but makes the result part of a graph: backward runs and leaves it without one."""
    q, k, v, g, do, _ = make_inputs(1, 2, M, 70, 64, device="cuda", head_first=True, seed=3)
    thr = torch.full((2,), -20.0, device="cuda", requires_grad=True)
    out = ft.forgetting_attention(q, k, v, g, head_first=True, adaptive_threshold=thr)
    assert out.requires_grad and torch.autograd.grad(out, [thr], do, allow_unused=True) == (None,)
    with torch.no_grad():
        assert torch.equal(ft.forgetting_attention(q, k, v, g, head_first=True, adaptive_threshold=thr), out)


# grids the paired kernel takes instead of two key splits, grids that stay split, and one that is neither
@pytest.mark.parametrize("B,H,M,N,D", [(2, 12, 1024, 1024, 128), (2, 16, 333, 5333, 128), (4, 32, 1024, 1024, 64)])
@pytest.mark.parametrize("epilogue,general", [(False, False), (True, False), (False, True)])
def test_no_scratch_is_kept_for_the_backward(ft, B, H, M, N, D, epilogue, general):
    """What a forward leaves behind is its results: the scratch of key splits is gone when the call returns."""
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    q, k, v, g, do, _ = make_inputs(B, H, M, N, D, device="cuda", head_first=True, seed=1, gate_mean=1.0)
    for x in (q, k, v, g):
        x.requires_grad_()
    w = torch.rand(H * D, device="cuda")
    def call():
        if general:
            return F.ForgettingAttention.apply(q, k, v, g, None, True, None, None)
        return ft.forgetting_attention_norm_gate(q, k, v, g, None, w, head_first=True) if epilogue else ft.forgetting_attention(q, k, v, g, head_first=True)
    call()
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    out = call()
    kept = torch.cuda.memory_allocated() - before
    rows = B * H * M * D * 2
    need = rows + 4 * B * H * (M + N) + ((rows + 4 * B * H * M) if epilogue else 0)
    assert kept <= need + (2 << 20) + 8 * 512, (kept, need)     # (the allocator hands out large blocks with up to 1 MiB left over)
    del out


def _layer_step(ft, x, k, v, logits, w):
    B, T, H, D = k.shape
    q = ft.group_norm(x, w, is_rms_norm=True, num_groups=H).view(B, T, H, D)
    return ft.forgetting_attention_norm_gate(q, k, v, logits, None, w, fgate_is_logit=True, adaptive_threshold=-20.0)[0]


@pytest.mark.parametrize("reentrant", [True, False])
def test_under_activation_checkpointing(ft, reentrant):
    from torch.utils.checkpoint import checkpoint
    B, T, H, D = 2, 130, 3, 64
    rnd = lambda *s: torch.randn(*s, device="cuda").bfloat16().requires_grad_()
    leaves = [rnd(B, T, H * D), rnd(B, T, H, D), rnd(B, T, H, D), torch.randn(B, T, H, device="cuda", requires_grad=True),
              torch.rand(H * D, device="cuda", requires_grad=True)]
    do = torch.randn(B, T, H, D, device="cuda").bfloat16()
    grads = []
    for again in (False, True):
        y = checkpoint(_layer_step, ft, *leaves, use_reentrant=reentrant) if again else _layer_step(ft, *leaves)
        grads.append([y.detach()] + [g.clone() for g in _backward_into_leaves(y, leaves, do)])
    _equal(*grads)


def _backward_into_leaves(y, leaves, do):
    for t in leaves:
        t.grad = None
    y.backward(do)
    return [t.grad for t in leaves]


def test_steps_on_several_threads_and_streams(ft):
    """Forward and backward from four threads at once, each on its own stream and device buffers, against the same steps one by one."""
    import threading
    B, T, H, D = 1, 300, 2, 64
    def inputs(i):
        gen = torch.Generator(device="cuda").manual_seed(i)
        rnd = lambda *s: torch.randn(*s, generator=gen, device="cuda")
        return [rnd(B, T + i, H * D).bfloat16(), rnd(B, T + i, H, D).bfloat16(), rnd(B, T + i, H, D).bfloat16(), rnd(B, T + i, H) + 1,
                rnd(H * D).abs() + 0.5], rnd(B, T + i, H, D).bfloat16()
    def step(i):
        leaves, do = inputs(i)
        leaves = [t.requires_grad_() for t in leaves]
        y = _layer_step(ft, *leaves)
        return [y.detach()] + list(torch.autograd.grad(y, leaves, do))
    want = [step(i) for i in range(4)]
    torch.cuda.synchronize()
    got, errors = [[None] * 5 for _ in range(4)], []

    def work(i):
        try:
            with torch.cuda.stream(torch.cuda.Stream()):
                for r in range(5):
                    got[i][r] = step(i)
                torch.cuda.current_stream().synchronize()
        except Exception as e:   # noqa: BLE001
            errors.append(e)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for i in range(4):
        for r in range(5):
            _equal(got[i][r], want[i])


@pytest.mark.filterwarnings("ignore")   # the tracer's remarks
def test_traces_are_refused(ft):
    """The general path's shape checks refuse the tracer's sizes; the native path must not turn the result into a constant instead."""
    q, k, v, g, _, _ = make_inputs(1, 2, 70, 70, 64, device="cuda", head_first=True, seed=3)
    with pytest.raises(AssertionError, match="head dims"):
        torch.jit.trace(lambda a, b, c, d: ft.forgetting_attention(a, b, c, d, head_first=True), (q, k, v, g), check_trace=False)
    x, w = torch.randn(2, 30, 128, device="cuda").bfloat16(), torch.rand(128, device="cuda")
    with pytest.raises(AssertionError, match="group size"):
        torch.jit.trace(lambda a, b: ft.group_norm(a, b, is_rms_norm=True, num_groups=2), (x, w), check_trace=False)


@pytest.mark.parametrize("first,thr", [("transform", -9.0625), ("mode", -9.1875)])   # numbers no other test uses
def test_a_number_as_threshold_under_a_transform_or_mode_first(ft, first, thr):
    """The tensor made of a number serves later calls: one that a transform wrapped, or a mode replaced, must not stay behind."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    F = import_module("forgetting_transformer.ops.forgetting_attention")
    q, k, v, g, _, _ = make_inputs(1, 2, 300, 300, 64, device="cuda", head_first=True, seed=3, gate_mean=-1.0)
    want = ft.forgetting_attention(q, k, v, g, head_first=True, adaptive_threshold=torch.full((1, 2), thr, device="cuda"))
    call = lambda: ft.forgetting_attention(q, k, v, g, head_first=True, adaptive_threshold=thr)
    if first == "transform":
        with pytest.raises(RuntimeError, match="setup_context"):
            torch.func.grad(lambda t: call().float().sum() + t)(torch.zeros((), device="cuda"))
    else:
        with FakeTensorMode():       # (what a call does there before anything looks at its tensors)
            F._native_threshold(thr, q, True)
    got = F._native_threshold(thr, q, True)
    assert type(got) is torch.Tensor and got.data_ptr() != 0 and (got == thr).all()
    assert torch.equal(call(), want)


@pytest.mark.parametrize("logits", [False, True])
def test_gates_changed_between_forward_and_backward(ft, logits):
    """The backward does not read log gates, so their buffer is free again after the forward; logits it does read."""
    q, k, v, g, do, _ = make_inputs(1, 2, 70, 70, 64, device="cuda", head_first=True, seed=3)
    leaves = [x.requires_grad_() for x in (q, k, v)]

    def call():
        return ft.forgetting_attention_from_logits(*leaves, g, head_first=True)[0] if logits else ft.forgetting_attention(*leaves, g, head_first=True)

    want, out = torch.autograd.grad(call(), leaves, do), call()
    g.zero_()
    if logits:
        with pytest.raises(RuntimeError, match="modified by an inplace operation"):
            torch.autograd.grad(out, leaves, do)
    else:
        _equal(torch.autograd.grad(out, leaves, do), want)


def test_log_gates_are_not_kept_for_the_backward(ft):
    B, H, T, D = 1, 16, 1 << 16, 16
    q, k, v, g, _, _ = make_inputs(B, H, 128, T, D, device="cuda", head_first=True, seed=3)
    q.requires_grad_()
    g_bytes = g.numel() * 4
    out = ft.forgetting_attention(q, k, v, g, head_first=True)
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    del g
    assert before - torch.cuda.memory_allocated() >= g_bytes
    del out


def test_a_negated_view_joins_the_cache_with_its_values(ft):
    """The imaginary part of a conjugate is a view that stands for the negated memory."""
    z = torch.complex(torch.randn(1, 2, 3, device="cuda"), torch.randn(1, 2, 3, device="cuda"))
    g = z.conj().imag
    assert g.is_neg()
    k = torch.randn(1, 2, 3, 64, device="cuda").bfloat16()
    got = ft.FgateDynamicCache().update(k, k, g, 0)
    assert torch.equal(got[2], -z.imag)
