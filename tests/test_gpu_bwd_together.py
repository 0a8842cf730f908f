"""The backward of small grids, dQ and dK/dV in one launch (fox_attn_bwd), against the same stages one after the other, bit for bit (both walks form
one and the same delta), and against the oracle."""
import ctypes as C

import pytest
import torch

from conftest import assert_parity, make_inputs
from oracle import fox_oracle as O

pytestmark = pytest.mark.gpu


class _Problem:
    """A backward's inputs, after their forward, and an argument block for results of its own at every call."""

    def __init__(self, B, H, M, N, D, dtype, thr, seq, head_first):
        from forgetting_transformer.ops import _lib
        from forgetting_transformer.ops.forgetting_attention import _view
        self._lib, self.view, self.lib = _lib, _view, _lib.load()
        q, k, v, g, do, ss = make_inputs(B, H, M, N, D, dtype=dtype, device="cuda", head_first=head_first, seed=N + D, gate_mean=1.0, seq_start=seq)
        if not head_first:   # head-first views of (B, T, H, D) memory
            q, k, v, g, do = (x.transpose(1, 2) for x in (q, k, v, g, do))
        self.q, self.k, self.v, self.g, self.do, self.ss, self.shape = q, k, v, g, do, ss, (B, H, M, N)
        self.dims = _lib.Dims(B, H, M, N, D, 0 if dtype == torch.bfloat16 else 1)
        self.stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
        self.thr = None if thr is None else torch.full((B, H), thr, device="cuda")
        self.c, self.lse, self.o = torch.empty(B, H, N, device="cuda"), torch.empty(B, H, M, device="cuda"), torch.empty_like(q)
        _lib.check(self.lib.fox_cumsum_fwd(g.data_ptr(), *g.stride(), _ptr(ss), self.c.data_ptr(), B, H, N, self.stream), "scan")
        fwd = _lib.FwdArgs(self.dims, _view(q), _view(k), _view(v), _view(self.o), self.c.data_ptr(), self.lse.data_ptr(), _ptr(ss), _ptr(self.thr), D ** -0.5,
                           None, None, 0)
        _lib.check(self.lib.fox_attn_fwd(C.byref(fwd), self.stream), "fwd")

    def args(self, dg=None):
        B, H, M, N = self.shape
        grads = [torch.full_like(x, float("nan")) for x in (self.q, self.k, self.v)]
        tmp = [torch.full((B, H, n), float("nan"), device="cuda") for n in (M, M, N)]   # delta, drow, dlog_lambda
        views = (self.view(x) for x in (self.q, self.k, self.v, self.o, self.do, *grads))
        a = self._lib.BwdArgs(self.dims, *views, self.c.data_ptr(), self.lse.data_ptr(), _ptr(self.ss), _ptr(self.thr), self.q.shape[-1] ** -0.5,
                              *(x.data_ptr() for x in tmp), _ptr(dg), *(dg.stride() if dg is not None else (0, 0, 0)), None, None)
        return a, grads, tmp

    def one_launch(self, args):
        yes = C.c_int32(-1)
        self._lib.check(self.lib.fox_attn_bwd_one_launch(C.byref(args), C.byref(yes)), "fox_attn_bwd_one_launch")
        return yes.value == 1

    def call(self, name, *args):
        self._lib.check(getattr(self.lib, name)(*args, self.stream), name)


def _ptr(x):
    return None if x is None else x.data_ptr()


def _run(B, H, M, N, D, dtype, thr, seq, head_first):
    p = _Problem(B, H, M, N, D, dtype, thr, seq, head_first)
    res = []
    for together in (False, True):
        dg = torch.full((B, H, N), float("nan"), device="cuda")
        args, grads, tmp = p.args(dg)
        if together:
            assert p.one_launch(args)
            p.call("fox_attn_bwd", C.byref(args))
        else:
            p.call("fox_attn_bwd_dq", C.byref(args))
            p.call("fox_attn_bwd_dkdv", C.byref(args))
            p.call("fox_cumsum_bwd", tmp[2].data_ptr(), dg.data_ptr(), *dg.stride(), _ptr(p.ss), B, H, N)
        res.append((*grads, dg, *tmp))
    for name, a, b in zip(("dq", "dk", "dv", "dlog_fgate", "delta", "drow", "dlog_lambda"), *res):
        assert torch.isfinite(b).all()
        assert torch.equal(a, b), name
    # (One or two query rows: a gradient is one or two products of three 16-bit roundings each, 3 * 2^-9 = 6e-3 and up to twice that of a scale that
    # is such a product itself.  The parity tests hold degenerate shapes to the bar with a floor on the scale; here the comparison above is the check.)
    if thr is None and M > 2:
        ref = O.forgetting_attention_ref_grads(p.q, p.k, p.v, p.g, p.do, head_first=True, seq_start=p.ss)
        for r in res:
            for name, x, y in zip(("dq", "dk", "dv", "dlog_fgate"), r, ref[1:]):
                assert_parity(name, x, y, rows=name != "dlog_fgate")


@pytest.mark.parametrize("D", [16, 32, 64])
@pytest.mark.parametrize("B,H,M,N,thr,seq,head_first,dtype", [
    (1, 1, 2, 2, None, None, True, torch.bfloat16),
    (1, 3, 1, 130, None, None, True, torch.bfloat16),                # a query tile less than key tiles
    (2, 3, 127, 129, None, [0, 60], False, torch.float16),           # query and key tiles that do not line up
    (2, 4, 128, 640, None, [0, 300], True, torch.bfloat16),
    (3, 5, 777, 777, None, [0, 5, 299], True, torch.float16),
    (2, 2, 300, 1000, -5.0, None, False, torch.bfloat16),
    (2, 8, 2000, 2000, None, None, False, torch.bfloat16),
    (2, 32, 1000, 1000, -3.0, [0, 128], False, torch.bfloat16),      # 512 tiles of either kind: the largest grid at head dim 64
])
def test_against_one_after_the_other(B, H, M, N, thr, seq, head_first, dtype, D):
    _run(B, H, M, N, D, dtype, thr, seq, head_first)


@pytest.mark.parametrize("logit", [None, torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,H,M,N,seq", [(2, 3, 130, 300, [0, 200]), (1, 3, 700, 1500, None), (1, 2, 1000, 8300, [17])])   # one span of each width: 256 threads, 1024, 1024 with sixteen positions each
def test_strided_gate_gradients(B, H, M, N, seq, logit):
    """The reverse scan with the row sums added, into gates and logits that lie as (B, T, H), against the stages on their own."""
    p = _Problem(B, H, M, N, 32, torch.bfloat16, None, seq, False)
    as_bth = lambda x: x.transpose(1, 2).contiguous().transpose(1, 2)
    res = []
    for together in (False, True):
        dg = as_bth(torch.full((B, H, N), float("nan"), device="cuda", dtype=logit or torch.float32))
        args, _, tmp = p.args(dg if logit is None else None)
        assert p.one_launch(args)
        if not together:
            p.call("fox_attn_bwd_dq", C.byref(args))
            p.call("fox_attn_bwd_dkdv", C.byref(args))
        if logit is None:
            if together:
                p.call("fox_attn_bwd", C.byref(args))
            else:
                p.call("fox_cumsum_bwd", tmp[2].data_ptr(), dg.data_ptr(), *dg.stride(), _ptr(p.ss), B, H, N)
        else:
            x = as_bth((p.g * 3 + 2).to(logit))
            gates = (x.data_ptr(), {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}[logit], *x.stride())
            if together:
                p.call("fox_attn_bwd_logits", C.byref(args), *gates, dg.data_ptr(), *dg.stride())
            else:
                p.call("fox_gate_cumsum_bwd", tmp[2].data_ptr(), *gates, _ptr(p.ss), dg.data_ptr(), *dg.stride(), B, H, N)
        res.append((dg, tmp[1], tmp[2]))
    for a, b in zip(*res):
        assert torch.isfinite(a).all() and torch.equal(a, b)


@pytest.mark.parametrize("logit", [None, torch.bfloat16, torch.float16, torch.float32])
def test_strided_gate_gradients_of_long_rows(logit):
    """The same where a row is two spans of sixteen positions a thread."""
    test_strided_gate_gradients(1, 2, 300, 16500, [17], logit)
