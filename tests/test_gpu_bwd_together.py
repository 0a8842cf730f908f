"""The backward of small grids, dQ and dK/dV in one launch (fox_attn_bwd), against the same stages one after the other, bit for bit (both walks form
one and the same delta), and against the oracle."""
import ctypes as C

import pytest
import torch

from conftest import assert_parity, make_inputs
from oracle import fox_oracle as O

pytestmark = pytest.mark.gpu


def _run(B, H, M, N, D, dtype, thr, seq, head_first):
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib = _lib.load()
    q, k, v, g, do, ss = make_inputs(B, H, M, N, D, dtype=dtype, device="cuda", head_first=head_first, seed=N + D, gate_mean=1.0, seq_start=seq)
    if not head_first:   # head-first views of (B, T, H, D) memory
        q, k, v, g, do = (x.transpose(1, 2) for x in (q, k, v, g, do))
    dims = _lib.Dims(B, H, M, N, D, 0 if dtype == torch.bfloat16 else 1)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda x: None if x is None else x.data_ptr()
    t = None if thr is None else torch.full((B, H), thr, device="cuda")
    c, lse, o = torch.empty(B, H, N, device="cuda"), torch.empty(B, H, M, device="cuda"), torch.empty_like(q)
    _lib.check(lib.fox_cumsum_fwd(g.data_ptr(), *g.stride(), ptr(ss), c.data_ptr(), B, H, N, stream), "scan")
    fwd = _lib.FwdArgs(dims, _view(q), _view(k), _view(v), _view(o), c.data_ptr(), lse.data_ptr(), ptr(ss), ptr(t), D ** -0.5, None, None, 0)
    _lib.check(lib.fox_attn_fwd(C.byref(fwd), stream), "fwd")
    res = []
    for together in (False, True):
        dq, dk, dv = (torch.full_like(x, float("nan")) for x in (q, k, v))
        tmp = [torch.full((B, H, n), float("nan"), device="cuda") for n in (M, M, N)]
        dg = torch.full((B, H, N), float("nan"), device="cuda")
        args = _lib.BwdArgs(dims, *(_view(x) for x in (q, k, v, o, do, dq, dk, dv)), c.data_ptr(), lse.data_ptr(), ptr(ss), ptr(t), D ** -0.5,
                            *(x.data_ptr() for x in tmp), dg.data_ptr(), *dg.stride(), None, None)
        if together:
            _lib.check(lib.fox_attn_bwd(C.byref(args), stream), "bwd")
        else:
            _lib.check(lib.fox_attn_bwd_dq(C.byref(args), stream), "dq")
            _lib.check(lib.fox_attn_bwd_dkdv(C.byref(args), stream), "dkdv")
            _lib.check(lib.fox_cumsum_bwd(tmp[2].data_ptr(), dg.data_ptr(), *dg.stride(), ptr(ss), B, H, N, stream), "scan")
        res.append((dq, dk, dv, dg, *tmp))
    for name, a, b in zip(("dq", "dk", "dv", "dlog_fgate", "delta", "drow", "dlog_lambda"), *res):
        assert torch.isfinite(b).all()
        assert torch.equal(a, b), name
    # (One or two query rows: a gradient is one or two products of three 16-bit roundings each, 3 * 2^-9 = 6e-3 and up to twice that of a scale that
    # is such a product itself.  The parity tests hold degenerate shapes to the bar with a floor on the scale; here the comparison above is the check.)
    if thr is None and M > 2:
        ref = O.forgetting_attention_ref_grads(q, k, v, g, do, head_first=True, seq_start=ss)
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
