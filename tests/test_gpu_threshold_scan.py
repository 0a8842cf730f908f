"""The "auto" threshold with the scan of the gates beside it (fox_auto_threshold_scan), against the two on their own, bit for bit.  The first shape streams
too little for that and takes the two launches; the others have rows of one and several spans of its 256 threads, with ends inside a span."""
import ctypes as C

import pytest
import torch

from conftest import make_inputs
from oracle import fox_oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("logit", [None, torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,H,M,N,D,dtype,padded", [(2, 3, 200, 300, 64, torch.bfloat16, False), (16, 32, 500, 513, 32, torch.float16, True),
                                                    (8, 16, 1000, 1000, 128, torch.bfloat16, False), (3, 60, 2048, 2049, 64, torch.bfloat16, True),
                                                    (4, 100, 4100, 4100, 16, torch.bfloat16, False)])
def test_against_the_two_launches(B, H, M, N, D, dtype, padded, logit):
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib = _lib.load()
    q, k, _, g, _, ss = make_inputs(B, H, M, N, D, dtype=dtype, device="cuda", seed=N, gate_mean=1.0, head_first=False,
                                    seq_start=[(N * b) // B for b in range(B)] if padded else None)
    q, k, g = (x.transpose(1, 2) for x in (q, k, g))   # strided gates
    kind = {None: 2, torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}[logit]
    if logit is not None:
        g = (g * 3 + 2).to(logit)
    dims = _lib.Dims(B, H, M, N, D, 0 if dtype == torch.bfloat16 else 1)
    one_launch = C.c_int32(-1)
    _lib.check(lib.fox_auto_threshold_scan_one_launch(C.byref(dims), C.byref(one_launch)), "one launch")
    assert one_launch.value == (N != 300)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ssp = None if ss is None else ss.data_ptr()
    res = []
    for together in (False, True):
        thr, scratch = torch.full((B, H), float("nan"), device="cuda"), torch.full((B, H, 3), -1, dtype=torch.int32, device="cuda")
        c, lg = (torch.full((B, H, N), float("nan"), device="cuda") for _ in range(2))
        views = C.byref(_view(q)), C.byref(_view(k))
        if together:
            gates = _lib.Gates(g.data_ptr(), logit is not None, kind, *g.stride(), lg.data_ptr() if logit is not None else None)
            _lib.check(lib.fox_auto_threshold_scan(C.byref(dims), *views, D ** -0.5, thr.data_ptr(), scratch.data_ptr(), C.byref(gates), ssp,
                                                   c.data_ptr(), stream), "together")
        else:
            _lib.check(lib.fox_auto_threshold(C.byref(dims), *views, D ** -0.5, thr.data_ptr(), scratch.data_ptr(), stream), "threshold")
            if logit is None:
                _lib.check(lib.fox_cumsum_fwd(g.data_ptr(), *g.stride(), ssp, c.data_ptr(), B, H, N, stream), "scan")
            else:
                _lib.check(lib.fox_gate_cumsum_fwd(g.data_ptr(), kind, *g.stride(), ssp, lg.data_ptr(), c.data_ptr(), B, H, N, stream), "scan")
        res.append((thr, c) + ((lg,) if logit is not None else ()))
    for a, b in zip(*res):
        assert torch.isfinite(b).all() and torch.equal(a, b)


@pytest.mark.parametrize("B,H,M,N,one", [(2, 3, 1, 1, False), (1, 5, 512, 512, False), (3, 1, 511, 514, False), (2, 2, 3, 1021, False), (1, 3, 5, 4363, True),
                                         (1, 2, 1, 40000, False), (2, 130, 100, 613, None)])   # (None: from head dim 64 on)
@pytest.mark.parametrize("D", [16, 64, 128])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_threshold_of_short_rows_and_few_queries(B, H, M, N, one, D, dtype):
    """One workgroup a (batch, head) up to 1024 rows of q and k, as many for q as it has rows beyond; the scan beside the norms or after them."""
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib = _lib.load()
    q, k, _, g, _, _ = make_inputs(B, H, M, N, D, dtype=dtype, device="cuda", seed=N + D, head_first=False)
    q, k, g = (x.transpose(1, 2) for x in (q, k, g))
    k[B - 1, H - 1, N - 1] = 3.0   # the last row has the largest norm
    dims, yes = _lib.Dims(B, H, M, N, D, 0 if dtype == torch.bfloat16 else 1), C.c_int32(-1)
    _lib.check(lib.fox_auto_threshold_scan_one_launch(C.byref(dims), C.byref(yes)), "one launch")
    assert yes.value == (D >= 64 if one is None else one)
    stream, views = C.c_void_p(torch.cuda.current_stream().cuda_stream), (C.byref(_view(q)), C.byref(_view(k)))
    thr, both = torch.full((B, H), float("nan"), device="cuda"), torch.full((B, H), float("nan"), device="cuda")
    c, want, scratch = torch.empty(B, H, N, device="cuda"), torch.empty(B, H, N, device="cuda"), torch.full((B, H, 3), -1, dtype=torch.int32, device="cuda")
    _lib.check(lib.fox_auto_threshold(C.byref(dims), *views, D ** -0.5, thr.data_ptr(), scratch.data_ptr(), stream), "threshold")
    gates = _lib.Gates(g.data_ptr(), False, 2, *g.stride(), None)
    _lib.check(lib.fox_auto_threshold_scan(C.byref(dims), *views, D ** -0.5, both.data_ptr(), scratch.data_ptr(), C.byref(gates), None, c.data_ptr(), stream), "scan")
    _lib.check(lib.fox_cumsum_fwd(g.data_ptr(), *g.stride(), None, want.data_ptr(), B, H, N, stream), "scan alone")
    assert torch.equal(thr, both) and torch.equal(c, want)
    ref = O.auto_threshold(q, k, D ** -0.5)   # rounded to 16 bits after every operation; the row norms may sit on either side of a rounding
    assert (thr - ref).abs().max().item() <= 2 * 2.0 ** (-7 if dtype == torch.bfloat16 else -10) * ref.abs().max().item()
