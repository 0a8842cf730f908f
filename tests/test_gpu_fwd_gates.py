"""The forward that forms the cumulative sums of its rows itself (fox_attn_fwd_gates): against the scan and the forward from its result, bit
for bit in everything they write, at row lengths around its steps (a wave, 256 and 512 threads, the longest row it takes), and against
the oracle.  Both sum in fp64 and round once, so only a sum within 1e-9 of a rounding boundary could differ."""
import ctypes as C

import pytest
import torch

from conftest import assert_parity, make_inputs
from oracle import fox_oracle as O

pytestmark = pytest.mark.gpu

DTYPES = {None: 2, torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}


def _both(B, H, M, N, D, dtype, thr, seq, logit, strided, faster=1):
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib = _lib.load()
    q, k, v, g, _, ss = make_inputs(B, H, M, N, D, dtype=dtype, device="cuda", seed=N + D, gate_mean=1.0, seq_start=seq)
    if logit is not None:
        g = (g * 3 + 2).to(logit)
    if strided:   # (B, T, H) memory
        g = g.transpose(1, 2).contiguous().transpose(1, 2)
    dims = _lib.Dims(B, H, M, N, D, 0 if dtype == torch.bfloat16 else 1)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    yes, need = C.c_int32(-1), C.c_int64(0)
    _lib.check(lib.fox_attn_fwd_takes_gates(C.byref(dims), thr is not None, C.byref(yes)), "takes_gates")
    assert yes.value == faster
    _lib.check(lib.fox_attn_fwd_workspace_bytes(C.byref(dims), C.byref(need)), "workspace")
    ws = torch.empty(max(need.value, 16), dtype=torch.uint8, device="cuda")
    t = None if thr is None else torch.full((B, H), thr, device="cuda")
    ptr = lambda x: None if x is None else x.data_ptr()
    res = []
    for own in (False, True):
        o, lse = torch.full_like(q, float("nan")), torch.full((B, H, M), float("nan"), device="cuda")
        c, lg = torch.full((B, H, N), float("nan"), device="cuda"), torch.full((B, H, N), float("nan"), device="cuda")
        first = torch.full((B, H, (M + 127) // 128), -1, dtype=torch.int32, device="cuda")
        args = _lib.FwdArgs(dims, _view(q), _view(k), _view(v), _view(o), c.data_ptr(), lse.data_ptr(), ptr(ss), ptr(t), D ** -0.5,
                            first.data_ptr(), ws.data_ptr(), need.value)
        if own:
            gates = _lib.Gates(g.data_ptr(), logit is not None, DTYPES[logit], *g.stride(), lg.data_ptr() if logit is not None else None)
            _lib.check(lib.fox_attn_fwd_gates(C.byref(args), C.byref(gates), None, stream), "fox_attn_fwd_gates")
        else:
            if logit is None:
                rc = lib.fox_cumsum_fwd(g.data_ptr(), *g.stride(), ptr(ss), c.data_ptr(), B, H, N, stream)
            else:
                rc = lib.fox_gate_cumsum_fwd(g.data_ptr(), DTYPES[logit], *g.stride(), ptr(ss), lg.data_ptr(), c.data_ptr(), B, H, N, stream)
            _lib.check(rc, "scan")
            _lib.check(lib.fox_attn_fwd(C.byref(args), stream), "fox_attn_fwd")
        res.append((o, lse, c, first) + (() if logit is None else (lg,)))
    for a, b in zip(*res):
        assert torch.equal(a, b)
    if thr is None:
        lf = g if logit is None else torch.nn.functional.logsigmoid(g.float())
        assert_parity("out", res[1][0], O.forgetting_attention_ref(q, k, v, lf, head_first=True, seq_start=ss))


@pytest.mark.parametrize("N,M", [(2, 2), (63, 63), (64, 64), (65, 2), (256, 256), (257, 130), (513, 513), (1025, 1025), (3584, 1800), (3583, 3583)])
@pytest.mark.parametrize("D,dtype", [(16, torch.bfloat16), (32, torch.float16), (64, torch.bfloat16), (128, torch.bfloat16)])
def test_against_the_scan(N, M, D, dtype):
    B, H = (2, 3) if N < 1025 else (2, 15) if N == 1025 else (2, 9)   # long rows: enough query tiles that the keys are not split
    _both(B, H, M, N, D, dtype, None, [0, N // 2], None, D == 64)


@pytest.mark.parametrize("thr", [None, -3.0])
@pytest.mark.parametrize("logit", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("B,H,M,N,D", [(2, 3, 700, 700, 64), (1, 3, 200, 333, 16), (8, 40, 300, 300, 128)])
def test_from_logits_and_pruned(B, H, M, N, D, logit, thr):
    _both(B, H, M, N, D, torch.bfloat16, thr, None, logit, True)
    _both(B, H, M, N, D, torch.bfloat16, thr, [min(n, N) for n in range(0, 97 * B, 97)], None, False)


@pytest.mark.parametrize("B,H,M,N,D,thr", [(8, 32, 130, 1600, 64, None), (2, 16, 2048, 2048, 64, None), (8, 24, 500, 500, 128, None), (8, 32, 130, 3500, 64, -10.0)])
def test_shapes_it_takes_where_a_scan_is_faster(B, H, M, N, D, thr):
    _both(B, H, M, N, D, torch.bfloat16, thr, None, None, True, faster=0)


def test_shapes_it_does_not_take():
    from forgetting_transformer.ops import _lib
    lib = _lib.load()
    yes = C.c_int32(-1)
    for B, H, M, N, D in [(2, 3, 1, 200, 64), (8, 40, 200, 3585, 64), (1, 2, 300, 3000, 128), (16, 32, 1025, 1025, 64)]:
        dims = _lib.Dims(B, H, M, N, D, 0)
        _lib.check(lib.fox_attn_fwd_takes_gates(C.byref(dims), 0, C.byref(yes)), "takes_gates")
        assert yes.value == 0
    x = torch.zeros(1, 2, 300, 128, device="cuda", dtype=torch.bfloat16)
    from forgetting_transformer.ops.forgetting_attention import _view
    g = torch.zeros(1, 2, 3000, device="cuda")
    kv = torch.zeros(1, 2, 3000, 128, device="cuda", dtype=torch.bfloat16)
    args = _lib.FwdArgs(_lib.Dims(1, 2, 300, 3000, 128, 0), _view(x), _view(kv), _view(kv), _view(x.clone()), None, g.data_ptr(), None, None, 0.1, None, None, 0)
    assert lib.fox_attn_fwd_gates(C.byref(args), C.byref(_lib.Gates(g.data_ptr(), 0, 2, *g.stride(), None)), None, None) == -1
