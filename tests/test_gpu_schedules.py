"""GPU tests of how the attention work is dealt out over workgroups: the launch order of the tiles, the key splits and
the variants that a shape selects, each at the sizes where its bookkeeping has an edge.  Every case is compared with the
oracle over all (batch, head) pairs at the operator's bar, so a tile that is visited twice, never, or for the
wrong pair shows."""
import ctypes as C

import pytest
import torch

from conftest import assert_parity, make_inputs
from oracle import fox_oracle as O
from test_gpu_parity import fa, run_case  # noqa: F401  (fa is a fixture)

pytestmark = pytest.mark.gpu


# (pairs, length, head dim): one group or several, of equal or unequal size, pairs that divide over the XCDs or do not;
# grids that just fill two workgroups per CU (32 tiles x 16 pairs: the folded order) and just exceed that
@pytest.mark.parametrize("B,H,T,D", [(1, 136, 2048, 128), (1, 131, 2048, 128), (1, 24, 4096, 128), (1, 16, 4096, 32),
                                     (1, 15, 4300, 32), (3, 11, 2000, 16), (1, 1, 4096, 64)])
def test_launch_order(fa, B, H, T, D):
    torch.cuda.empty_cache()
    run_case(fa, B, H, T, T, D, seed=H + T, gate_mean=1.0)


# rows shorter than a cache line with the heads of a token side by side: two groups; one pair after the other under a threshold
@pytest.mark.parametrize("B,H,T,D,thr", [(1, 512, 1030, 16, None), (1, 131, 1020, 16, -10.0), (1, 91, 1500, 16, -10.0), (3, 45, 1024, 32, -6.0)])
def test_launch_order_of_shared_lines(fa, B, H, T, D, thr):
    torch.cuda.empty_cache()
    run_case(fa, B, H, T, T, D, seed=H + T, gate_mean=1.0, head_first=False, thr=thr)


# few query rows behind many keys: key splits that fill the chip once, also where one split more would not fit
@pytest.mark.parametrize("B,H,M,N,D", [(2, 16, 333, 1100, 32), (1, 8, 129, 3000, 64), (3, 7, 300, 2000, 16)])
def test_key_splits(fa, B, H, M, N, D):
    run_case(fa, B, H, M, N, D, seed=M + N, gate_mean=2.0)


# three splits at head dims up to 64 where two would leave some CUs with one workgroup: tiles of equal weight, a causal triangle
@pytest.mark.parametrize("B,H,M,N", [(8, 8, 333, 1500), (5, 8, 600, 2000), (1, 10, 2600, 2600)])
@pytest.mark.parametrize("D", [16, 64])
def test_three_key_splits(fa, B, H, M, N, D):
    run_case(fa, B, H, M, N, D, seed=M + N, gate_mean=2.0)


# few query tiles: two groups of waves share a tile's walk.  Walks of one tile (group 1 has none), of odd and even length, with three,
# four and five interior tiles (where the pipelined path begins), with left padding inside the walk and without a diagonal-free part
@pytest.mark.parametrize("B,H,M,N", [(1, 2, 257, 513), (2, 3, 512, 512), (1, 3, 449, 577), (1, 3, 513, 576), (2, 2, 640, 640),
                                     (1, 2, 300, 512), (1, 3, 900, 1025), (1, 5, 1500, 1533), (3, 5, 777, 777), (1, 16, 2100, 2100)])
@pytest.mark.parametrize("D,dtype", [(32, torch.bfloat16), (64, torch.float16), (128, torch.bfloat16)])
def test_paired_forward(fa, B, H, M, N, D, dtype):
    run_case(fa, B, H, M, N, D, dtype=dtype, seed=M + D, gate_mean=2.0)
    run_case(fa, B, H, M, N, D, dtype=dtype, seed=M + D, gate_mean=0.0, head_first=False, seq_start=[(N * (2 * b + 1)) // (2 * B) for b in range(B)])


@pytest.mark.parametrize("D", [32, 128])
def test_paired_forward_with_a_negative_scale(fa, D):   # every tile takes the masked path
    run_case(fa, 1, 2, 700, 900, D, seed=3, gate_mean=2.0, sm_scale=-0.1)


# grids beyond one tile per CU and in place of two key splits, on both sides of the rule: the output alone.  384 tiles are paired
# from 2048 keys on, 511 from 4080 on, 512 never; 240 and 252 tiles would take two splits, which the pairing replaces up to 2560 keys
@pytest.mark.parametrize("B,H,T,paired", [(2, 16, 1500, False), (1, 17, 1921, True), (3, 10, 1024, True), (1, 12, 2560, True), (1, 12, 2561, False),
                                          (1, 24, 2047, False), (1, 24, 2048, True), (2, 16, 2048, False), (1, 7, 9300, True)])
@pytest.mark.parametrize("D,dtype", [(64, torch.bfloat16), (128, torch.float16)])
def test_paired_forward_of_larger_grids(fa, B, H, T, paired, D, dtype):
    from forgetting_transformer.ops import _lib
    lib, plan = _lib.load(), C.c_int32(-1)
    dims = _lib.Dims(B, H, T, T, D, int(dtype == torch.float16))
    _lib.check(lib.fox_attn_fwd_plan(C.byref(dims), 0, None, C.byref(plan), None), "fox_attn_fwd_plan")
    assert plan.value == paired
    q, k, v, g, _, ss = make_inputs(B, H, T, T, D, dtype=dtype, device="cuda", head_first=False, seed=T, gate_mean=2.0)
    with torch.no_grad():
        out = fa(q, k, v, g)
    assert_parity("out", out, O.forgetting_attention_ref(q, k, v, g))


@pytest.mark.parametrize("B,H,T,D", [(3, 10, 1024, 64), (1, 3, 600, 32), (1, 17, 1921, 128)])
def test_paired_forward_with_and_without_scratch(fa, B, H, T, D):
    """The plan asks for no scratch where the paired kernel runs; a caller that brings what key splits would need gets the same
    results, bit for bit."""
    from test_zz_no_alloc import _fwd_pair
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib = _lib.load()
    (own, noalloc), _, (q, k, v, g, _) = _fwd_pair(lib, _lib, _view, B, H, T, T, D, seed=5)
    with torch.no_grad():
        out = fa(q, k, v, g, head_first=True)
    assert torch.equal(out, own[0]) and torch.equal(out, noalloc[0]) and torch.equal(own[1], noalloc[1])
