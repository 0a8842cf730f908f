"""The kernels of token-by-token generation: one query row straight from the log gates (no graph, no threshold), its merge of key
splits, and the append of new tokens to the cache."""
import ctypes as C

import pytest
import torch

from conftest import assert_parity, make_inputs
from oracle import fox_oracle as O

pytestmark = pytest.mark.gpu


@pytest.fixture
def ft():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    import forgetting_transformer
    return forgetting_transformer


# a batch of keys per wave is 4096 / D, a workgroup takes four: one key, edges of a batch and of a workgroup's share, several
# batches per wave (no more splits to give), one split (many heads)
@pytest.mark.parametrize("B,H,N,D", [(1, 1, 1, 64), (1, 3, 63, 64), (2, 2, 65, 64), (1, 2, 255, 64), (1, 2, 257, 64), (1, 12, 1500, 64),
                                     (2, 3, 33, 128), (1, 2, 129, 128), (2, 2, 9001, 128), (1, 2, 1025, 16), (2, 2, 70000, 16),
                                     (3, 5, 700, 32), (1, 1, 40000, 64), (16, 130, 300, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gate_mean", [3.0, -1.0])
def test_single_query(ft, B, H, N, D, dtype, gate_mean):
    ss = [(N * i) // (2 * B) for i in range(B)]
    ss[-1] = N if B > 2 else N - 1                     # a row with nothing to see, or only its own key
    q, k, v, g, _, ss = make_inputs(B, H, 1, N, D, dtype=dtype, device="cuda", head_first=True, seq_start=ss, seed=N + D, gate_mean=gate_mean)
    ref = O.forgetting_attention_ref(q, k, v, g, head_first=True, seq_start=ss)
    with torch.no_grad():
        out = ft.forgetting_attention(q, k, v, g, head_first=True, seq_start=ss)
        swap = [x.transpose(1, 2).contiguous() for x in (q, k, v, g)]
        other = ft.forgetting_attention(*swap, seq_start=ss)
    assert_parity("out", out, ref)
    assert torch.equal(other.transpose(1, 2), out)     # strided gates and rows: the same arithmetic


@pytest.mark.parametrize("N,at", [(3000, 1234), (300, 100), (300, 299)])
def test_single_query_behind_a_closed_gate(ft, N, at):
    """A log gate of -inf hides every key left of it and nothing else."""
    q, k, v, g, _, _ = make_inputs(1, 2, 1, N, 64, device="cuda", head_first=True, seed=5, gate_mean=2.0)
    g[:, :, at] = float("-inf")
    with torch.no_grad():
        out = ft.forgetting_attention(q, k, v, g, head_first=True)
        ref = O.forgetting_attention_ref(q, k[:, :, at:], v[:, :, at:], g[:, :, at:].clamp(min=-50), head_first=True)
    assert_parity("out", out, ref)


# how many splits a row is cut into (decode_splits): 192 pairs are the fewest that go without a merge, 191 and 257 are not enough and too many, 461 and 512
# fill the CUs twice; one batch of keys a wave or several; with padding, which never goes without
@pytest.mark.parametrize("B,H,N,D", [(1, 191, 700, 128), (1, 192, 700, 128), (16, 16, 1409, 64), (1, 257, 641, 128), (1, 460, 700, 64), (1, 461, 700, 64), (4, 128, 520, 128),
                                     (3, 16, 2049, 128), (3, 16, 9000, 16), (8, 12, 2300, 64)])
@pytest.mark.parametrize("padded", [False, True])
def test_single_query_splits(ft, B, H, N, D, padded):
    ss = [(N * i) // B for i in range(B)] if padded else None
    q, k, v, g, _, ss = make_inputs(B, H, 1, N, D, device="cuda", head_first=True, seq_start=ss, seed=N + H, gate_mean=2.0)
    with torch.no_grad():
        out = ft.forgetting_attention(q, k, v, g, head_first=True, seq_start=ss)
    assert_parity("out", out, O.forgetting_attention_ref(q, k, v, g, head_first=True, seq_start=ss))


# shapes whose number of splits is another with padding than without; the scratch lies inside a larger allocation, of the size that the query asks for
# and one piece smaller, where the call makes do with fewer splits
@pytest.mark.parametrize("B,H,N,D", [(4, 12, 16384, 128), (8, 12, 8192, 128), (8, 16, 6500, 128), (16, 8, 10000, 64), (4, 16, 13000, 128), (4, 16, 9232, 128),
                                     (10, 32, 16384, 128), (12, 32, 16384, 128), (10, 32, 1808, 128), (33, 1, 64513, 16), (2, 520, 16384, 128)])
@pytest.mark.parametrize("padded", [False, True])
def test_splits_stay_inside_their_scratch(ft, B, H, N, D, padded):
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib, stream = _lib.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    gen = torch.Generator(device="cuda").manual_seed(N)   # (up to 2 * 10^9 elements: drawn there)
    q, k, v = (torch.randn(B, H, T, D, generator=gen, device="cuda", dtype=torch.bfloat16) for T in (1, N, N))
    g = torch.nn.functional.logsigmoid(torch.randn(B, H, N, generator=gen, device="cuda") + 2.0)
    ss = torch.tensor([(N * i) // (4 * B) for i in range(B)], device="cuda") if padded else None
    ref = O.forgetting_attention_ref(q, k, v, g, head_first=True, seq_start=ss)
    dims, need = _lib.Dims(B, H, 1, N, D, _lib.DTYPE_BF16), C.c_int64(0)
    _lib.check(lib.fox_attn_decode_workspace_bytes(C.byref(dims), C.byref(need)), "fox_attn_decode_workspace_bytes")
    guard = 4 << 20   # more than the partial results of 64 splits of any of these shapes would run over
    for room in (need.value, need.value - 16):
        block, o = torch.full((guard + need.value + guard,), 0xA5, dtype=torch.uint8, device="cuda"), torch.full_like(q, float("nan"))
        args = _lib.FwdArgs(dims, _view(q), _view(k), _view(v), _view(o), None, None, None if ss is None else ss.data_ptr(), None, D ** -0.5, None,
                            block.data_ptr() + guard, room)
        _lib.check(lib.fox_attn_decode(C.byref(args), g.data_ptr(), *g.stride(), stream), "fox_attn_decode")
        assert (block[:guard] == 0xA5).all() and (block[guard + room:] == 0xA5).all()
        assert_parity("out", o, ref)
        if room == need.value:
            with torch.no_grad():
                assert torch.equal(ft.forgetting_attention(q, k, v, g, head_first=True, seq_start=ss), o)


# one workgroup of sixteen waves takes a (batch, head) whole: two batches of keys with few heads, up to four with many, and
# the first sizes beyond
@pytest.mark.parametrize("B,H,N,D", [(2, 3, 257, 64), (2, 3, 512, 64), (2, 3, 513, 64), (1, 3, 129, 128), (2, 2, 2048, 16), (2, 2, 600, 32),
                                     (4, 32, 1024, 64), (4, 32, 1025, 64), (5, 26, 300, 128), (8, 63, 2047, 32), (8, 64, 700, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_single_query_in_one_workgroup(ft, B, H, N, D, dtype):
    ss = [(N * i) // B for i in range(B)]
    ss[-1] = N if B > 2 else N - 1
    q, k, v, g, _, ss = make_inputs(B, H, 1, N, D, dtype=dtype, device="cuda", head_first=True, seq_start=ss, seed=N + D, gate_mean=1.0)
    with torch.no_grad():
        out = ft.forgetting_attention(q, k, v, g, head_first=True, seq_start=ss)
    assert_parity("out", out, O.forgetting_attention_ref(q, k, v, g, head_first=True, seq_start=ss))


# through the C ABI: splits and their merge, one workgroup of sixteen waves, one key; with the scratch and without (one workgroup of
# four waves walks the whole cache), with lse and without, gates with strides; the last sequence is all padding
@pytest.mark.parametrize("B,H,N,D", [(3, 2, 5000, 64), (3, 2, 400, 64), (2, 3, 9001, 128), (2, 2, 3000, 16), (3, 40, 700, 32), (2, 1, 1, 64)])
def test_decode_entry_point(ft, B, H, N, D):
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib, stream = _lib.load(), C.c_void_p(torch.cuda.current_stream().cuda_stream)
    ss = [(N * i) // (2 * B) for i in range(B - 1)] + [N]
    q, k, v, g, _, ss = make_inputs(B, H, 1, N, D, device="cuda", head_first=True, seq_start=ss, seed=N, gate_mean=3.0)
    gates = g.transpose(1, 2).contiguous().transpose(1, 2)       # (B, H, N) with the heads adjacent
    dims, need = _lib.Dims(B, H, 1, N, D, _lib.DTYPE_BF16), C.c_int64(0)
    _lib.check(lib.fox_attn_decode_workspace_bytes(C.byref(dims), C.byref(need)), "fox_attn_decode_workspace_bytes")
    scores = (k.double() @ q.double().transpose(-1, -2)).squeeze(-1) / D ** 0.5
    scores += g.double().flip(-1).cumsum(-1).flip(-1) - g.double()          # the gates behind each key
    scores = scores.masked_fill(torch.arange(N, device="cuda") < ss[:, None, None], float("-inf"))
    lse_ref = scores.logsumexp(-1)
    ref = O.forgetting_attention_ref(q, k, v, g, head_first=True, seq_start=ss)
    for scratch in (True, False):
        for with_lse in (True, False):
            ws = torch.empty(max(need.value, 16), dtype=torch.uint8, device="cuda")
            o, lse = torch.full_like(q, float("nan")), torch.full((B, H), float("nan"), device="cuda")
            args = _lib.FwdArgs(dims, _view(q), _view(k), _view(v), _view(o), None, lse.data_ptr() if with_lse else None, ss.data_ptr(), None,
                                1.0 / D ** 0.5, None, ws.data_ptr() if scratch and need.value else None, need.value if scratch else 0)
            _lib.check(lib.fox_attn_decode(C.byref(args), gates.data_ptr(), *gates.stride(), stream), "fox_attn_decode")
            assert_parity("out", o, ref, context=(scratch, with_lse))
            assert (o[-1] == 0).all()
            if not with_lse:
                assert lse.isnan().all()
                continue
            assert (lse[-1] == float("-inf")).all()
            # fp32: D products summed (scores of a few units), the bias of the keys that count (tens at most) rounded once, 2^x and log
            assert (lse[:-1].double() - lse_ref[:-1]).abs().max() <= 2e-5, (scratch, (lse[:-1].double() - lse_ref[:-1]).abs().max())


@pytest.mark.parametrize("D,T,dtype", [(64, 1, torch.bfloat16), (128, 1, torch.float16), (16, 7, torch.bfloat16), (40, 300, torch.float16),
                                       (12, 3, torch.bfloat16), (64, 2, torch.float32)])
def test_cache_append(ft, D, T, dtype):
    """Appending against concatenation, from strided sources; head dims and types the kernel does not take go through torch."""
    B, H = 2, 3
    rnd = lambda n: torch.randn(B, n, H, D, device="cuda").to(dtype).transpose(1, 2)
    gates = lambda n: -torch.rand(B, n, H, device="cuda").transpose(1, 2)
    cache, parts = ft.FgateDynamicCache(min_capacity=64), []
    for n in (T, 5, T):
        parts.append((rnd(n), rnd(n), gates(n)))
        got = cache.update(*parts[-1], 0)
        for a, b, c in zip(got, zip(*parts), cache[0]):
            assert torch.equal(a, torch.cat(b, dim=2)) and c.data_ptr() == a.data_ptr()
    version = cache._key_buf[0]._version
    cache.crop(T + 5)
    with torch.inference_mode():
        got = cache.update(*parts[2], 0)
    assert torch.equal(got[1], torch.cat([p[1] for p in parts], dim=2)) and cache._key_buf[0]._version > version
