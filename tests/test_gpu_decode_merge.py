"""Generation steps whose splits are merged by the one that arrives last (fox_attn_decode_counted): bit for bit what the two launches give, whatever
runs before, beside or after them."""
import ctypes as C
import threading

import pytest
import torch

from conftest import make_inputs

pytestmark = pytest.mark.gpu


@pytest.fixture()
def ft():
    import forgetting_transformer as ft
    assert torch.cuda.is_available(), "these tests need the MI355X"
    return ft


SHAPES = [(1, 12, 1500, 64), (1, 1, 5000, 128), (2, 3, 4000, 16), (1, 5, 700, 32), (4, 32, 600, 64), (4, 32, 700, 64),   # (the last three: one workgroup a pair)
          (1, 64, 1000, 64), (1, 4, 8192, 128), (1, 64, 1200, 64)]   # 256 workgroups in splits of 4 and of 64, the most of either, and more than 256
MERGES = {(1, 12, 1500, 64), (1, 1, 5000, 128), (2, 3, 4000, 16), (1, 64, 1000, 64), (1, 4, 8192, 128)}


def _inputs(shape, seq=None):
    B, H, N, D = shape
    q, k, v, g, _, ss = make_inputs(B, H, 1, N, D, device="cuda", seed=N, gate_mean=2.0, seq_start=seq)
    return q, k, v, g, ss


def _two_launches(q, k, v, g, ss, counters=None):
    from forgetting_transformer.ops import _lib
    from forgetting_transformer.ops.forgetting_attention import _view
    lib = _lib.load()
    B, H, _, D = q.shape
    dims = _lib.Dims(B, H, 1, k.shape[2], D, 0)
    need = C.c_int64(0)
    _lib.check(lib.fox_attn_decode_workspace_bytes(C.byref(dims), C.byref(need)), "workspace")
    ws, o, lse = torch.empty(max(need.value, 16), dtype=torch.uint8, device="cuda"), torch.empty_like(q), torch.empty(B, H, device="cuda")
    args = _lib.FwdArgs(dims, _view(q), _view(k), _view(v), _view(o), None, lse.data_ptr(), None if ss is None else ss.data_ptr(), None, D ** -0.5, None,
                        ws.data_ptr(), need.value)
    stream = C.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.fox_attn_decode_counted(C.byref(args), g.data_ptr(), *g.stride(), None if counters is None else counters.data_ptr(), stream), "decode")
    return o, lse


def _counters(shape):
    from forgetting_transformer.ops import _lib
    B, H, N, D = shape
    n = C.c_int32(-1)
    _lib.check(_lib.load().fox_attn_decode_counters(C.byref(_lib.Dims(B, H, 1, N, D, 0)), C.byref(n)), "fox_attn_decode_counters")
    return n.value


def test_no_counters_where_the_splits_do_not_merge(ft):
    """A step of more workgroups than CUs allocates its output and its workspace, and no block of counters on a stream that has none."""
    q, k, v, g, _ = _inputs((1, 64, 1200, 64))
    with torch.no_grad(), torch.cuda.stream(torch.cuda.Stream()):
        before = torch.cuda.memory_stats()["allocation.all.allocated"]
        ft.forgetting_attention(q, k, v, g, head_first=True)
        assert torch.cuda.memory_stats()["allocation.all.allocated"] - before == 2
    torch.cuda.synchronize()


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("padded", [False, True])
def test_same_bits_and_zero_counters(ft, shape, padded):
    B, H, N, D = shape
    ins = _inputs(shape, [(N * (b + 1)) // B for b in range(B)] if padded else None)   # the last one: nothing but padding
    want = _two_launches(*ins)
    assert _counters(shape) == (B * H if shape in MERGES else 0)
    counters = torch.zeros(B * H, dtype=torch.int32, device="cuda")
    for _ in range(3):
        got = _two_launches(*ins, counters=counters)
        assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
        assert not counters.any()
    q, k, v, g, ss = ins
    with torch.no_grad():
        for _ in range(20):
            out = ft.forgetting_attention(q, k, v, g, head_first=True, seq_start=ss)
        assert torch.equal(out, want[0])


@pytest.mark.parametrize("shape", [(1, 3, 16391, 64), (1, 3, 67584, 16), (3, 1, 10240, 128), (1, 64, 1200, 64)])
def test_counters_are_left_alone_where_none_are_asked_for(ft, shape):
    """Also where the plan without padding would merge in the launch and the one with it would not."""
    ins = _inputs(shape)
    assert _counters(shape) == 0
    counters = torch.full((shape[0] * shape[1],), 7, dtype=torch.int32, device="cuda")
    want, got = _two_launches(*ins), _two_launches(*ins, counters=counters)
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1]) and (counters == 7).all()


def test_streams_threads_and_graphs(ft):
    ins = [_inputs(s) for s in (*SHAPES[:3], SHAPES[7])]
    want = [_two_launches(*x)[0] for x in ins]
    torch.cuda.synchronize()
    bad = []

    def work(stream):
        with torch.no_grad(), torch.cuda.stream(stream):
            for i in range(60):
                q, k, v, g, _ = ins[i % 4]
                out = ft.forgetting_attention(q, k, v, g, head_first=True)
                if i % 7 == 0 and not torch.equal(out, want[i % 4]):
                    bad.append(i)

    shared = torch.cuda.Stream()
    owned = torch.cuda.Stream()
    streams = [torch.cuda.current_stream(), shared, shared, torch.cuda.Stream(), torch.cuda.ExternalStream(owned.cuda_stream)]
    threads = [threading.Thread(target=work, args=(s,)) for s in streams]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    torch.cuda.synchronize()
    assert not bad

    q, k, v, g, _ = ins[0]
    q = q.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.no_grad(), torch.cuda.graph(graph):
        out = ft.forgetting_attention(q, k, v, g, head_first=True)
    for r in range(4):
        q.copy_(torch.randn(q.shape, device="cuda").to(q.dtype))
        with torch.no_grad():
            eager = ft.forgetting_attention(q, k, v, g, head_first=True)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)
