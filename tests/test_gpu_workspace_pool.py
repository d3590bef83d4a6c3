"""The split-K workspace: one for the functions that the extension launches and those that go through ctypes, another
for SBVRLinear."""
import pytest
import torch

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")


def _encoded(rows, K, S=4, G=128, L=16, seed=0):
    from sbvr import synth
    return [t.to(DEV) for t in synth.random_encoding(rows, K, S, G, L, seed=seed)]


def test_a_stream_warmed_by_one_function_is_warm_for_all():
    """After the functional linear (ctypes) the products of encoded operands (extension) find their accumulators on that
    stream: no allocation but their outputs', inside a capture as well, and right replays."""
    import sbvr
    from sbvr import _sbvr_hip_ops as ops, hip
    N, K = 1024, 2048
    w = _encoded(N, K, seed=1)
    l = _encoded(1, K, seed=2)
    t = _encoded(K, N, seed=3)                                 # (the transposed weight)
    x = torch.randn((2, K), generator=torch.Generator().manual_seed(4)).to(torch.float16).to(DEV)
    none = torch.zeros(0, dtype=torch.float16, device=DEV)
    lib = hip._load()
    assert lib.sbvr_hip_row_deq_mm_T_workspace(2, N) > 0 and lib.sbvr_hip_mm_T_workspace(1, N) > 0
    want = [sbvr._sbvr_row_deq_mm_T(x, *t, none, bvr_len=128), sbvr._sbvr_mm_T(*l, *w, none, bvr_len=128)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        assert lib.sbvr_hip_linear_f16_workspace(2, N, K, 4, 128) > 0
        sbvr._sbvr_linear_f16(x, *w, bvr_len=128)              # warms the stream
        ws = hip._workspaces[(DEV.index, side.cuda_stream)]
        assert ops._workspace(1, DEV.index).data_ptr() == ws.data_ptr()
        side.synchronize()
        before = torch.cuda.memory_allocated()
        got = [sbvr._sbvr_row_deq_mm_T(x, *t, none, bvr_len=128), sbvr._sbvr_mm_T(*l, *w, none, bvr_len=128)]
        assert torch.cuda.memory_allocated() - before <= sum((2 * y.numel() + 511) // 512 * 512 for y in got)
        side.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=side):
        got = [sbvr._sbvr_row_deq_mm_T(x, *t, none, bvr_len=128), sbvr._sbvr_mm_T(*l, *w, none, bvr_len=128)]
        assert ops._workspace(1, DEV.index).data_ptr() == ws.data_ptr()
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        with torch.cuda.stream(side):                          # eager work on the same workspace in between
            assert torch.equal(sbvr._sbvr_row_deq_mm_T(x, *t, none, bvr_len=128), want[0])
        side.synchronize()
    assert int(ws.count_nonzero()) == 0


def test_growing_requests_hold_little_more_than_the_largest():
    """Rising requests on one stream: the buffers that were outgrown (kept for graphs that point at them) and the one
    in use together stay below four times the largest request."""
    from sbvr import _sbvr_hip_ops as ops, hip
    with torch.cuda.stream(torch.cuda.Stream()):
        sizes = {}
        for mib in range(2, 26):
            for ws in (ops._workspace(mib << 20, DEV.index), hip._workspace(mib << 20, DEV)):
                assert ws.numel() >= mib << 20 and ws.data_ptr() % 16 == 0
                sizes[ws.data_ptr()] = ws.numel()
        assert int(ws.count_nonzero()) == 0
        assert sum(sizes.values()) <= 4 * (25 << 20)


def test_layers_keep_out_of_the_accumulators_of_recorded_functions():
    """A graph of the functions holds its stream's buffer and may be replayed on another stream while a layer is called
    on the first: the two never use one buffer."""
    import sbvr
    from sbvr import hip
    N, K = 1024, 2048
    w = _encoded(N, K, seed=1)
    x = torch.randn((2, K), generator=torch.Generator().manual_seed(4)).to(torch.float16).to(DEV)
    layer = sbvr.SBVRLinear(K, N, *w, 128)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        want = sbvr._sbvr_linear_f16(x, *w, bvr_len=128)
        ws = hip._workspaces[(DEV.index, side.cuda_stream)]
        side.synchronize()
        ws.view(torch.int64)[:2 * N] = 1 << 40           # (a launch under way elsewhere has left its sums here)
        y = layer(x)
        side.synchronize()
        assert torch.equal(y, want) and int((ws.view(torch.int64)[:2 * N] != 1 << 40).sum()) == 0
        ws.zero_()
        side.synchronize()


def _pool_of(t):
    return [seg["segment_pool_id"] for seg in torch.cuda.memory_snapshot()
            if seg["address"] <= t.data_ptr() < seg["address"] + seg["total_size"]]


@pytest.mark.parametrize("grow", [False, True])
def test_a_graph_recorded_on_a_stream_that_no_call_has_warmed(grow):
    """The accumulators of such a recording are the graph's own: calls on the stream before the first replay, between replays
    and after the graph's end have theirs, and every replay is right.  grow: the stream's buffer is there but too small."""
    import sbvr
    from sbvr import hip
    N, K = 4096, 4096
    x = torch.randn((24, K), generator=torch.Generator().manual_seed(4)).to(torch.float16).to(DEV)
    none = torch.zeros(0, dtype=torch.float16, device=DEV)
    t, small = _encoded(K, N, seed=3, L=256), _encoded(1024, K, seed=4)
    halves = sbvr.SBVRLinear(12800, 731, *_encoded(731, 12800, G=64, seed=5), 64)
    wide = sbvr.SBVRLinear(8192, 1304, *_encoded(1304, 8192, S=8, seed=6), 128)
    xh, xw = x.reshape(-1)[:12800].view(1, -1), x.reshape(-1)[:24 * 4096 // 8192 * 8192].view(-1, 8192).repeat(2, 1)
    calls = [lambda: sbvr._sbvr_linear_f16(x[:1], *small, bvr_len=128), lambda: sbvr._sbvr_row_deq_mm_T(x[:3], *t, none, bvr_len=128),
             lambda: sbvr._sbvr_row_deq_mm_T(x[:8], *t, none, bvr_len=128), lambda: halves(xh), lambda: wide(xw)]
    want, parts = [], []
    for call in calls:
        want.append(call())
        parts.append(max(hip.last_parts(), hip.row_deq_last()[1]))
    assert xw.shape[0] == 24 and min(parts) > 1
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    if grow:
        many = x.repeat(2, 1)                                  # 48 rows x 4096: more than the least buffer of 1 MiB holds
        calls.append(lambda: sbvr._sbvr_row_deq_mm_T(many, *t, none, bvr_len=128))
        want.append(calls[-1]())
        assert hip.row_deq_last()[1] > 1 and 8 * many.shape[0] * N > 1 << 20
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            assert all(torch.equal(call(), y) for call, y in zip(calls[:1], want))
            assert hip._workspace(1, DEV).numel() == 1 << 20
        side.synchronize()
    never_run, graph = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(never_run, stream=side):
        got = [call() for call in calls]
        of_the_first = hip._workspace(8 * 48 * N, DEV)
    with torch.cuda.graph(graph, stream=side):
        got = [call() for call in calls]
        assert hip._workspace(8 * 48 * N, DEV).data_ptr() != of_the_first.data_ptr()
    del never_run, of_the_first
    with torch.cuda.stream(side):
        for call, y in zip(calls, want):
            assert torch.equal(call(), y)
        ws = hip._workspace(8 * 8 * N, DEV)
        assert _pool_of(ws) == [(0, 0)] and int(ws.count_nonzero()) == 0
    for _ in range(3):
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))
        with torch.cuda.stream(side):
            assert all(torch.equal(call(), y) for call, y in zip(calls, want))
        torch.cuda.synchronize()
    del graph, got
    with torch.cuda.stream(side):
        assert all(torch.equal(call(), y) for call, y in zip(calls, want))
    torch.cuda.synchronize()
