"""The arrival counters of decode launches that merge inside: they outlive a call, so only calls that cannot overlap may
share them.  A step recorded into a HIP graph, whose replays run on any stream, takes none of the Python path's."""
import pytest
import torch


def test_a_recorded_call_takes_no_shared_counters(monkeypatch):
    from moa_amd.kernels import mixture_of_attention as M
    dev, stream = torch.device("cuda:0"), -12345   # no stream of this value exists
    kept = M._DecodeScratch()   # as an eager call on that stream leaves it
    kept.ws, kept.ws_ptr, kept.ws_bytes = torch.zeros(512, dtype=torch.uint8), 4096, 512
    kept.counters, kept.counters_ptr = torch.zeros(4, dtype=torch.int32), 8192
    monkeypatch.setitem(M._scratch, (0, stream), kept)
    monkeypatch.setitem(M._scratch, (0, 0), kept)   # the stream that cannot be recorded
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert M._decode_scratch(dev, stream, 512) == (4096, 512, 8192)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert M._decode_scratch(dev, stream, 512) == (4096, 512, None)
    assert M._decode_scratch(dev, 0, 512) == (4096, 512, 8192)


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from moa_amd import _lib
    _lib.load()
    return torch.device("cuda:0")


def _rings(dev, G, D, B, sizes):
    g = torch.Generator(device=dev).manual_seed(G * D + B)
    H, sumC = len(sizes), sum(sizes)
    q = torch.randn(B, H * G, 1, D, generator=g, device=dev, dtype=torch.float16)
    kc, vc = (torch.randn(B, sumC, D, generator=g, device=dev, dtype=torch.float16) for _ in range(2))
    start = torch.tensor([sum(sizes[:h]) for h in range(H)], device=dev).expand(B, H).contiguous()
    valid = torch.tensor(sizes, device=dev).expand(B, H).contiguous()
    return q, kc, vc, start, valid


@pytest.mark.gpu
@pytest.mark.parametrize("G", [1, 4])
def test_replays_beside_eager_calls_of_the_capture_stream(dev, G):
    """A step recorded on the stream that eager calls ran on before: replays, with eager calls in between, are right
    and neither look at that stream's counters nor touch them."""
    from moa_amd import mixture_of_sparse_attention
    from moa_amd.kernels import mixture_of_attention as M
    q, kc, vc, start, valid = _rings(dev, G, 128, 1, [700, 1100, 300, 900])

    def step():
        return mixture_of_sparse_attention(q, kc, vc, 0.1, head_start_index=start, head_valid_length=valid)

    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        step()
        counters = M._scratch[(0, stream.cuda_stream)].counters
        with torch.cuda.graph(graph, stream=stream):
            recorded = step()
        for i in range(4):
            q.normal_(generator=torch.Generator(device=dev).manual_seed(i))
            want = step()
            stream.synchronize()
            assert not counters.any(), i
            counters.fill_(1)   # as a launch under way holds them
            graph.replay()
            stream.synchronize()
            assert (counters == 1).all(), i
            counters.zero_()
            assert torch.equal(recorded, want), i


@pytest.mark.gpu
@pytest.mark.parametrize("G", [1, 4])
def test_a_graph_with_counters_of_its_own(dev, G):
    """Through the C entry point a graph may bring counters: every replay finds them zero and leaves them so."""
    from moa_amd import _lib
    lib = _lib.load()
    B, D = 1, 128
    q, kc, vc, start, valid = _rings(dev, G, D, B, [700, 1100, 300, 900])
    Hq, Hkv, sumC = q.shape[1], valid.shape[1], kc.shape[1]
    need = lib.moa_decode_workspace_bytes(B, Hq, Hkv, D, sumC)
    ws = torch.empty(need, dtype=torch.uint8, device=dev)
    counters = torch.zeros(B * Hkv, dtype=torch.int32, device=dev)

    def call(o, n):
        rc = lib.moa_decode_fwd_counted(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), o.data_ptr(), ws.data_ptr(), need,
                                        counters.data_ptr(), n, start.data_ptr(), valid.data_ptr(), B, Hq, Hkv, D, sumC,
                                        D ** -0.5, _lib.MOA_DTYPE_F16, _lib.current_stream_ptr(dev))
        assert rc == 0, _lib.last_error()

    recorded, want = torch.empty_like(q), torch.empty_like(q)
    call(recorded, counters.numel())
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        call(recorded, counters.numel())
    for i in range(4):
        q.normal_(generator=torch.Generator(device=dev).manual_seed(i))
        valid.sub_(97)   # other chunk counts in every replay
        call(want, 0)
        recorded.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, want), i
        assert not counters.any(), i


@pytest.mark.gpu
@pytest.mark.parametrize("G,D,B,sizes", [
    (4, 128, 1, [2048] * 8),                    # 64 chunks of a batch row: the most that merges inside
    (4, 128, 1, [2048] * 7 + [2056]),           # 65
    (2, 64, 1, [16000, 100, 100]),              # nearly all of them in one ring
    (3, 64, 1, [8192]),                         # 32 of an average ring
    (3, 64, 1, [8200]),                         # 33
    (8, 128, 1, [768] * 8),                     # two rounds of query heads: 24
    (8, 128, 1, [768] * 7 + [776]),             # 25
    (5, 64, 2, [5500, 100, 100, 100, 100]),
    (7, 64, 1, [4096]),                         # 16 of an average ring
    (7, 64, 1, [4100]),                         # 17
    (6, 128, 11, [1536] * 4),
    (8, 64, 13, [4400, 300, 300, 300]),
    (8, 64, 40, [700, 64]),                     # chunks of 2048 rows
])
def test_lines_of_the_merge_inside(dev, G, D, B, sizes):
    """On both sides of every line of the rule for merging inside, with rings of equal length and one ring that is
    nearly all of the batch row: the same bits as with the merge launch, and zeroed counters, call after call."""
    from moa_amd import _lib
    lib = _lib.load()
    q, kc, vc, start, valid = _rings(dev, G, D, B, sizes)
    Hq, Hkv, sumC = q.shape[1], len(sizes), kc.shape[1]
    need = lib.moa_decode_workspace_bytes(B, Hq, Hkv, D, sumC)
    counters = torch.zeros(B * Hkv, dtype=torch.int32, device=dev)
    for step in range(3):
        outs = []
        for n in (0, counters.numel()):
            ws = torch.full((need,), 0xff, dtype=torch.uint8, device=dev)   # NaN partials: none is read unwritten
            o = torch.full_like(q, float("nan"))
            rc = lib.moa_decode_fwd_counted(q.data_ptr(), kc.data_ptr(), vc.data_ptr(), o.data_ptr(), ws.data_ptr(), need,
                                            counters.data_ptr(), n, start.data_ptr(), valid.data_ptr(), B, Hq, Hkv, D,
                                            sumC, D ** -0.5, _lib.MOA_DTYPE_F16, _lib.current_stream_ptr(dev))
            assert rc == 0, _lib.last_error()
            outs.append(o)
        assert torch.isfinite(outs[0]).all() and torch.equal(outs[1], outs[0]), step
        assert not counters.any(), step
        valid = (valid * 2) // 3   # rings that are not full
