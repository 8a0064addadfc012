"""The workspace that decode calls keep from one to the next: who may share it."""
import threading

import pytest
import torch


def _in_threads(n, work):
    """Runs work(i) in n threads; what they return, or the first exception."""
    results, errors = [None] * n, []

    def body(i):
        try:
            results[i] = work(i)
        except BaseException as e:   # noqa: B902 (the caller raises it)
            errors.append(e)

    threads = [threading.Thread(target=body, args=(i,)) for i in range(n)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    if errors:
        raise errors[0]
    return results


def test_threads_do_not_share_a_workspace():
    """Two threads on one stream, alive at the same time: neither is given the other's memory, and one's longer call leaves
    the other's where it is."""
    from moa_amd.kernels import mixture_of_attention as M
    place = torch.device("cpu")   # the bookkeeping does not care
    both = threading.Barrier(2, timeout=60)

    def work(i):
        first = M._decode_scratch(place, 0, 512)
        both.wait()
        grown = M._decode_scratch(place, 0, 1 << 20) if i == 0 else None
        both.wait()
        again = M._decode_scratch(place, 0, 512)
        both.wait()
        return first, again, grown

    (first0, again0, grown0), (first1, again1, _) = _in_threads(2, work)
    assert first0[0] != first1[0] and first0[2] != first1[2]
    assert again0 == grown0 and again0[1] >= 1 << 20
    assert again1 == first1


def test_a_recorded_call_leaves_no_workspace_behind(monkeypatch):
    """What is allocated while a stream is recorded belongs to the graph: it is not kept for the stream's eager calls, and
    theirs is not replaced."""
    from moa_amd.kernels import mixture_of_attention as M
    place, stream = torch.device("cpu"), -54321   # no stream of this value exists
    monkeypatch.setitem(M._scratch, (0, stream), M._DecodeScratch())
    recording = True
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: recording)
    assert M._decode_scratch(place, stream, 512)[2] is None and M._scratch[(0, stream)].ws is None
    recording = False
    eager = M._decode_scratch(place, stream, 512)
    recording = True
    assert M._decode_scratch(place, stream, 1 << 20)[2] is None
    recording = False
    assert M._decode_scratch(place, stream, 512) == eager


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from moa_amd import _lib
    _lib.load()
    return torch.device("cuda:0")


def _case(dev, G, B, sizes, D, seed):
    g = torch.Generator(device=dev).manual_seed(seed)
    H, sumC = len(sizes), sum(sizes)
    q = torch.randn(B, H * G, 1, D, generator=g, device=dev, dtype=torch.float16)
    kc, vc = (torch.randn(B, sumC, D, generator=g, device=dev, dtype=torch.float16) for _ in range(2))
    start = torch.tensor([sum(sizes[:h]) for h in range(H)], device=dev).expand(B, H).contiguous()
    valid = torch.tensor(sizes, device=dev).expand(B, H).contiguous()
    return q, kc, vc, start, valid


def _attend(q, kc, vc, start, valid):
    from moa_amd import mixture_of_sparse_attention
    return mixture_of_sparse_attention(q, kc, vc, 0.1, head_start_index=start, head_valid_length=valid)


@pytest.mark.gpu
@pytest.mark.parametrize("G,B,sizes", [(1, 40, [5000, 3000, 700]),      # two launches
                                       (8, 1, [2000, 9000, 300]),       # two launches, grouped
                                       (4, 1, [700, 1100, 300, 900])])  # one that counts
def test_threads_on_one_stream(dev, G, B, sizes):
    """Threads that decode on the same stream, with sizes that grow: every result is that of the call made alone."""
    cases = [[_case(dev, G, b, sizes, 64, 10 * i + b) for b in sorted({1, (B + 1) // 2, B})] for i in range(3)]
    want = [[_attend(*c) for c in cs] for cs in cases]
    torch.cuda.synchronize()

    def work(i):
        return [[_attend(*c) for c in cases[i]] for _ in range(20)]

    got = _in_threads(3, work)
    torch.cuda.synchronize()
    for i in range(3):
        for outs in got[i]:
            assert all(torch.equal(a, b) for a, b in zip(outs, want[i])), i


@pytest.mark.gpu
@pytest.mark.parametrize("compiled", [True, False])
@pytest.mark.parametrize("G,B,sizes", [(1, 40, [5000, 3000, 700]), (8, 1, [2000, 9000, 300]), (4, 1, [700, 1100, 300, 900])])
def test_a_graph_keeps_its_workspace(dev, monkeypatch, compiled, G, B, sizes):
    """Two graphs of one stream, the second with the longer call, and longer eager calls on it afterwards: replays of the
    first, on another stream and beside them, are right and write to nothing of theirs."""
    from moa_amd import _lib
    if not compiled:
        class Declines:
            attend = staticmethod(lambda *args: None)
        monkeypatch.setattr(_lib, "host", lambda: Declines)
    small, large, larger = (_case(dev, G, b, sizes, 64, b) for b in (B, 2 * B, 4 * B))
    want = [_attend(*c) for c in (small, large, larger)]
    stream, other = torch.cuda.Stream(), torch.cuda.Stream()
    graphs, recorded = [], []
    with torch.cuda.stream(stream):
        _attend(*small)
        stream.synchronize()
        for c in (small, large):
            graphs.append(torch.cuda.CUDAGraph())
            with torch.cuda.graph(graphs[-1], stream=stream):
                recorded.append(_attend(*c))
        eager = _attend(*larger)   # replaces the stream's workspace
        # what is given back is given out again
        others = [torch.full((n << 10,), 7, dtype=torch.uint8, device=dev) for n in (64, 256, 512, 1024, 1024, 2048, 4096)]
    torch.cuda.synchronize()
    assert torch.equal(eager, want[2])
    for i in range(4):
        for r in recorded:
            r.fill_(float("nan"))
        torch.cuda.synchronize()
        with torch.cuda.stream(other):
            graphs[0].replay()
        with torch.cuda.stream(stream):
            eager = _attend(*larger)
            graphs[1].replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded[0], want[0]) and torch.equal(recorded[1], want[1]) and torch.equal(eager, want[2]), i
        assert all((t == 7).all() for t in others), i
