"""The compiled host side of the attention and the append against the Python code that it stands in front of: over every form of
operands, the same bits; what needs a conversion, and what is wrong, is left to that code."""
import pickle

import pytest
import torch


class _Declines:
    """A host side that takes no call."""
    attend = rope_append = append = staticmethod(lambda *args: None)


class _Counts:
    """The real one, which notes the calls that it took."""

    def __init__(self, real):
        self.real, self.taken = real, []

    def __getattr__(self, name):
        def call(*args):
            r = getattr(self.real, name)(*args)
            if r is not None:
                self.taken.append(name)
            return r
        return call


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from moa_amd import _lib
    _lib.load()
    return torch.device("cuda:0")


def _operands(dev, form, dtype, B, Hq, H, D, seed):
    g = torch.Generator(device=dev).manual_seed(seed)

    def make(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=torch.float32).to(dtype)

    if form == "fused":       # views of one projection buffer
        qkv = make(B, 1, Hq + 2 * H, D).transpose(1, 2)
        q, k, v = qkv[:, :Hq], qkv[:, Hq:Hq + H], qkv[:, Hq + H:]
    elif form == "strided":   # heads apart, head_dim not in one piece
        q, k, v = (make(B, h, D, 2).permute(0, 1, 3, 2)[:, :, :1] for h in (Hq, H, H))
    else:
        q, k, v = (make(B, 1, h, D).transpose(1, 2) for h in (Hq, H, H))
    rows = B if form == "per_row" else 1
    cos, sin = make(rows, 1, D), make(rows, 1, D)
    if form == "odd_sin":     # laid out unlike cos
        sin = make(rows, 1, 2 * D)[..., ::2]
    return q, k, v, cos, sin


def _pass(dev, host, monkeypatch, form, fused, dtype, B, Hq, H, D, restore):
    from moa_amd import StaticCircularCache, _lib, mixture_of_sparse_attention
    monkeypatch.setattr(_lib, "host", lambda: host)
    sizes = [70 + 37 * h for h in range(H)]
    cache = StaticCircularCache([sizes], static_size=[[5] * H], batch_size=B, head_dim=D, device=dev, dtype=dtype)
    outs = []
    for step in range(9):   # through the static part and into the ring
        q, k, v, cos, sin = _operands(dev, form, dtype, B, Hq, H, D, step)
        if restore and step == 5:   # a cache that comes out of a file
            cache = pickle.loads(pickle.dumps(cache))
        if fused:
            q, keys, values = cache.rope_update(q, k, v, cos, sin, 0)
        else:
            keys, values = cache.update(k, v, 0)
        if dtype != torch.float32:   # the attention runs in 16 bits
            outs.append(mixture_of_sparse_attention(q, keys, values, 0.1, head_start_index=cache.cache_head_start_index[0],
                                                    head_valid_length=cache.cache_valid_length[0]).clone())
        outs.append(q.clone())
    return outs + [cache.key_cache[0], cache.value_cache[0], cache.mask_cache[0], cache.cache_update_index[0],
                   cache.cache_valid_length[0]]


@pytest.mark.gpu
@pytest.mark.parametrize("fused", [True, False])
@pytest.mark.parametrize("form", ["plain", "fused", "per_row", "strided", "odd_sin", "restored"])
@pytest.mark.parametrize("dtype,B,Hq,H,D", [(torch.float16, 1, 4, 4, 128), (torch.bfloat16, 3, 7, 1, 64),
                                            (torch.float32, 2, 4, 2, 64)])
def test_same_bits_as_the_general_path(dev, monkeypatch, fused, form, dtype, B, Hq, H, D):
    from moa_amd import _lib
    counts = _Counts(_lib.host())
    got, want = (_pass(dev, host, monkeypatch, form, fused, dtype, B, Hq, H, D, form == "restored")
                 for host in (counts, _Declines()))
    assert len(got) == len(want)
    for i, (a, b) in enumerate(zip(got, want)):
        assert torch.equal(a, b), i
    # what has to be converted first is not taken: rows in pieces by either append, a sin unlike cos by the rotary one,
    # queries that are not in one piece by the attention
    appends = 0 if form == "strided" or (form == "odd_sin" and fused) else 9
    in_one_piece = fused or not (form == "strided" or (form == "fused" and B > 1))
    assert counts.taken.count("rope_append" if fused else "append") == appends
    assert counts.taken.count("attend") == (9 if dtype != torch.float32 and in_one_piece else 0)


@pytest.mark.gpu
def test_wrong_calls_are_the_general_paths(dev):
    from moa_amd import _lib, mixture_of_sparse_attention
    q = torch.randn(2, 4, 1, 128, device=dev, dtype=torch.float16)
    k = torch.randn(2, 300, 128, device=dev, dtype=torch.float16)
    start = torch.tensor([[0, 100]] * 2, device=dev)
    valid = torch.tensor([[100, 200]] * 2, device=dev)
    host = _lib.host()
    assert host.attend(q, k, k, 0.1, start, valid, None, None) is not None
    for bad in ((q.float(), k, k, start, valid), (q, k.bfloat16(), k, start, valid), (q, k, k[:, :-1], start, valid),
                (q[:, :, :, :64], k, k, start, valid), (q, k, k, start[:1], valid), (q, k.cpu(), k, start, valid),
                (q, k, k, start.int(), valid), (q, k, k, start, None), (q, k[:, ::2], k[:, ::2], start, valid),
                (q.repeat(1, 1, 2, 1), k, k, start, valid), (q, k, k, start, valid[:, :1])):
        assert host.attend(*bad[:3], 0.1, *bad[3:], None, None) is None
    assert host.attend(q, k, k, "0.1", start, valid, None, None) is None
    # refused by the library: the exception is the general path's
    with pytest.raises(AssertionError, match="not a multiple"):
        mixture_of_sparse_attention(q[:, :3].contiguous(), k, k, 0.1, head_start_index=start, head_valid_length=valid)
    with pytest.raises(NotImplementedError):
        mixture_of_sparse_attention(torch.randn(2, 2, 1, 32, device=dev, dtype=torch.float16), k[..., :32].contiguous(),
                                    k[..., :32].contiguous(), 0.1, head_start_index=start, head_valid_length=valid)


@pytest.mark.gpu
@pytest.mark.parametrize("form", ["plain", "contiguous", "fused", "in_pieces", "expanded"])
@pytest.mark.parametrize("dtype,B,Hq,H,N,D", [(torch.float16, 1, 2, 2, 65, 64), (torch.bfloat16, 3, 6, 2, 130, 128)])
def test_prompts_same_bits_as_the_general_path(dev, monkeypatch, form, dtype, B, Hq, H, N, D):
    from moa_amd import _lib, mixture_of_sparse_attention
    g = torch.Generator(device=dev).manual_seed(N)

    def make(*shape):
        return torch.randn(*shape, generator=g, device=dev, dtype=dtype)

    if form == "contiguous":
        q, k, v = make(B, Hq, N, D), make(B, H, N, D), make(B, H, N, D)
    elif form == "fused":
        qkv = make(B, N, Hq + 2 * H, D).transpose(1, 2)
        q, k, v = qkv[:, :Hq], qkv[:, Hq:Hq + H], qkv[:, Hq + H:]
    elif form == "in_pieces":
        q, k, v = (make(B, h, D, N).transpose(2, 3) for h in (Hq, H, H))
    else:
        q, k, v = (make(B, N, h, D).transpose(1, 2) for h in (Hq, H, H))
        if form == "expanded":
            k, v = (t[:, :1].expand(B, H, N, D) for t in (k, v))
    sink = torch.full((H,), 64, device=dev)
    local = torch.full((H,), 64, device=dev)
    counts = _Counts(_lib.host())
    got, want = [], []
    for host, outs in ((counts, got), (_Declines(), want)):
        monkeypatch.setattr(_lib, "host", lambda: host)
        outs.append(mixture_of_sparse_attention(q, k, v, 0.1, sink_size=sink, local_size=local))
        outs.append(mixture_of_sparse_attention(q, k, v, 1, sink_size=sink.expand(H), local_size=local.int()))
    assert got[0].stride() == want[0].stride()
    assert all(torch.equal(a, b) for a, b in zip(got, want))
    assert len(counts.taken) == (0 if form == "in_pieces" else 1)   # 32-bit spans are converted first
    with pytest.warns(UserWarning, match="dense prefill"):   # one block
        monkeypatch.setattr(_lib, "host", lambda: counts)
        mixture_of_sparse_attention(q[:, :, :64], k[:, :, :64], v[:, :, :64], 0.1)
