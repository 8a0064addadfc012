"""The two prompt kernels at the sizes where each can go wrong: work-groups of one 128-row item (short prompts, few
items) and resident work-groups of 256-row items (the others).  Tolerances as in prefill_checks.py.

The tests of test_gpu_prefill.py are mostly of short prompts, which the first kernel does; what they look at (plans, scales,
peaked scores, many heads, launches in flight) is looked at here for the resident one, in prompts that are just long and many
enough for it."""
import numpy as np
import pytest
import torch

from oracle.moa_oracle import moa_token_mask
from prefill_checks import check_prefill, close_stated, masked_attention_gpu
from test_gpu_prefill import _qkv, _run

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    return torch.device("cuda:0")


# remainders of the 32-row wave, the 64-token block and the 128-row item; one pair, pairs shared out to the XCDs evenly
# and not; one round of work-groups with an odd and an even number of query tiles
@pytest.mark.parametrize("D,dtype", [(128, torch.float16), (128, torch.bfloat16), (64, torch.float16), (64, torch.bfloat16)])
@pytest.mark.parametrize("N,B,H,G", [(65, 1, 1, 1), (96, 2, 4, 1), (127, 1, 9, 1), (128, 1, 8, 2), (129, 3, 5, 1), (193, 2, 4, 4),
                                     (255, 1, 3, 3), (257, 1, 8, 1), (385, 1, 16, 8), (641, 2, 8, 1)])
def test_items_of_128_rows(dev, D, dtype, N, B, H, G):
    hkv = H // G
    rng = np.random.default_rng(N * 1000 + D)
    nb = (N + 63) // 64
    ns = [int(x) for x in rng.integers(0, 3, size=hkv)]
    nl = [int(x) for x in rng.integers(0, nb + 2, size=hkv)]
    if hkv > 2:
        ns[1], nl[1] = 0, 0          # sees nothing
        ns[2], nl[2] = 0, 1          # its own block only
    q, k, v = _qkv(B, H, N, D, dtype, dev, seed=N, hkv=hkv)
    out = _run(q, k, v, D ** -0.5, ns, nl, dev)
    kr, vr = (x.repeat_interleave(G, dim=1) for x in (k, v))
    check_prefill(out, q, kr, vr, D ** -0.5, [n for n in ns for _ in range(G)], [n for n in nl for _ in range(G)],
                  ("128 rows", N, B, H, G, D, dtype))


# the shortest prompts of the resident kernel with few heads: ragged query tiles and keys, heads without tiles, with fewer
# tiles than are copied ahead, with more; more than one item to a work-group
@pytest.mark.parametrize("N,H,D,dtype", [(3073, 24, 128, torch.float16), (3073, 24, 128, torch.bfloat16),
                                         (4097, 17, 64, torch.float16), (4161, 24, 64, torch.bfloat16)])
def test_resident_work_groups(dev, N, H, D, dtype):
    nb = (N + 63) // 64
    ns = ([1, 0, 2, 0, 1, 0] * H)[:H]
    nl = ([5, 0, 0, 1, nb, 2] * H)[:H]
    q, k, v = _qkv(1, H, N, D, dtype, dev, seed=N + H)
    assert _takes_resident_kernel(q)
    out = _run(q, k, v, D ** -0.5, ns, nl, dev)
    for h in range(0, 6):
        mask = torch.from_numpy(moa_token_mask(N, ns[h], nl[h])).to(dev)[None]
        sl = (slice(None), slice(h, h + 1))
        if nl[h] == 0 and ns[h] == 0:
            assert not out[sl].any()
            continue
        seen = mask.any(-1)[0]       # rows that see a key
        ref = masked_attention_gpu(q[sl], k[sl], v[sl], mask, D ** -0.5, dtype if dtype == torch.bfloat16 else None)
        close_stated(out[sl][:, :, seen], ref[:, :, seen], ("resident", N, h))
        assert not out[sl][:, :, ~seen].any()
    # a head's rows do not depend on which work-group did them, nor on what it did before
    again = _run(q, k, v, D ** -0.5, ns, nl, dev)
    assert torch.equal(out, again)


def _takes_resident_kernel(q):
    """The rule of the library's dispatch (short_items in moa_prefill.hip)."""
    B, H, N, D = q.shape
    cus = torch.cuda.get_device_properties(q.device).multi_processor_count
    return N > (4096 if D == 64 else 2048) and B * H * -(-N // 128) > 2 * cus


def _resident(q, k, v, sm, ns, nl, dev, which, tag):
    """A prompt by the resident kernel, and the (batch row, query head) pairs `which` of it against plain attention in fp32."""
    assert _takes_resident_kernel(q), tag
    out = _run(q, k, v, sm, ns, nl, dev)
    G = q.shape[1] // k.shape[1]
    for b, h in which:
        hk = h // G
        mask = torch.from_numpy(moa_token_mask(q.shape[2], ns[hk], nl[hk])).to(dev)[None]
        one = (slice(b, b + 1), slice(h, h + 1))
        ref = masked_attention_gpu(q[one], k[b:b + 1, hk:hk + 1], v[b:b + 1, hk:hk + 1], mask, sm,
                                   torch.bfloat16 if q.dtype == torch.bfloat16 else None)
        close_stated(out[one], ref, (tag, b, h))
    return out


@pytest.mark.parametrize("seed", range(8))
def test_resident_random_plans(dev, seed):
    """Odd lengths, batch rows, groups of query heads and spans; narrow bands, nothing at all, more than there are blocks."""
    rng = np.random.default_rng(500 + seed)
    D, dtype = [64, 128][seed % 2], [torch.float16, torch.bfloat16][(seed // 2) % 2]
    N = int(rng.integers(4097, 4700)) if D == 64 else int(rng.integers(2049, 2700))
    B, G = int(rng.integers(1, 4)), int(rng.choice([1, 3, 5]))
    hkv = -(-(17 if D == 64 else 31) // (B * G)) + int(rng.integers(0, 3))
    nb = -(-N // 64)
    ns = [int(x) for x in rng.integers(0, 5, size=hkv)]
    nl = [int(x) for x in (rng.integers(0, 4, size=hkv) if seed % 3 == 0 else rng.integers(0, nb + 3, size=hkv))]
    q, k, v = _qkv(B, hkv * G, N, D, dtype, dev, seed=seed, hkv=hkv)
    which = [(int(rng.integers(0, B)), int(h)) for h in rng.permutation(hkv * G)[:8]]
    _resident(q, k, v, D ** -0.5, ns, nl, dev, which, (seed, N, D, B, G, ns, nl))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sm", [-0.11, 0.0])
def test_resident_negative_and_zero_scale(dev, dtype, sm):
    """Two and more items to a work-group, so that most Q rows were asked for by the item before theirs; a batch of two with
    three query heads to a kv head."""
    B, hkv, G, N, D = 2, 11, 3, 2050, 128
    ns, nl = ([1, 0, 1] * hkv)[:hkv], ([2, 3, 1, 40] * hkv)[:hkv]
    q, k, v = _qkv(B, hkv * G, N, D, dtype, dev, seed=51, hkv=hkv)
    _resident(q, k, v, sm, ns, nl, dev, [(0, 0), (0, 4), (1, 8), (1, 11), (0, 32), (1, 17)], (sm, dtype))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
def test_resident_peaked_and_drifting_scores(dev, dtype):
    """Scores in the hundreds, larger ones the later the key: the reference exponent is raised many times in an item, and
    starts anew in the next."""
    B, H, N, D = 1, 32, 2100, 128
    q, k, v = _qkv(B, H, N, D, dtype, dev, seed=31)
    q = (q * 6).contiguous()
    k = (k * torch.linspace(0.2, 3.0, N, device=dev)[None, None, :, None].to(dtype)).contiguous()
    ns, nl = ([1, 0, 2, 1] * H)[:H], ([33, 3, 5, 1] * H)[:H]
    _resident(q, k, v, D ** -0.5, ns, nl, dev, [(0, h) for h in (0, 1, 2, 3, 17, 30)], ("peaked", dtype))


def test_resident_more_heads_than_the_sorted_schedule_covers(dev):
    """Past 512 kv heads they are taken in the given order; spans in tokens and in blocks."""
    from moa_amd.kernels.mixture_of_attention import moa_prefill
    B, H, N, D = 1, 520, 2049, 128
    rng = np.random.default_rng(21)
    ns = [int(x) for x in rng.integers(0, 2, size=H)]
    nl = [int(x) for x in rng.integers(0, 5, size=H)]
    g = torch.Generator(device=dev).manual_seed(22)
    q, k, v = (torch.randn(B, N, H, D, generator=g, device=dev, dtype=torch.float16).transpose(1, 2) for _ in range(3))
    out = _resident(q, k, v, D ** -0.5, ns, nl, dev, [(0, h) for h in (0, 1, 100, 257, 511, 512, 519)], "520 heads")
    blocks = (torch.tensor(x, device=dev) for x in (ns, nl))
    want = moa_prefill(q.transpose(1, 2), k, v, num_global_blocks=next(blocks), num_band_blocks=next(blocks), sm_scale=D ** -0.5)
    assert torch.equal(out, want.transpose(1, 2))


def test_many_resident_launches_in_flight_on_two_streams(dev):
    """600 launches of two shapes, alternating between two streams with nothing waiting in between: the 256 work queues go
    round more than twice, each cleared by the last work-group of the launch that had it before.  Every result is that of
    the same call made alone."""
    cases = []
    for i, (H, N, D, dtype) in enumerate([(16, 4097, 64, torch.float16), (31, 2049, 128, torch.bfloat16)]):
        q, k, v = _qkv(1, H, N, D, dtype, dev, seed=70 + i)
        assert _takes_resident_kernel(q)
        ns, nl = ([1, 0, 2, 1] * H)[:H], ([2, 5, 1, 3, 0] * H)[:H]
        cases.append((q, k, v, D ** -0.5, ns, nl))
    alone = [_run(*c, dev).clone() for c in cases]
    spans = [[torch.tensor([64 * x for x in c[j]], device=dev) for j in (4, 5)] for c in cases]
    torch.cuda.synchronize()
    from moa_amd import mixture_of_sparse_attention
    streams, outs = [torch.cuda.Stream(), torch.cuda.Stream()], []
    for i in range(600):
        (q, k, v, sm, _, _), (sink, local) = cases[i % 2], spans[i % 2]
        with torch.cuda.stream(streams[(i // 2) % 2]):
            outs.append(mixture_of_sparse_attention(q, k, v, sm, sink_size=sink, local_size=local))
    torch.cuda.synchronize()
    for i, out in enumerate(outs):
        assert torch.equal(out.transpose(1, 2), alone[i % 2]), i


def test_resident_launches_in_flight_on_two_streams(dev):
    """Launches of the resident kernel overlap on two streams; each has a work queue of its own."""
    cases = []
    for i, (N, H, D, dtype) in enumerate([(4097, 17, 64, torch.float16), (3073, 24, 128, torch.bfloat16)]):
        ns, nl = ([1, 0, 2] * H)[:H], ([3, 2, 0, 9] * H)[:H]
        q, k, v = _qkv(1, H, N, D, dtype, dev, seed=90 + i)
        cases.append((q, k, v, D ** -0.5, ns, nl))
    alone = [_run(*c, dev).clone() for c in cases]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    outs = []
    for i in range(40):
        with torch.cuda.stream(streams[(i // 2) % 2]):
            outs.append((i % 2, _run(*cases[i % 2], dev)))
    torch.cuda.synchronize()
    assert all(torch.equal(out, alone[c]) for c, out in outs)


def test_resident_launch_replays_like_eager(dev):
    """Recorded into a HIP graph: every replay, on new inputs and with eager launches in between, finds its work queue as the
    last one left it."""
    H, N, D = 31, 2049, 128
    ns, nl = ([1, 0, 2, 1] * H)[:H], ([2, 5, 1, 3, 0] * H)[:H]
    q, k, v = _qkv(1, H, N, D, torch.bfloat16, dev, seed=80)
    assert _takes_resident_kernel(q)
    sink, local = (torch.tensor([64 * x for x in y], device=dev) for y in (ns, nl))
    from moa_amd import mixture_of_sparse_attention

    def call():
        return mixture_of_sparse_attention(q, k, v, D ** -0.5, sink_size=sink, local_size=local)

    call()   # looks up what a capture cannot
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        recorded = call()
    for i in range(4):
        q.normal_(generator=torch.Generator(device=dev).manual_seed(i))
        recorded.fill_(float("nan"))
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(recorded, call()), i
