"""The start of a generation in one launch (moa_rope_prefill_insert) at the sizes where its parts can go wrong, against
the separate rotary embedding and insert, bit for bit: rings full of NaN before the call, several pieces of heads to a
token, padded prompts past one part of the mask scan, launches that go by the caches, head strides of 0, and launches
recorded into a graph."""
import pytest
import torch

from oracle.moa_oracle import rope_cos_sin

pytestmark = pytest.mark.gpu

TABLES = ("mask_cache", "cache_update_index", "cache_valid_length")


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from moa_amd import _lib
    _lib.load()
    return torch.device("cuda:0")


def _bits(t):
    return t.view({2: torch.int16, 4: torch.int32}[t.element_size()])


def _same(a, b):
    return a.shape == b.shape and torch.equal(_bits(a.contiguous()), _bits(b.contiguous()))


def _inputs(dev, dtype, B, Hq, H, S, D, at=0, seed=0):
    g = torch.Generator(device=dev).manual_seed(seed + S + D)
    q, k, v = (torch.randn(B, S, n, D, generator=g, device=dev, dtype=dtype).transpose(1, 2) for n in (Hq, H, H))
    cos, sin = (t.to(dev) for t in rope_cos_sin(torch.arange(S)[None, :] + at, D, dtype=dtype))
    return q, k, v, cos, sin


def _padding(dev, B, S):
    """Left padding whose end lies in another part of the scan than its begin, holes, a row of padding only."""
    mask = (torch.rand(B, S, generator=torch.Generator().manual_seed(S)) < 0.9).to(torch.int64)
    mask[0, :S // 3] = 0
    mask[-1] = 0
    return mask.to(dev)


def _cache(dev, dtype, B, D, sizes, static):
    from moa_amd import StaticCircularCache
    return StaticCircularCache([sizes], static_size=[static], batch_size=B, head_dim=D, device=dev, dtype=dtype)


def _ring_plan(H):
    """(sizes, static sizes): several slices of ring rows, a head without a ring, one without a static part."""
    plan = [(700, 64), (64, 64), (257, 0), (333, 64)]
    return [plan[h % 4][0] for h in range(H)], [plan[h % 4][1] for h in range(H)]


def _one_launch(cache, q, k, v, cos, sin, mask, zero_rest):
    """moa_rope_prefill_insert through the C ABI on the cache's own tensors."""
    from moa_amd import _lib
    lib = _lib.load()
    B, Hq, S, D = q.shape
    H = k.shape[1]
    q_out, k_out = torch.empty_like(q), torch.empty_like(k)
    ws = torch.empty(lib.moa_cache_prefill_workspace_bytes(B, S), dtype=torch.uint8, device=q.device)
    rc = lib.moa_rope_prefill_insert(
        q.data_ptr(), k.data_ptr(), v.data_ptr(), q_out.data_ptr(), k_out.data_ptr(),
        *(_lib.i64_array(t.stride()) for t in (q, k, v, q_out, k_out)), cos.data_ptr(), sin.data_ptr(),
        _lib.i64_array([0, cos.stride(1), 1]), cache.key_cache[0].data_ptr(), cache.value_cache[0].data_ptr(),
        cache.mask_cache[0].data_ptr(), cache.cache_update_index[0].data_ptr(), cache.cache_valid_length[0].data_ptr(),
        cache.circular_cache_head_index[0].data_ptr(), cache.circular_cache_size[0].data_ptr(),
        cache.static_cache_size[0].data_ptr(), _lib.ptr(mask), 0 if mask is None else mask.stride(0), ws.data_ptr(),
        ws.numel(), cache._kv_len[0], B, Hq, H, S, D, cache.layer_cache_size[0], cache._max_cache_size[0], zero_rest,
        _lib.dtype_code(q.dtype), _lib.current_stream_ptr(q.device))
    assert rc == 0, _lib.last_error()
    return q_out, k_out


def _two_steps(cache, q, k, v, cos, sin, mask):
    from moa_amd.kernels.rotary import apply_rotary_pos_emb
    q_out, k_out = apply_rotary_pos_emb(q, k, cos, sin)
    cache.update(k_out, v, 0, mask)
    return q_out, k_out


def _check(got, want, one, two, tag):
    for a, b in zip(got, want):
        assert _same(a, b), tag
    for name in ("key_cache", "value_cache"):
        assert _same(getattr(one, name)[0], getattr(two, name)[0]), (name, tag)
    for name in TABLES:
        assert torch.equal(getattr(one, name)[0], getattr(two, name)[0]), (name, tag)


@pytest.mark.parametrize("Hq,H", [(8, 4), (33, 33), (64, 64), (96, 8)])   # one to several pieces of q and of kv heads
@pytest.mark.parametrize("D,dtype", [(128, torch.bfloat16), (64, torch.float16), (128, torch.float32)])
@pytest.mark.parametrize("S", [3, 300, 1100])
@pytest.mark.parametrize("zero_rest", [0, 1])
def test_rings_full_of_nan(dev, Hq, H, D, dtype, S, zero_rest):
    """zero_rest = 1: every row of every segment is written, the free ones with zeros.  0: rows that no token goes to
    keep their bits."""
    B = 2
    sizes, static = _ring_plan(H)
    for mask in (None, _padding(dev, B, S)):
        one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
        for c in (one, two):
            c._to_device(0, dev)
        for ring in (one.key_cache[0], one.value_cache[0]) + (() if zero_rest else (two.key_cache[0], two.value_cache[0])):
            ring.fill_(float("nan"))
        args = _inputs(dev, dtype, B, Hq, H, S, D)
        _check(_one_launch(one, *args, mask, zero_rest), _two_steps(two, *args, mask), one, two, mask is None)


@pytest.mark.parametrize("S", [4095, 4096, 4097, 8193, 16385])
def test_padded_prompts_past_a_part_of_the_mask_scan(dev, S):
    B, Hq, H, D, dtype = 3, 8, 8, 64, torch.bfloat16
    sizes, static = [5000] + [700, 64, 257, 333, 4100, 96, 128], [64] * 8
    one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
    args, mask = _inputs(dev, dtype, B, Hq, H, S, D), _padding(dev, B, S)
    assert one._prompt_fits_one_launch(*args, 0, mask)
    _check(one.rope_update(*args, 0, mask)[:2], _two_steps(two, *args, mask), one, two, S)


@pytest.mark.parametrize("H", [1, 5, 64])
@pytest.mark.parametrize("S", [2, 900])
def test_heads_of_very_different_rings(dev, H, S):
    """One ring that is most of the batch row, first, last and in the middle, among rings of a few rows, of less than
    one and of exactly one slice, and heads without a ring: every slice finds its head."""
    B, Hq, D, dtype = 3, 64, 64, torch.float16
    for at in {0, H // 2, H - 1}:
        sizes = [[3, 64, 65, 128, 129, 256, 1][h % 7] for h in range(H)]
        static = [min(64, n) if h % 2 else n // 2 for h, n in enumerate(sizes)]
        sizes[at], static[at] = 5001, 64
        for mask in (None, _padding(dev, B, S)):
            one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
            for piece in range(2):   # new rings, then rings in use
                args = _inputs(dev, dtype, B, Hq, H, S, D, at=piece * S, seed=piece)
                if H > 1:
                    assert one._prompt_fits_one_launch(*args, 0, mask)
                _check(one.rope_update(*args, 0, mask)[:2], _two_steps(two, *args, mask), one, two, (at, piece))


@pytest.mark.parametrize("S,rows", [(64, 16383), (64, 16384), (4095, 16384), (4096, 16384)])
def test_first_prompts_shorter_than_the_new_rings(dev, S, rows):
    """On both sides of 64 MiB of rings and of a quarter of their rows: filled and walked by tokens, or walked by rows."""
    B, H, D, dtype = 1, 8, 128, torch.bfloat16
    sizes, static = [rows] * H, [64] * H
    junk = [torch.full((B, rows * H, D), float("nan"), dtype=dtype, device=dev) for _ in range(4)]
    del junk   # memory that the rings may be given
    one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
    args = _inputs(dev, dtype, B, H, H, S, D)
    _check(one.rope_update(*args, 0, None)[:2], _two_steps(two, *args, None), one, two, (S, rows))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("S", [8191, 8193])   # around 256 MiB of q and k, from which on they pass the caches by
def test_large_prompts_of_both_load_kinds(dev, dtype, S):
    B, H, D = 2, 32, 128
    sizes, static = _ring_plan(H)
    sizes[0] = 6000
    one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
    args, mask = _inputs(dev, dtype, B, H, H, S, D), _padding(dev, B, S)
    assert (B * S * 2 * H * D * 2 >= 256 << 20) == (S > 8192)
    for piece in range(2):   # rings that the call allocates, then rings in use
        assert one._prompt_fits_one_launch(*args, 0, mask)
        _check(one.rope_update(*args, 0, mask)[:2], _two_steps(two, *args, mask), one, two, piece)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16, torch.float32])
@pytest.mark.parametrize("wild_tables", [False, True])
def test_every_kind_of_number(dev, dtype, wild_tables):
    """Random bit patterns: subnormals, infinities, NaN, products that overflow or vanish.  The same bits as the two
    steps, but for which NaN comes out where two meet."""
    B, Hq, H, S, D = 2, 8, 8, 300, 128
    sizes, static = _ring_plan(H)
    g = torch.Generator(device=dev).manual_seed(1)

    def wild(*shape):
        lo = -2 ** (31 if dtype == torch.float32 else 15)
        ints = torch.randint(lo, -lo, shape, generator=g, device=dev)
        return ints.to(torch.int32 if dtype == torch.float32 else torch.int16).view(dtype)

    q, k, v = (wild(B, S, n, D).transpose(1, 2) for n in (Hq, H, H))
    cos, sin = (wild(1, S, D), wild(1, S, D)) if wild_tables else _inputs(dev, dtype, B, Hq, H, S, D)[3:]
    one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
    got, want = one.rope_update(q, k, v, cos, sin, 0)[:2], _two_steps(two, q, k, v, cos, sin, None)
    for a, b in list(zip(got, want)) + [(one.key_cache[0], two.key_cache[0])]:
        assert (torch.isnan(a) == torch.isnan(b)).all()
        assert _same(a.masked_fill(torch.isnan(a), 0), b.masked_fill(torch.isnan(b), 0))
    assert _same(one.value_cache[0], two.value_cache[0])


def test_head_strides_of_zero(dev):
    """One projected head seen as many (expand): the reads repeat, the results are whole."""
    B, Hq, H, S, D, dtype = 2, 16, 8, 130, 64, torch.float16
    sizes, static = _ring_plan(H)
    q, k, v, cos, sin = _inputs(dev, dtype, B, 1, 1, S, D)
    args = (q.expand(B, Hq, S, D), k.expand(B, H, S, D), v.expand(B, H, S, D), cos, sin)
    one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
    assert one._prompt_fits_one_launch(*args, 0, None)
    _check(one.rope_update(*args, 0, None)[:2], _two_steps(two, *args, None), one, two, "expanded")


@pytest.mark.parametrize("fresh", [True, False])
def test_recorded_into_a_graph(dev, fresh):
    """Replays on new inputs equal the two steps run eagerly: with rings that the recorded call allocates (every replay
    writes all of their rows) and with rings in use."""
    B, Hq, H, S, D, dtype = 2, 8, 8, 300, 64, torch.float16
    sizes, static = _ring_plan(H)
    one, two = (_cache(dev, dtype, B, D, sizes, static) for _ in range(2))
    args, mask = _inputs(dev, dtype, B, Hq, H, S, D), _padding(dev, B, S)
    if not fresh:
        one.rope_update(*args, 0, mask)
        _two_steps(two, *args, mask)
    start = {n: getattr(one, n)[0].clone() for n in TABLES}
    warm = _cache(dev, dtype, B, D, sizes, static)
    warm.rope_update(*args, 0, mask)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = one.rope_update(*args, 0, mask)[:2]
    for i in range(3):
        for t in args[:3]:
            t.copy_(torch.randn(t.shape, generator=torch.Generator().manual_seed(i)).to(dev, dtype))
        mask.copy_(mask.roll(7, dims=1))
        if fresh:   # a replay starts where the recorded call did: in front of the prompt
            two = _cache(dev, dtype, B, D, sizes, static)
            for n in TABLES:
                getattr(one, n)[0].copy_(start[n])
            for ring in (one.key_cache[0], one.value_cache[0]):
                ring.fill_(float("nan"))
        else:       # the recorded length of what the ring had seen
            two._kv_len[0] = S
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        _check(got, _two_steps(two, *args, mask), one, two, i)
