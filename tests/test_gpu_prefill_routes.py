"""The two prompt kernels at the sizes where each can go wrong: work-groups of one 128-row item (short prompts, few
items) and resident work-groups of 256-row items (the others).  Tolerances as in prefill_checks.py."""
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
