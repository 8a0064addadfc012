"""The work whose time matters to a user of this package, as cases that a timing program can prepare and run.

Three kinds of calls make up a generation, each through the public entry points a model calls them by:

  decode    one generated token in ``layers`` decoder layers: ``StaticCircularCache.rope_update`` (or ``update`` on
            keys that are rotated already) and ``mixture_of_sparse_attention`` over the rings, layer by layer
  attention the prompt's block-sparse attention alone: ``mixture_of_sparse_attention`` on q, k, v of one layer
  prompt    the start of a generation in ``layers`` layers: a new ``StaticCircularCache``, ``rope_update`` on the whole
            prompt (rotary embedding and ring insert) and, with ``attend``, the prompt's attention

Every kv head has a window of its own, ``alpha + beta * context`` rounded up to blocks of 64 tokens with alpha and beta
drawn per head (``elastic_spans``), behind 64 sink tokens: the spans of the benchmark's configurations.  There is no
backward pass in this package: it is inference only.
"""
import math

import torch

from moa_amd import StaticCircularCache, mixture_of_sparse_attention
from moa_amd.models.llama.modeling_llama import rotary_cos_sin
from moa_amd.workloads import (append_bytes, decode_bytes, elastic_spans, prefill_work, ring_cache_sizes,
                               rope_append_bytes)

SINK = 64
DTYPES = {"float16": torch.float16, "bfloat16": torch.bfloat16}


def _decode(batch, heads, kv_heads, head_dim, context, alpha_hi, dtype, fused, layers):
    return {"kind": "decode", "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
            "context": context, "alpha_hi": alpha_hi, "dtype": dtype, "fused": fused, "layers": layers}


def _attention(batch, heads, kv_heads, head_dim, context, alpha_hi, dtype):
    return {"kind": "attention", "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
            "context": context, "alpha_hi": alpha_hi, "dtype": dtype}


def _prompt(batch, heads, kv_heads, head_dim, context, alpha_hi, dtype, padded, attend, layers):
    return {"kind": "prompt", "batch": batch, "heads": heads, "kv_heads": kv_heads, "head_dim": head_dim,
            "context": context, "alpha_hi": alpha_hi, "dtype": dtype, "padded": padded, "attend": attend,
            "layers": layers}


def listed():
    cases = {
        # one user's chat on a small grouped-query model, short context: latency and launches are everything
        "decode_one_short": _decode(1, 32, 8, 128, 1024, 256, "bfloat16", True, 1),
        # one user at 16k tokens, a ring per query head (the 7B shape), four layers in a row
        "decode_one_long": _decode(1, 32, 32, 128, 16384, 2048, "float16", True, 4),
        # the 7B whole-decoder configuration's step: batch 8, 16k tokens
        "decode_batch8": _decode(8, 32, 32, 128, 16384, 2048, "bfloat16", True, 4),
        # the headline workload: batch 64 at 16k tokens, append and attention as two calls
        "decode_batch64": _decode(64, 32, 32, 128, 16384, 2048, "float16", False, 1),
        # the 70B whole-decoder configuration's step: 64 query heads on 8 rings, batch 4, 32k tokens
        "decode_grouped": _decode(4, 64, 8, 128, 32768, 8192, "bfloat16", True, 4),
        # an odd batch, an odd context and a group of 7 with 64-element heads
        "decode_ragged": _decode(13, 28, 4, 64, 5001, 1024, "float16", True, 2),
        # the smallest benchmark prompt: one sequence of 2048 tokens, 64-element heads
        "attention_small": _attention(1, 32, 32, 64, 2048, 1024, "float16"),
        # a prompt batch whose length is not a multiple of the block
        "attention_ragged": _attention(2, 32, 32, 128, 3001, 1024, "float16"),
        # the headline prompt: batch 4 of 8192 tokens
        "attention_8k": _attention(4, 32, 32, 128, 8192, 2048, "bfloat16"),
        # the longest prompt: 32k tokens, 64 query heads on 8 kv heads
        "attention_32k": _attention(1, 64, 8, 128, 32768, 8192, "bfloat16"),
        # a short question to a 7B-shaped model, start of the generation with the attention, two layers
        "prompt_short": _prompt(1, 32, 32, 128, 517, 256, "float16", False, True, 2),
        # filling the rings from a batch of long prompts with left padding, without the attention
        "prompt_fill": _prompt(8, 32, 32, 128, 16384, 2048, "bfloat16", True, False, 1),
    }
    return [dict(c, name=name) for name, c in cases.items()]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(case):
    """A rough time of one pass in seconds, to keep drawn cases within the listed ones."""
    w = work(case)
    return max(w["bytes"] / 5e12, w["flops"] / 1e15)


def draw(rng):
    """One more case of the same ranges: batch 1 to 64, contexts of some hundred to 32k tokens (odd ones mostly), one
    to eight query heads per ring, both head sizes and both types."""
    limit = {"decode": 1.1e-3, "attention": 1.0e-2, "prompt": 1.0e-2}
    while True:
        kind = rng.choice(["decode", "decode", "attention", "prompt"])
        group = rng.choice([1, 1, 1, 2, 4, 5, 7, 8])
        kv_heads = rng.choice([4, 8, 12, 16, 32, 40]) if group == 1 else rng.choice([1, 2, 4, 8])
        head_dim = rng.choice([64, 128, 128])
        dtype = rng.choice(["float16", "bfloat16"])
        context = _log_int(rng, 300 if kind == "decode" else 130, 32768)
        batch = _log_int(rng, 1, 64 if kind == "decode" else 8)
        alpha_hi = rng.choice([256, 1024, 2048, 8192])
        heads = kv_heads * group
        if kind == "decode":
            case = _decode(batch, heads, kv_heads, head_dim, context, alpha_hi, dtype, rng.random() < 0.6,
                           rng.choice([1, 2, 4]))
        elif kind == "attention":
            case = _attention(batch, heads, kv_heads, head_dim, context, alpha_hi, dtype)
        else:
            case = _prompt(batch, heads, kv_heads, head_dim, context, alpha_hi, dtype, rng.random() < 0.5,
                           rng.random() < 0.5, rng.choice([1, 2]))
        if _cost(case) <= limit[kind]:
            return case


def _spans(case, layer):
    """The windows of a layer's kv heads (part of the model's plan, so the same for every seed of the inputs)."""
    lo = min(64.0, case["alpha_hi"])
    if case["alpha_hi"] >= 8192:
        lo = 256.0
    return elastic_spans(case["kv_heads"], case["context"], layer, (lo, float(case["alpha_hi"])))


def _rings(case):
    sizes = [ring_cache_sizes(_spans(case, l), SINK) for l in range(case.get("layers", 1))]
    return [c for c, _ in sizes], [s for _, s in sizes]


def _new_cache(case):
    cache_size, static_size = _rings(case)
    return StaticCircularCache(cache_size, batch_size=case["batch"], head_dim=case["head_dim"],
                               static_size=static_size, device="cuda", dtype=DTYPES[case["dtype"]])


def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    B, Hq, Hkv, D, N = (case[k] for k in ("batch", "heads", "kv_heads", "head_dim", "context"))

    def projection(heads, tokens):
        """What a projection leaves: [B, tokens, heads, D], viewed [B, heads, tokens, D] as the model views it."""
        return torch.randn(B, tokens, heads, D, generator=gen, device="cuda", dtype=dtype).transpose(1, 2)

    state = {"case": case, "sm_scale": D ** -0.5}
    tokens = 1 if case["kind"] == "decode" else N
    layers = case.get("layers", 1)
    state["qkv"] = [(projection(Hq, tokens), projection(Hkv, tokens), projection(Hkv, tokens)) for _ in range(layers)]
    if case["kind"] == "attention":
        state["sink"] = torch.full((Hkv,), SINK, dtype=torch.int64, device="cuda")
        state["local"] = torch.tensor(_spans(case, 0), dtype=torch.int64, device="cuda")
        return state
    first = N if case["kind"] == "decode" else 0
    position = torch.arange(first, first + tokens, device="cuda")[None, :]
    state["cos"], state["sin"] = rotary_cos_sin(position, D, dtype)
    if case["kind"] == "decode":
        # the rings as a prompt of N tokens leaves them: the bookkeeping through the prompt's own update (of keys
        # that are all the same, so that no prompt has to be made), then contents of their own
        cache = _new_cache(case)
        blank = torch.zeros(1, 1, 1, D, dtype=dtype, device="cuda").expand(B, Hkv, N, D)
        for layer in range(layers):
            cache.update(blank, blank, layer)
            cache.key_cache[layer].normal_(generator=gen)
            cache.value_cache[layer].normal_(generator=gen)
        state["cache"] = cache
    else:
        state["mask"] = None
        if case["padded"]:   # left padding: up to a quarter of a row; the longest row has none
            pad = torch.randint(0, max(1, N // 4), (B, 1), generator=gen, device="cuda")
            pad[0] = 0
            state["mask"] = (torch.arange(N, device="cuda")[None, :] >= pad).to(torch.int64)
    return state


def _attend(state, cache, layer, q, keys, values):
    return mixture_of_sparse_attention(
        q, keys, values, state["sm_scale"], sink_size=cache.static_cache_size[layer],
        local_size=cache.circular_cache_size[layer], head_start_index=cache.cache_head_start_index[layer],
        head_valid_length=cache.cache_valid_length[layer])


def _rings_of(cache, layer):
    return [cache.key_cache[layer], cache.value_cache[layer], cache.mask_cache[layer],
            cache.cache_update_index[layer], cache.cache_valid_length[layer]]


def run(state):
    case = state["case"]
    if case["kind"] == "attention":
        q, k, v = state["qkv"][0]
        return mixture_of_sparse_attention(q, k, v, state["sm_scale"], sink_size=state["sink"],
                                           local_size=state["local"])
    results = []
    if case["kind"] == "decode":
        cache = state["cache"]
        for layer, (q, k, v) in enumerate(state["qkv"]):
            if case["fused"]:
                q, keys, values = cache.rope_update(q, k, v, state["cos"], state["sin"], layer)
            else:
                keys, values = cache.update(k, v, layer)
            results.append([_attend(state, cache, layer, q, keys, values)] + _rings_of(cache, layer))
        return results
    cache = _new_cache(case)
    for layer, (q, k, v) in enumerate(state["qkv"]):
        q, keys, values = cache.rope_update(q, k, v, state["cos"], state["sin"], layer, state["mask"])
        out = [_attend(state, cache, layer, q, keys, values)] if case["attend"] else [q, keys]
        results.append(out + _rings_of(cache, layer))
    return results


def work(case):
    B, Hq, Hkv, D, N = (case[k] for k in ("batch", "heads", "kv_heads", "head_dim", "context"))
    group = Hq // Hkv
    total_bytes = flops = 0.0
    for layer in range(case.get("layers", 1)):
        spans = _spans(case, layer)
        if case["kind"] == "decode":
            rows = B * sum(min(N + 1, SINK + s) for s in spans)
            # q in, o out, both of all query heads; K and V rows of the rings once
            total_bytes += decode_bytes(rows, B, Hkv, D) + 4 * B * (Hq - Hkv) * D
            total_bytes += append_bytes(B, Hkv, D)
            if case["fused"]:   # the rotated q is a result of its own
                total_bytes += rope_append_bytes(B, Hkv, D) - append_bytes(B, Hkv, D) + 4 * B * (Hq - Hkv) * D
            flops += 4.0 * D * rows * group
            continue
        q_bytes, kv_bytes = 2.0 * B * Hq * N * D, 2.0 * B * Hkv * N * D
        if case["kind"] == "prompt":
            # rotary embedding of q and k, both results of their own; the kept rows of K and V into new rings, whose
            # other rows are zero; v is read where it is kept
            ring_bytes = 2.0 * B * sum(SINK + s for s in spans) * D
            kept = 2.0 * B * sum(min(N, SINK + s) for s in spans) * D
            total_bytes += 2 * (q_bytes + kv_bytes) + 4.0 * N * D + kept + 2 * ring_bytes + 4 * ring_bytes / D
        if case["kind"] == "attention" or case["attend"]:
            total_bytes += 2 * q_bytes + 2 * kv_bytes
            flops += group * prefill_work(N, [SINK // 64] * Hkv, [s // 64 for s in spans], B, D)[0]
    return {"bytes": total_bytes, "flops": flops}


def tolerance(case):
    # The output's own rounding to 16 bits, and in the matrix kernels that of the softmax weights; sums are fp32.
    # Against the same attention in 64 bits these cases are off by 2.1e-4 to 3.0e-4 in float16 and by 1.6e-3 to
    # 2.7e-3 in bfloat16: four times that.
    return {"rel": 1.2e-3 if case["dtype"] == "float16" else 1e-2}


def _rotated(x, cos, sin):
    """Rotary embedding in 64 bits (cos and sin are inputs, in 16 bits as the model holds them)."""
    a = x.double()
    half = a.shape[-1] // 2
    turned = torch.cat((-a[..., half:], a[..., :half]), dim=-1)
    return a * cos.double()[:, None] + turned * sin.double()[:, None]


def _exact_prompt_attention(q, k, v, scale, spans):
    """Block-sparse causal attention in 64 bits, a head and some query blocks at a time: [B, N, Hq, D]."""
    B, Hq, N, D = q.shape
    group = Hq // k.shape[1]
    out = torch.empty(B, N, Hq, D, dtype=torch.float64, device=q.device)
    col = torch.arange(N, device=q.device)[None, :]
    step = 2048
    for b in range(B):
        for h in range(Hq):
            kd, vd = k[b, h // group].double(), v[b, h // group].double()
            for lo in range(0, N, step):
                hi = min(N, lo + step)
                row = torch.arange(lo, hi, device=q.device)[:, None]
                live = (col[:, :hi] <= row) & ((col[:, :hi] < SINK) |
                                               (row // 64 - col[:, :hi] // 64 < spans[h // group] // 64))
                score = (q[b, h, lo:hi].double() @ kd[:hi].t()) * scale
                out[b, lo:hi, h] = torch.softmax(score.masked_fill_(~live, -math.inf), dim=-1) @ vd[:hi]
    return out


def exact(case, seed):
    """What ``run`` returns, by torch in 64 bits.  Rotated keys are rounded to the 16 bits of the rings they are kept
    in; None stands for what is bookkeeping or a copy of other outputs."""
    state = prepare(case, seed)
    scale, group, D = state["sm_scale"], case["heads"] // case["kv_heads"], case["head_dim"]
    if case["kind"] == "attention":
        q, k, v = state["qkv"][0]
        return _exact_prompt_attention(q, k, v, scale, _spans(case, 0))
    results = []
    for layer, (q, k, v) in enumerate(state["qkv"]):
        if case["kind"] == "prompt" or case["fused"]:
            q, k = (_rotated(x, state["cos"], state["sin"]) for x in (q, k))
        if case["kind"] == "prompt":
            if case["attend"]:
                q, k = q.to(v.dtype), k.to(v.dtype)
                results.append([_exact_prompt_attention(q, k, v, scale, _spans(case, layer))] + [None] * 5)
            else:
                results.append([q, k] + [None] * 5)
            continue
        q, k = q.to(v.dtype), k.to(v.dtype)
        cache = state["cache"]
        keys, values = cache.key_cache[layer].clone(), cache.value_cache[layer].clone()
        slot, valid = cache.cache_update_index[layer], cache.cache_valid_length[layer]
        start, room = cache.cache_head_start_index[layer], cache.cache_max_length[layer]
        each = torch.arange(case["batch"], device=keys.device)[:, None]
        keys[each, slot], values[each, slot] = k[:, :, 0], v[:, :, 0]
        out = torch.empty(case["batch"], 1, case["heads"], D, dtype=torch.float64, device=keys.device)
        for h in range(case["kv_heads"]):   # no padding here: the rows of a batch are filled alike
            first = int(start[0, h])
            rows = slice(first, first + min(int(valid[0, h]) + 1, int(room[h])))
            heads = slice(h * group, (h + 1) * group)
            score = q[:, heads, 0].double() @ keys[:, rows].double().transpose(1, 2).contiguous() * scale
            out[:, 0, heads] = torch.softmax(score, dim=-1) @ values[:, rows].double()
        results.append([out, keys, values, None, None, None])
    return results
