"""The workloads by which the speed of this package is judged, through its public entry points.

Six kinds of work, each a pass as a serving program makes it:

* ``decode``    one token's attention through ``polar_cache.compute`` for every layer of a stack: collision vote, candidate
                select, 4-bit rerank, top-k, gather, attention.  K/V in HBM or in pinned host memory, bf16 or fp32.
* ``adaptive``  the same through the two adaptive-k cache classes (per-row k with K/V on the host, and the dense form).
* ``prefill``   ``prefill_update_kv_cache`` of a prompt: K/V stored (and offloaded), keys encoded, cluster sizes counted, value
                norms kept where the class needs them.
* ``chat``      a short conversation: prompt, then tokens one by one (append + attention), with index refreshes on the way.
* ``model``     the decode loop of the Qwen3-shaped model glue over a cached prompt, with given tokens.
* ``operators`` the stand-alone operators in the tensor layouts of the original project (subspace-major index): vote count,
                coarse filter, 4-bit rerank, top-k.

Keys are ~N(0, 1) with four outlier channels and a mean that turns along the prompt, values ~N(0, 1), queries the mean of the
recent keys + N(0, 0.5), as in this repository's tests and benchmark.
"""
import math

import torch

from pariskv_amd import ops

DEV = "cuda:0"
D = 128
RECENT = 512            # keys whose mean the queries lie around
SINK, LOCAL, INTERVAL = 64, 512, 512


def listed():
    return [
        # one user, a short context, one layer: launches and latency are everything
        dict(name="decode_4k_b1", kind="decode", bs=1, heads=8, group=4, ctx=4096, layers=1, dtype="bf16", host=False,
             topk=100, buffered=17),
        # one user, a document in context, K/V in HBM
        dict(name="decode_32k_b1", kind="decode", bs=1, heads=8, group=4, ctx=32768, layers=4, dtype="bf16", host=False,
             topk=512, buffered=100),
        # a full serving batch, K/V in HBM
        dict(name="decode_64k_b8", kind="decode", bs=8, heads=8, group=4, ctx=65536, layers=2, dtype="bf16", host=False,
             topk=100, buffered=211),
        # long contexts with the K/V store in pinned host memory, the caches' default mode: the gather crosses PCIe
        dict(name="decode_128k_b2_host", kind="decode", bs=2, heads=8, group=4, ctx=131072, layers=1, dtype="bf16", host=True,
             topk=1024, buffered=64),
        # fp32 cache (the CPU reference's type), odd length, seven query heads to a KV head
        dict(name="decode_9001_b3_f32", kind="decode", bs=3, heads=4, group=7, ctx=9001, layers=2, dtype="f32", host=False,
             topk=256, buffered=33),
        # adaptive k on a million keys, K/V on the host
        dict(name="adaptive_1m_b1_host", kind="adaptive", bs=1, heads=8, group=4, ctx=1048576, layers=1, form="varlen",
             host=True, buffered=10),
        # adaptive k in its dense form, everything in HBM, ragged sizes
        dict(name="adaptive_41k_b3", kind="adaptive", bs=3, heads=8, group=4, ctx=41003, layers=2, form="dense", host=False,
             buffered=75),
        # a batch of prompts into HBM
        dict(name="prefill_64k_b4", kind="prefill", bs=4, heads=8, ctx=65536, layers=2, dtype="bf16", cls="fixed", host=False,
             per_sample=False),
        # one prompt of odd length into the adaptive cache: value norms, and the copy to the host
        dict(name="prefill_30011_b1_host", kind="prefill", bs=1, heads=8, ctx=30011, layers=3, dtype="bf16", cls="varlen",
             host=True, per_sample=True),
        # a short chat in the default mode: starts below the length where retrieval pays, refreshes the index once
        dict(name="chat_1500", kind="chat", bs=1, heads=8, group=4, ctx=1500, tokens=160, interval=128, layers=2, host=True,
             topk=100),
        # the model's own decode loop, four layers of the 8B shape
        dict(name="model_12k_b2", kind="model", bs=2, ctx=12000, tokens=16, layers=4, host=False, topk=100),
        # the operators on the original project's contiguous subspace-major tensors
        dict(name="operators_20011_b2", kind="operators", bs=2, heads=8, ctx=20011, topk=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choices(["decode", "adaptive", "prefill", "chat", "model", "operators"], [36, 16, 18, 10, 6, 14])[0]
    heads, group = rng.choice([(8, 4), (8, 4), (8, 4), (4, 7), (4, 8), (2, 8), (8, 8), (8, 5), (2, 4)])
    host = rng.random() < 0.4
    if kind == "decode":
        f32 = rng.random() < 0.2
        bs = rng.choice([1, 1, 2, 3, 4, 8])
        ctx = _log(rng, 2700, min(262144, (1 << 20 if host else 1 << 22) // (bs * heads * (2 if f32 else 1))))
        return dict(kind=kind, bs=bs, heads=heads, group=group, ctx=ctx, layers=rng.choice([1, 2, 4]) if ctx * bs < 100000 else 1,
                    dtype="f32" if f32 else "bf16", host=host, topk=_log(rng, 40, 1024), buffered=rng.randrange(0, 256))
    if kind == "adaptive":
        form = "varlen" if host else rng.choice(["dense", "dense", "varlen"])
        host = True if form == "varlen" else host
        bs = rng.choice([1, 1, 2, 4])
        ctx = _log(rng, 2700, (1 << 22) // (bs * 8))
        return dict(kind=kind, bs=bs, heads=min(heads, 8), group=group, ctx=ctx, layers=rng.choice([1, 2]) if ctx < 60000 else 1,
                    form=form, host=host, buffered=rng.randrange(0, 256))
    if kind == "prefill":
        cls = rng.choice(["fixed", "fixed", "varlen", "dense"])
        host = True if cls == "varlen" else host
        bs = rng.choice([1, 1, 2, 4])
        f32 = rng.random() < 0.2
        ctx = _log(rng, 900, min(131072, (1 << 18 if host else 1 << 21) // (bs * heads)))
        return dict(kind=kind, bs=bs, heads=heads, ctx=ctx, layers=rng.choice([1, 2]), dtype="f32" if f32 else "bf16", cls=cls,
                    host=host, per_sample=bs == 1 or rng.random() < 0.3)
    if kind == "chat":
        return dict(kind=kind, bs=rng.choice([1, 1, 2]), heads=heads, group=group, ctx=_log(rng, 700, 6000),
                    tokens=rng.randrange(40, 160), interval=rng.choice([32, 64, 128]), layers=rng.choice([1, 2]), host=host,
                    topk=_log(rng, 40, 256))
    if kind == "model":
        return dict(kind=kind, bs=rng.choice([1, 2, 4, 8]), ctx=_log(rng, 3000, 16000), tokens=rng.randrange(4, 15),
                    layers=rng.choice([2, 3, 4]), host=rng.random() < 0.3, topk=_log(rng, 40, 256))
    return dict(kind=kind, bs=rng.choice([1, 2, 3]), heads=heads, ctx=_log(rng, 3000, 80000), topk=_log(rng, 40, 1024))


# ------------------------------------------------------------------------------------------------ what a program has in hand


def _dtype(case):
    return torch.float32 if case.get("dtype") == "f32" else torch.bfloat16


def _class(case):
    cls = case.get("cls") or case.get("form") or "fixed"
    if cls == "varlen":
        from pariskv_amd.cache_hub.polar_cache_adaptivek_varlen import polar_cache
    elif cls == "dense":
        from pariskv_amd.cache_hub.polar_cache_atten_value_indices_adaptive_k import polar_cache
    else:
        from pariskv_amd.cache_hub.polar_cache import polar_cache
    return polar_cache


def _make_cache(case, new_tokens):
    bs, H, G, S = case["bs"], case.get("heads", 8), case.get("group", 4), case["ctx"]
    return _class(case)(valid_start=[0] * bs, layer_num=case["layers"], batch_size=bs, max_length=S + new_tokens,
                        num_key_value_heads=H, num_heads=H * G, head_dim=D, dtype=_dtype(case),
                        layer_mapping={i: DEV for i in range(case["layers"])}, max_new_length=new_tokens, sink_size=SINK,
                        local_size=LOCAL, num_gpus=1, model_size=8, final_topk=case.get("topk", 100),
                        dynamic_update_interval=case.get("interval", INTERVAL), full_attention_threshold=2000,
                        enable_offload=case["host"])


def _keys(g, bs, S, H, dtype, phase=0.0):
    k = torch.randn(bs, S, H, D, generator=g, device=DEV, dtype=dtype)
    ang = phase + torch.arange(S, device=DEV, dtype=torch.float32) * (0.5 / 1000.0) * (math.pi / 180.0)
    k[..., 0] += (2.0 * ang.cos()).to(dtype)[None, :, None]
    k[..., 1] += (2.0 * ang.sin()).to(dtype)[None, :, None]
    k[..., [7, 31, 64, 101]] *= 10.0
    return k


def _prompt(g, case):
    bs, H, S, dt = case["bs"], case.get("heads", 8), case["ctx"], _dtype(case)
    k = _keys(g, bs, S, H, dt)
    v = torch.randn(bs, S, H, D, generator=g, device=DEV, dtype=dt)
    return k, v


def _queries(g, recent, group):
    """recent [bs, n, H, D] -> queries [bs, 1, H * group, D] around the mean of these keys."""
    bs, _, H, _ = recent.shape
    mean = recent.float().mean(dim=1).repeat_interleave(group, dim=1)
    return (mean + 0.5 * torch.randn(bs, H * group, D, generator=g, device=DEV)).to(recent.dtype).view(bs, 1, H * group, D)


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    kind, bs, S = case["kind"], case["bs"], case["ctx"]
    if kind in ("decode", "adaptive"):
        cache, qs = _make_cache(case, case["buffered"] + 8), []
        for l in range(case["layers"]):
            k, v = _prompt(g, case)
            cache.prefill_update_kv_cache(None, k, v, l, 0)
            qs.append(_queries(g, k[:, -RECENT:], case["group"]))
        new_k = _keys(g, bs, case["buffered"] + 1, case["heads"], _dtype(case))
        new_v = torch.randn(new_k.shape, generator=g, device=DEV, dtype=new_k.dtype)
        for t in range(case["buffered"]):
            for l in range(case["layers"]):
                cache.decode_update_kv_cache(new_k[:, t:t + 1], new_v[:, t:t + 1], l)
        torch.cuda.synchronize()   # a prompt's copies to the host are over long before its later tokens
        return dict(kind=kind, cache=cache, q=qs)
    if kind == "prefill":
        return dict(kind=kind, cache=_make_cache(case, 64), kv=[_prompt(g, case) for _ in range(case["layers"])],
                    per_sample=case["per_sample"], bs=bs)
    if kind == "chat":
        T, L, H, G = case["tokens"], case["layers"], case["heads"], case["group"]
        kv = [_prompt(g, case) for _ in range(L)]
        new = [[(_keys(g, bs, 1, H, torch.bfloat16), torch.randn(bs, 1, H, D, generator=g, device=DEV, dtype=torch.bfloat16),
                 _queries(g, kv[l][0][:, -RECENT:], G)) for l in range(L)] for _ in range(T)]
        return dict(kind=kind, cache=_make_cache(case, T + 8), kv=kv, new=new)
    if kind == "model":
        from pariskv_amd.model_hub import QwenConfig, QwenModel

        cfg = QwenConfig(num_layers=case["layers"], vocab_size=32000)
        cache = _make_cache(case, case["tokens"] + 8)
        model = QwenModel(cfg, cache, device=DEV, max_positions=S + case["tokens"] + 8, seed=seed)
        ids = torch.randint(0, cfg.vocab_size, (bs, case["tokens"]), generator=g, device=DEV)
        return dict(kind=kind, cache=cache, model=model, kv=[_prompt(g, case) for _ in range(case["layers"])], ids=ids)
    # operators: the index as the original project lays it out (contiguous, subspace-major) and a step's query side
    H, N = case["heads"], S
    keys = _keys(g, bs, N, H, torch.bfloat16).permute(0, 2, 1, 3)
    signs = ops.srht_signs(DEV)
    codebook = torch.zeros(bs, H, 16, N, dtype=torch.uint8, device=DEV)
    key_4bit = torch.zeros(bs, H, 16, N, 4, dtype=torch.uint8, device=DEV)
    weight = torch.zeros(bs, H, 16, N, dtype=torch.bfloat16, device=DEV)
    counts = torch.zeros(bs, H, 16, 256, dtype=torch.int32, device=DEV)
    ops.encode_append(keys, signs, codebook, key_4bit, weight, counts)
    q = _queries(g, keys[:, :, -RECENT:].permute(0, 2, 1, 3), 4)
    tiers = [int(math.ceil(N * 0.25 * r)) for r in ops.TIER_RATIOS]
    qhat, qnorm, _, sorted_ids = ops.query_prep_lut(q, H, signs, counts, tiers, want_sorted_ids=True)
    return dict(kind=kind, sorted_ids=sorted_ids, counts=counts, codebook=codebook, key_4bit=key_4bit, weight=weight,
                q_blocks=qhat.view(bs, H, 16, 8), q_norm=qnorm.view(bs, H, 1), centers=ops.mag_centers(DEV), tiers=tiers,
                ratio=_ratio(N), topk=case["topk"])


# ------------------------------------------------------------------------------------------------------------------ one pass


def _fill(cache, kv, per_sample, bs):
    for l, (k, v) in enumerate(kv):
        if per_sample:
            for b in range(bs):
                cache.prefill_update_kv_cache(None, k[b:b + 1], v[b:b + 1], l, b)
        else:
            cache.prefill_update_kv_cache(None, k, v, l, 0)


def run(state):
    kind = state["kind"]
    if kind == "operators":
        from pariskv_amd.cache_hub.collision_fused import update_cache_cnt_cuda_interface
        from pariskv_amd.cache_hub.rerank.rerank import rerank_rabitq_fused

        cnt = update_cache_cnt_cuda_interface(state["sorted_ids"], state["counts"], state["codebook"], state["tiers"])
        final, scores, v4b = rerank_rabitq_fused(cnt, state["key_4bit"], state["weight"], state["q_blocks"], state["q_norm"],
                                                 state["centers"], state["ratio"], state["topk"], 16, 8)
        return dict(votes=cnt, ids=final, scores=scores, values=v4b)
    cache = state["cache"]
    if kind in ("decode", "adaptive"):
        return [cache.compute(q, l) for l, q in enumerate(state["q"])]
    cache.context = 0   # a new prompt in the same cache
    if kind == "prefill":
        _fill(cache, state["kv"], state["per_sample"], state["bs"])
        out = {}
        for l in range(len(state["kv"])):
            out[f"index{l}"] = (cache.codebook_gpu[l], cache.key_4bit_packed_gpu[l], cache.key_block_weight_gpu[l],
                                cache.cluster_key_counts_gpu[l])
            out[f"kv{l}"] = (cache.unified_keys_gpu[l], cache.unified_values_gpu[l])
            if cache.enable_offload:
                out[f"host{l}"] = (cache.unified_keys_cpu[l], cache.unified_values_cpu[l])
            if hasattr(cache, "value_norm_gpu"):
                out[f"norms{l}"] = (cache.value_norm_gpu[l], cache._sl_vnorm_cache[l])
        return out
    _fill(cache, state["kv"], False, 0)
    if kind == "model":
        ids = state["ids"]
        return [state["model"].decode_forward(ids[:, t:t + 1]) for t in range(ids.shape[1])]
    out = []
    for token in state["new"]:
        for l, (k, v, q) in enumerate(token):
            cache.decode_update_kv_cache(k, v, l)
            out.append(cache.compute(q, l))
    return torch.cat(out, dim=1)   # [bs, tokens * layers, heads, 128]


# ------------------------------------------------------------------------------- what a pass cannot do without, and how exact


def _ratio(n):
    return 0.5 if n < 5000 else 0.25 if n < 10000 else 0.2 if n < 30000 else 0.1


def _step(bs, heads, group, n, dense, topk, cand, es, norms=False):
    """Bytes and operations of one layer's retrieval + attention: codes, candidates' records, attended rows, query and output."""
    rows = bs * heads
    b = rows * (16 * n + (96 + 4 * norms) * cand + 2 * D * es * (dense + topk) + 2 * group * D * es)
    f = rows * (16 * n + 2 * D * cand + 4 * group * D * (dense + topk))
    return b, f


def work(case):
    kind, bs, H, S = case["kind"], case["bs"], case.get("heads", 8), case["ctx"]
    es = 4 if case.get("dtype") == "f32" else 2
    group, topk = case.get("group", 4), case.get("topk", 100)
    n0 = max(0, S - SINK - LOCAL)
    prefill = (bs * H * (S * 4 * D * es + n0 * 112), bs * H * n0 * 3000)
    if kind in ("decode", "adaptive"):
        dense = SINK + LOCAL + case["buffered"]
        if kind == "decode":
            c = math.ceil(n0 * _ratio(n0))
            b, f = _step(bs, H, group, n0, dense, min(topk, c), c, es)
        else:
            c = math.ceil(n0 * (0.05 if n0 >= 30000 else _ratio(n0)))
            k = min(800 if case["form"] == "varlen" else 1300, c)   # the cap of the one form, what the other takes on such keys
            b, f = _step(bs, H, group, n0, dense, k, c, es, norms=True)
        return dict(bytes=b * case["layers"], flops=f * case["layers"])
    if kind == "prefill":
        norms = bs * H * S * 4 if case["cls"] != "fixed" else 0
        return dict(bytes=(prefill[0] + norms) * case["layers"], flops=prefill[1] * case["layers"])
    if kind in ("chat", "model"):
        interval = case.get("interval", INTERVAL)
        b, f = prefill
        for t in range(case["tokens"]):
            seq, moved = S + t + 1, ((t + 1) // interval) * interval
            n = n0 + moved
            if seq < 2000:
                tb, tf = _step(bs, H, group, 0, seq, 0, 0, es)
            else:
                c = math.ceil(n * _ratio(n))
                tb, tf = _step(bs, H, group, n, seq - n, min(topk, c), c, es)
            b, f = b + tb + bs * H * 4 * D * es, f + tf
        b, f = b * case["layers"], f * case["layers"]
        if kind == "model":
            hid, inter, vocab = 4096, 12288, 32000
            weights = case["layers"] * hid * (6144 + 4096 + 3 * inter) + vocab * hid
            b, f = b + case["tokens"] * 2 * weights, f + case["tokens"] * 2 * weights * bs
        return dict(bytes=b, flops=f)
    # operators: codes in, int32 votes out and in again (two calls), candidates' entries in, ids + scores + unpacked values out
    c, rows = math.ceil(S * _ratio(S)), bs * H
    return dict(bytes=rows * (16 * S + 8 * S + 16 * 256 * 12 + c * (96 + 4 + 256) + 8 * min(topk, c)),
                flops=rows * (16 * S + 2 * D * c))


def tolerance(case):
    kind = case["kind"]
    if kind == "prefill":
        # copies, codes and counts are exact; a value norm is rounded to the cache's type from a sum in some order: a few in a
        # million land on the neighbouring bf16 value (1.1e-5 in the norms against sums in 64 bits)
        return "exact" if case["cls"] == "fixed" else dict(rel=5e-5)
    if kind == "operators":
        return dict(rel=1e-5, differ=1e-3)   # fp32 sums of 128 products; ids of equal scores may change places
    if kind == "model":
        # four layers, each of which keeps the best 100 of 12000 keys: a last-bit difference of a projection moves keys over
        # that border.  Summing the projections in another order changes the logits by 0.03 to 0.08.
        return dict(rel=2e-1)
    # bf16: 2.1e-3 against attention over the same set in 64 bits; fp32: 4e-7, and a wider border case of the selection
    return dict(rel=5e-6 if case.get("dtype") == "f32" else 8e-3)
