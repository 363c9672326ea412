"""Cases of the framework's work for timing and for comparing results.

``listed`` names them, ``draw`` gives more of the same ranges, ``prepare``
makes what a program holds before the call, ``run`` is one pass through the
public entry points, ``work`` what a pass cannot do without, ``exact`` the
result in float64 from plain torch and ``tolerance`` how far another correct
implementation at the same precision may be from it.

Kinds of cases:

``hook``     one attention layer's call, ``fpv2.fpv2_sdpa`` on ``[1, H, L, D]``
             tensors (what the SDPA hook calls): a whole prompt
             (queries == keys) or one chunk of queries at the end of a prefix.
``chunked``  a prompt fed to ``fpv2.ChunkedPrefill`` chunk by chunk.
``ops``      the operators one by one on padded tensors: ``pool_blocks``,
             ``block_scores_and_select``, ``density``,
             ``compact_block_indices``, ``sparse_attention``.
``select``   ``block_scores_and_select`` alone, with its raw scores.
``prefill``  chunked prefill of a random-init decoder (Qwen3-4B layer
             geometry, fewer layers) to the first logits.

Data: i.i.d. N(0, 1) with a unit direction per KV head planted in the keys of
block 0 and of a few other blocks and in every query.  ``sparse`` plants it
strongly, so that most blocks are pruned (a long prompt with a few relevant
places); otherwise weakly, so that every block passes alpha.
"""

from __future__ import annotations

import math
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "flashprefillv2-mlx_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

import fpv2  # noqa: E402
from fpv2.kernel import compact_block_indices, sparse_attention  # noqa: E402
from fpv2.prefill_harness import (ChunkedPrefillRunner, DecoderShape,  # noqa: E402
                                  RandomDecoder)

BLOCK = 128
ALPHA = 0.1
DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _hook(name, keys, *, queries=None, heads=32, kv_heads=8, dim=128, dtype="bf16", sparse=False,
          correction=True):
    return {"name": name, "kind": "hook", "keys": keys, "queries": queries or keys, "heads": heads,
            "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "sparse": sparse,
            "correction": correction}


def _chunked(name, total, chunk, *, heads=32, kv_heads=8, dim=128, dtype="bf16", sparse=True):
    return {"name": name, "kind": "chunked", "keys": total, "chunk": chunk, "heads": heads,
            "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "sparse": sparse,
            "correction": True}


def listed():
    return [
        # the shortest prompt that the hook takes by default: launches and latency
        _hook("hook_4k", 4096),
        # a serving chunk of odd length at the end of a ragged prefix, small heads, float16
        _hook("hook_chunk_d64_f16", 9001, queries=1501, heads=16, kv_heads=2, dim=64, dtype="f16",
              sparse=True),
        # the layer at 32k tokens, every block kept
        _hook("hook_32k", 32768),
        # large heads, ragged, without the mean correction (its ablation)
        _hook("hook_20001_d256", 20001, heads=16, kv_heads=4, dim=256, correction=False),
        # the layer at 128k tokens where most blocks are pruned: what FPV2 is for
        _hook("hook_128k_sparse", 131072, sparse=True),
        # the same length with every block kept: the headline layer
        _hook("hook_128k", 131072),
        # a long prompt prefilled in 2048-token chunks over a KV cache
        _chunked("chunked_64k_sparse", 65536, 2048),
        # one GPU's share of a layer split over 8 GPUs (one KV head), chunked
        _chunked("chunked_share_32k", 32768, 2048, heads=4, kv_heads=1, sparse=False),
        # the operators one by one at their default tile, ragged query and key lengths
        {"name": "ops_15000", "kind": "ops", "keys": 15000, "heads": 32, "kv_heads": 8, "dim": 128,
         "dtype": "bf16", "sparse": True, "correction": True},
        # selection with its default configuration, which returns the raw scores
        {"name": "select_8k", "kind": "select", "keys": 8192, "heads": 32, "kv_heads": 8,
         "dim": 128, "dtype": "bf16", "sparse": True},
        # the same in float32, ragged: calibrating alpha, comparing with float32 pooling
        {"name": "select_5000_f32", "kind": "select", "keys": 5000, "heads": 8, "kv_heads": 2,
         "dim": 128, "dtype": "f32", "sparse": True},
        # the whole path of a served prompt: embeddings to the first logits
        {"name": "prefill_6k", "kind": "prefill", "tokens": 6000, "chunk": 2048, "layers": 2},
    ]


def _spread(rng, lo, hi):
    """A size spread over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


_GROUPS = [(32, 8), (32, 8), (32, 4), (16, 2), (16, 16), (8, 1), (4, 1)]


def draw(rng):
    kind = rng.choice(["hook"] * 5 + ["chunked"] * 3 + ["ops", "select", "select", "prefill"])
    heads, kv_heads = rng.choice(_GROUPS)
    dim = rng.choice([64, 96, 128, 128, 256])
    sparse = rng.random() < 0.5
    if kind == "hook":
        keys = _spread(rng, 4096, 65536)
        queries = keys if rng.random() < 0.5 else _spread(rng, 256, keys)
        case = _hook("", keys, queries=queries, heads=heads, kv_heads=kv_heads, dim=dim,
                     dtype=rng.choice(["bf16", "bf16", "f16"]), sparse=sparse,
                     correction=rng.random() < 0.75)
    elif kind == "chunked":
        total = _spread(rng, 8192, 49152)
        case = _chunked("", total, max(_spread(rng, 512, 4096), -(-total // 48)), heads=heads,
                        kv_heads=kv_heads, dim=dim, dtype=rng.choice(["bf16", "bf16", "f16"]),
                        sparse=sparse)
    elif kind == "ops":
        case = {"name": "", "kind": "ops", "keys": _spread(rng, 2048, 32768), "heads": heads,
                "kv_heads": kv_heads, "dim": dim, "dtype": rng.choice(["bf16", "f16"]),
                "sparse": sparse, "correction": rng.random() < 0.75}
    elif kind == "select":
        dtype = rng.choice(["bf16", "f16", "f32"])
        # (float32 selection is used on short contexts)
        case = {"name": "", "kind": "select", "keys": _spread(rng, 1024, 6144 if dtype == "f32" else 12288),
                "heads": heads, "kv_heads": kv_heads, "dim": dim, "dtype": dtype, "sparse": True}
    else:
        case = {"name": "", "kind": "prefill", "tokens": rng.randrange(4096, 9000),
                "chunk": rng.choice([1024, 1536, 2048]), "layers": rng.choice([1, 2])}
    del case["name"]
    return case


# ---------------------------------------------------------------------------
# What a program holds before the call
# ---------------------------------------------------------------------------


def _inputs(case, seed):
    """q [Hq, Lq, D], k and v [Hkv, Lk, D] (the queries are the last Lq positions)."""
    lk, lq = case["keys"], case.get("queries", case["keys"])
    hq, hkv, dim, dtype = case["heads"], case["kv_heads"], case["dim"], DTYPES[case["dtype"]]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    blocks = lk // BLOCK
    heavy_count = round((0.03 if lk >= 65536 else 0.06) * (blocks - 1))
    planted = 3.0 * math.sqrt(dim) if case["sparse"] else 3.0
    q = torch.empty((hq, lq, dim), dtype=dtype, device=DEVICE)
    k = torch.empty((hkv, lk, dim), dtype=dtype, device=DEVICE)
    v = torch.empty_like(k)
    group = hq // hkv
    for h in range(hkv):
        u = torch.randn(dim, generator=gen, device=DEVICE)
        u /= u.norm()
        kh = torch.randn((lk, dim), generator=gen, device=DEVICE)
        heavy = torch.randperm(blocks - 1, generator=gen, device=DEVICE)[:heavy_count] + 1
        heavy = torch.cat([torch.zeros_like(heavy[:1]), heavy])
        kh[:blocks * BLOCK].view(blocks, BLOCK, dim)[heavy] += planted * u
        k[h] = kh
        v[h] = torch.randn((lk, dim), generator=gen, device=DEVICE)
        for g in range(group):
            q[h * group + g] = torch.randn((lq, dim), generator=gen, device=DEVICE) + 0.5 * u
    return q, k, v


def _pad(x, multiple):
    """x [H, L, D] with zero rows up to a multiple."""
    n = -(-x.shape[1] // multiple) * multiple
    out = x.new_zeros((x.shape[0], n, x.shape[2]))
    out[:, :x.shape[1]] = x
    return out


def _pooled(x):
    """Block means of padded x, in float64 and in x's dtype (what a pooled tensor holds)."""
    mean = x.double().view(x.shape[0], -1, BLOCK, x.shape[2]).mean(2)
    return mean.to(x.dtype)


def _config(case):
    return fpv2.FPV2Config(alpha=ALPHA, sink_tokens=BLOCK,
                           mean_correction=case.get("correction", True))


def _decoder_shape(case):
    return DecoderShape(layers=case["layers"])


def _prompt(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed + 1)
    return torch.randint(0, _decoder_shape(case).vocab, (case["tokens"],), generator=gen,
                         device=DEVICE)


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] == "prefill":
        model = RandomDecoder(_decoder_shape(case), device=DEVICE, seed=seed)
        state["runner"] = ChunkedPrefillRunner(model, case["tokens"], config=_config(case))
        state["tokens"] = _prompt(case, seed)
        return state
    q, k, v = _inputs(case, seed)
    state["config"] = _config(case)
    state["scale"] = case["dim"] ** -0.5
    if case["kind"] == "hook":
        state["qkv"] = q[None], k[None], v[None]
    elif case["kind"] == "chunked":
        total, chunk = case["keys"], case["chunk"]
        state["chunks"] = [tuple(x[:, a:a + chunk] for x in (q, k, v))
                           for a in range(0, total, chunk)]
        state["layer"] = fpv2.ChunkedPrefill(
            case["heads"], case["kv_heads"], case["dim"], total, dtype=q.dtype, device=DEVICE,
            config=state["config"], total_tokens=total)
    elif case["kind"] == "ops":
        state["qkv"] = _pad(q, BLOCK), _pad(k, BLOCK), _pad(v, BLOCK)
        state["config"] = fpv2.FPV2Config(alpha=ALPHA, score_chunk_tiles=16,
                                          mean_correction=case["correction"])
    else:
        state["config"] = fpv2.FPV2Config(alpha=ALPHA)
        state["q"], state["pooled"] = _pad(q, BLOCK), _pooled(_pad(k, BLOCK))
    return state


# ---------------------------------------------------------------------------
# One pass
# ---------------------------------------------------------------------------


def run(state):
    case = state["case"]
    if case["kind"] == "hook":
        q, k, v = state["qkv"]
        return fpv2.fpv2_sdpa(q, k, v, scale=state["scale"], config=state["config"])
    if case["kind"] == "chunked":
        layer = state["layer"]
        layer.reset()
        return [layer.step(q, k, v) for q, k, v in state["chunks"]]
    if case["kind"] == "ops":
        q, k, v = state["qkv"]
        config, scale, n = state["config"], state["scale"], case["keys"]
        pooled_k, pooled_v = fpv2.pool_blocks(k), fpv2.pool_blocks(v)
        selected, _ = fpv2.block_scores_and_select(q, pooled_k, scale=scale, config=config,
                                                   query_length=n)
        share = fpv2.density(selected, config=config, query_length=n)
        lists = compact_block_indices(selected, config=config, query_length=n, key_length=n)
        out = sparse_attention(q, k, v, pooled_k, pooled_v, *lists, scale=scale, config=config,
                               query_length=n, key_length=n)
        return {"pooled_k": pooled_k, "selected": selected, "density": share, "ids": lists[0],
                "counts": lists[1], "pruned_ids": lists[2], "pruned_counts": lists[3], "out": out}
    if case["kind"] == "select":
        selected, scores = fpv2.block_scores_and_select(
            state["q"], state["pooled"], scale=state["scale"], config=state["config"],
            query_length=case["keys"])
        return {"selected": selected, "scores": scores}
    runner = state["runner"]
    runner.reset()
    logits = runner.prefill(state["tokens"], case["chunk"])
    # the caches are what the decode phase goes on with
    return {"logits": logits, "caches": [(c.k, c.v) for c in runner.caches]}


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------


def _attention_work(case, lq, lk):
    """One attention call of lq queries at the end of lk keys."""
    hq, hkv, dim = case["heads"], case["kv_heads"], case["dim"]
    pairs = lq * lk - lq * (lq - 1) / 2  # causal (query, key) pairs of one head
    blocks = pairs / BLOCK
    if case["sparse"]:
        # block 0, the planted blocks and the window are kept, the rest corrected
        share = 0.03 if case["keys"] >= 65536 else 0.06
        kept = min(pairs, lq * (BLOCK + 384) + share * pairs)
        pairs = kept + (blocks - kept / BLOCK if case["correction"] else 0)
    flops = 4 * dim * hq * pairs + 2 * dim * hq * blocks
    size = 4 if case["dtype"] == "f32" else 2
    return size * dim * (2 * hq * lq + 2 * hkv * lk), flops


def work(case):
    kind = case["kind"]
    if kind == "hook":
        b, f = _attention_work(case, case["queries"], case["keys"])
    elif kind == "ops":
        n = case["keys"]
        b, f = _attention_work(case, n, n)
        b += case["kv_heads"] * (n // BLOCK + 1) ** 2 * 9  # mask and lists
    elif kind == "chunked":
        b = f = 0
        for a in range(0, case["keys"], case["chunk"]):
            end = min(a + case["chunk"], case["keys"])
            cb, cf = _attention_work(case, end - a, end)
            b, f = b + cb, f + cf
    elif kind == "select":
        n, hq, hkv, dim = case["keys"], case["heads"], case["kv_heads"], case["dim"]
        blocks, size = -(-n // BLOCK), 4 if case["dtype"] == "f32" else 2
        b = size * dim * (hq * n + hkv * blocks) + 4 * hq * blocks * BLOCK * blocks
        f = 2 * dim * hq * blocks * BLOCK * blocks
    else:
        s, n = _decoder_shape(case), case["tokens"]
        qd, kd = s.query_heads * s.head_dim, s.kv_heads * s.head_dim
        weights = s.hidden * (2 * qd + 2 * kd + 3 * s.intermediate)
        f = s.layers * (2 * n * weights + 2 * qd * n * n) + 2 * s.vocab * s.hidden
        b = 2 * (s.layers * weights + s.vocab * s.hidden + 2 * s.layers * n * kd + n * s.hidden)
    return {"bytes": int(b), "flops": int(f)}


# ---------------------------------------------------------------------------
# The result in float64, from plain torch
# ---------------------------------------------------------------------------


def _selection64(scores, first, last, rows, tile, alpha, sink, window, dense_from):
    """Selected and pruned blocks of whole tiles of one KV head.

    scores [G, T * tile, Nb] (scaled logits), first [T] / last [T] the tiles'
    first and last absolute positions, rows [T * tile] the rows' positions
    (-1: padding), dense_from: index of the first dense tile."""
    group, _, nb = scores.shape
    tiles = first.numel()
    starts = torch.arange(nb, device=scores.device) * BLOCK
    ends = starts + BLOCK
    scored = (ends[None, :] <= last[:, None] + 1).repeat_interleave(tile, 0)
    seen = scored & (starts[None, :] <= rows[:, None]) & (rows[:, None] >= 0)
    s = scores.masked_fill(~seen[None], -math.inf).view(group, tiles, tile, nb)
    top = s.amax(dim=(0, 2, 3), keepdim=True)
    top = torch.where(top == -math.inf, torch.zeros_like(top), top)
    energy = (s - top).exp().sum(dim=(0, 2))
    passed = energy >= alpha * energy.amax(-1, keepdim=True)
    forced = (starts < sink)[None, :] | (ends[None, :] > first[:, None] - window)
    forced = forced | (torch.arange(tiles, device=scores.device) >= dense_from)[:, None]
    return (passed | forced) & (starts[None, :] <= last[:, None])


def _attention64(q, k, v, *, tile, alpha, sink, window, tail, correction, scale, with_selection=False):
    """FPV2 attention of q (the last positions of k, v) in float64."""
    hq, lq, dim = q.shape
    hkv, lk, _ = k.shape
    group, offset = hq // hkv, lk - lq
    tiles = -(-lq // tile)
    nb = -(-max(lk, offset + tiles * tile) // BLOCK)
    grid = k.new_zeros((hkv, nb * BLOCK, dim))
    grid[:, :lk] = k
    pk = _pooled(grid).double()
    grid[:, :lk] = v
    pv = _pooled(grid).double()
    out = torch.empty((hq, lq, dim), dtype=torch.float64, device=q.device)
    masks = torch.empty((hkv, tiles, nb), dtype=torch.bool, device=q.device)
    step = max(1, min(tiles, int(3e8 / (group * tile * (lk + nb)))))
    for h in range(hkv):
        kh, vh = k[h].double(), v[h].double()
        for t0 in range(0, tiles, step):
            t1 = min(tiles, t0 + step)
            a, b = t0 * tile, min(t1 * tile, lq)
            n, padded = b - a, (t1 - t0) * tile
            qt = q.new_zeros((group, padded, dim), dtype=torch.float64)
            qt[:, :n] = q[h * group:(h + 1) * group, a:b].double()
            rows = offset + a + torch.arange(padded, device=q.device)
            rows[n:] = -1
            first = offset + torch.arange(t0, t1, device=q.device) * tile
            last = torch.clamp(first + tile, max=offset + lq) - 1
            flat = qt.view(-1, dim)
            scores = (flat @ pk[h].T).view(group, padded, nb) * scale
            sel = _selection64(scores, first, last, rows, tile, alpha, sink, window,
                               max(tiles - tail, 0) - t0)
            masks[h, t0:t1] = sel
            ends = torch.clamp((torch.arange(nb, device=q.device) + 1) * BLOCK, max=lk)
            pruned = ~sel & (ends[None, :] <= first[:, None])
            per_row = sel.repeat_interleave(tile, 0)
            cols = offset + b  # keys visible to some row
            allowed = per_row.repeat_interleave(BLOCK, 1)[:, :cols]
            allowed &= torch.arange(cols, device=q.device)[None, :] <= rows[:, None]
            logits = (flat @ kh[:cols].T).view(group, padded, cols) * scale
            logits.masked_fill_(~allowed[None], -math.inf)
            if correction:
                extra = scores + math.log(BLOCK)
                extra = extra.masked_fill(~pruned.repeat_interleave(tile, 0)[None], -math.inf)
                logits = torch.cat([logits, extra], -1)
            logits = logits[:, :n]
            logits -= logits.amax(-1, keepdim=True)
            logits.exp_()
            total = logits.sum(-1, keepdim=True)
            acc = logits[..., :cols].reshape(-1, cols) @ vh[:cols]
            if correction:
                acc += logits[..., cols:].reshape(-1, nb) @ pv[h]
            out[h * group:(h + 1) * group, a:b] = acc.view(group, n, dim) / total
            del logits
    return (out, masks, pk) if with_selection else out


def _lists64(mask):
    """Padded ascending lists of a mask [Hkv, Nt, Nb]: ids, counts."""
    order = torch.argsort((~mask).to(torch.int8), dim=-1, stable=True)
    return order.to(torch.int32), mask.sum(-1, dtype=torch.int32)


def _prefill64(case, seed):
    """The decoder in float64 on the whole prompt (every block passes alpha
    with random weights, so the attention is exact causal attention)."""
    s, n = _decoder_shape(case), case["tokens"]
    gen = torch.Generator(device=DEVICE).manual_seed(seed)

    def w(*dims):
        x = torch.randn(dims, generator=gen, device=DEVICE, dtype=torch.float32) * 0.02
        return x.to(torch.bfloat16)

    qd, kd = s.query_heads * s.head_dim, s.kv_heads * s.head_dim
    embed = w(s.vocab, s.hidden)
    layers = [(w(qd + 2 * kd, s.hidden), w(s.hidden, qd), w(2 * s.intermediate, s.hidden),
               w(s.hidden, s.intermediate)) for _ in range(s.layers)]

    def norm(x):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + s.rms_eps)

    half = s.head_dim // 2
    inv = s.rope_theta ** (-torch.arange(half, device=DEVICE, dtype=torch.float64) / half)
    ang = torch.arange(n, device=DEVICE, dtype=torch.float64)[:, None] * inv
    cos, sin = ang.cos(), ang.sin()

    def rope(x):  # [H, n, D]
        a, b = x[..., :half], x[..., half:]
        return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)

    x = embed[_prompt(case, seed)].double()
    caches = []
    for qkv, o, gate_up, down in layers:
        y = norm(x) @ qkv.double().T
        heads = y.view(n, -1, s.head_dim).transpose(0, 1)
        q = rope(norm(heads[:s.query_heads]))
        k = rope(norm(heads[s.query_heads:s.query_heads + s.kv_heads]))
        v = heads[s.query_heads + s.kv_heads:]
        caches.append((k, v))
        attn = torch.empty((n, s.query_heads, s.head_dim), dtype=torch.float64, device=DEVICE)
        above = torch.ones((n, n), dtype=torch.bool, device=DEVICE).triu(1)
        for h in range(s.query_heads):
            kv = h // (s.query_heads // s.kv_heads)
            p = (q[h] @ k[kv].T) * s.head_dim ** -0.5
            p.masked_fill_(above, -math.inf)
            attn[:, h] = torch.softmax(p, -1) @ v[kv].contiguous()
        x = x + attn.view(n, qd) @ o.double().T
        gu = norm(x) @ gate_up.double().T
        g, u = gu[:, :s.intermediate], gu[:, s.intermediate:]
        x = x + (g * torch.sigmoid(g) * u) @ down.double().T
    logits = embed.double() @ norm(x[-1])
    return {"logits": logits, "caches": caches}


def exact(case, seed):
    kind = case["kind"]
    if kind == "prefill":
        return _prefill64(case, seed)
    if case["keys"] * case.get("queries", case["keys"]) > 70000 * 70000:
        return None  # too long in float64
    q, k, v = _inputs(case, seed)
    scale = case["dim"] ** -0.5
    packed = BLOCK // (case["heads"] // case["kv_heads"])  # query positions of a hook tile
    rule = {"alpha": ALPHA, "window": 384, "scale": scale,
            "correction": case.get("correction", True)}
    if kind == "hook":
        return _attention64(q, k, v, tile=packed, sink=BLOCK, tail=2, **rule)[None]
    if kind == "chunked":
        outs = []
        for a in range(0, case["keys"], case["chunk"]):
            b = min(a + case["chunk"], case["keys"])
            # below 4096 keys, or with less than one tile of queries, every block is kept
            kept = b < 4096 or b - a < packed
            outs.append(_attention64(q[:, a:b], k[:, :b], v[:, :b], tile=packed, sink=BLOCK,
                                     tail=2 if b == case["keys"] else 0,
                                     **dict(rule, alpha=0.0 if kept else ALPHA))[None])
        return outs
    n = case["keys"]
    if kind == "ops":
        out, mask, pk = _attention64(q, k, v, tile=BLOCK, sink=256, tail=2, with_selection=True,
                                     **rule)
        tiles, nb = mask.shape[1:]
        first = torch.arange(tiles, device=q.device) * BLOCK
        ends = torch.clamp((torch.arange(nb, device=q.device) + 1) * BLOCK, max=n)
        ids, counts = _lists64(mask)
        pruned_ids, pruned_counts = _lists64(~mask & (ends[None, :] <= first[:, None]))
        visible = sum((min((t + 1) * BLOCK, n) - 1) // BLOCK + 1 for t in range(tiles))
        return {"pooled_k": pk, "selected": mask,
                "density": mask.sum(dtype=torch.float64) / (visible * case["kv_heads"]),
                "ids": ids, "counts": counts, "pruned_ids": pruned_ids,
                "pruned_counts": pruned_counts, "out": _pad(out, BLOCK)}
    qp, pooled = _pad(q, BLOCK), _pooled(_pad(k, BLOCK))
    hkv, group = case["kv_heads"], case["heads"] // case["kv_heads"]
    padded, nb = qp.shape[1], pooled.shape[1]
    scores = torch.empty((hkv, group, padded, nb), dtype=torch.float64, device=q.device)
    masks = []
    first = torch.arange(padded // BLOCK, device=q.device) * BLOCK
    last = torch.clamp(first + BLOCK, max=n) - 1
    rows = torch.arange(padded, device=q.device)
    rows[n:] = -1
    for h in range(hkv):
        flat = qp[h * group:(h + 1) * group].double().reshape(-1, case["dim"])
        scores[h] = (flat @ pooled[h].double().T).view(group, padded, nb) * scale
        masks.append(_selection64(scores[h], first, last, rows, BLOCK, ALPHA, 256, 384,
                                  padded // BLOCK - 2))
    return {"selected": torch.stack(masks), "scores": scores}


def tolerance(case):
    """About four times the distance measured against ``exact``: 2.6e-3 to
    3.2e-3 for bfloat16 attention (P, Q and the output round to 8 bits),
    3e-4 for float16, 2e-7 for float32 scores, 1.1e-2 for the logits after
    two bfloat16 decoder layers.  A block whose energy is alpha times the
    largest to float32 rounding may fall to either side of the test."""
    kind = case["kind"]
    if kind == "select":
        return {"rel": 1e-6, "differ": 1e-4}
    if kind == "prefill":
        return {"rel": 4e-2}
    limit = {"rel": 1.2e-3 if case["dtype"] == "f16" else 1.2e-2}
    return dict(limit, differ=2e-3) if kind == "ops" else limit
