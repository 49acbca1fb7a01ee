"""Performance cases: the work a serving program has this package do.

A DeepSeek-style sparse-attention layer calls the package four ways, and every
case is one of them:

* ``attend``   -- ``dsa_amd.forward`` over given top-k indices, on bf16 or fp8
  cache rows, contiguous or paged, with the reference's scale or a model's own,
  with or without the W_UV projection after it;
* ``select``   -- the lightning indexer, logits and top-k;
* ``layer``    -- both, one after the other, as a decode step runs them;
* ``kv_write`` -- new cache rows written in the fp8 format.

``listed`` holds the measured cases, ``draw`` gives more of the same ranges,
``prepare``/``run`` make the inputs of a case and run one pass, ``work`` counts
what the pass cannot do without, ``exact`` computes its result in 64 bits with
plain torch, and ``tolerance`` bounds the difference of two correct results.
"""
from __future__ import annotations

import math

import torch

import dsa_amd

DEVICE = "cuda"
LATENT, ROPE, FP8_ROW, INDEX_DIM = 512, 64, 656, 128
DEFAULT_SCALE = 1.0 / 24.0
MODEL_SCALE = 192.0 ** -0.5  # a model's own (d_nope + d_rope) ** -0.5, 128 + 64
MAX_FLOPS = 2.0 * 4096 * 128 * 2048 * (576 + 512)  # the largest listed pass

ATTEND = dict(op="attend", cache="bf16", block=0, value_dim=0, model_scale=False, order="any", ragged=False)
SELECT = dict(op="select", ragged=False)
LAYER = dict(op="layer", cache="bf16", block=0, value_dim=0, model_scale=False, ragged=False)


def listed():
    """The measured cases.  ``first`` is the position of a sequence's first
    query (its keys are [0, first]); decode queries are the last of the context."""
    return [
        # One sequence being decoded, nothing batched: latency and launches.
        dict(ATTEND, name="decode_b1", batch=1, queries=1, heads=128, context=8192, topk=2048, first=8191),
        # The ordinary decode batch (the benchmark's headline shape).
        dict(ATTEND, name="decode_b8", batch=8, queries=1, heads=128, context=32768, topk=2048, first=32767),
        # A tensor-parallel slice of a draft-and-verify step: few sequences of
        # unequal length, three tokens each, an odd number of selected slots,
        # a paged cache with small blocks.
        dict(ATTEND, name="decode_ragged_paged", batch=5, queries=3, heads=48, context=10000, topk=1000, first=9997,
             block=16, model_scale=True, ragged=True, order="ascending"),
        # A serving engine's decode step on its fp8 paged cache, value projection included.
        dict(ATTEND, name="decode_b32_fp8", batch=32, queries=1, heads=128, context=32768, topk=2048, first=32767,
             cache="fp8", block=64, value_dim=128, model_scale=True, ragged=True, order="ascending"),
        # A decode step of a whole layer at large batch with one draft token:
        # the indexer picks the slots, a tensor-parallel slice attends to them.
        dict(LAYER, name="layer_decode_b64", batch=64, queries=2, heads=16, index_heads=64, context=65536,
             topk=2048, first=65534),
        # A 4096-token prefill chunk after 4096 tokens, tensor-parallel slice of 16 heads.
        dict(ATTEND, name="prefill_h16", batch=1, queries=4096, heads=16, context=8192, topk=2048, first=4096),
        # Two fresh prompts of odd length, from position 0: the first 2047
        # queries have fewer keys than slots, the rest of the row is -1.
        dict(ATTEND, name="prefill_fresh_h64", batch=2, queries=3001, heads=64, context=3001, topk=2048, first=0,
             order="ascending"),
        # The largest attention: the last 4096-token chunk of a 32k prompt, all heads.
        dict(ATTEND, name="prefill_h128", batch=1, queries=4096, heads=128, context=32768, topk=2048, first=28672),
        # A prefill chunk of a serving engine on its fp8 paged cache, value projection included.
        dict(ATTEND, name="prefill_fp8_h128", batch=1, queries=2048, heads=128, context=32768, topk=2048,
             first=30720, cache="fp8", block=64, value_dim=128, model_scale=True, order="ascending"),
        # The selector alone at an ordinary decode batch.
        dict(SELECT, name="select_decode_b8", batch=8, queries=1, index_heads=64, context=32768, topk=2048,
             first=32767),
        # The selector for the last 4096-token chunk of a 32k prompt.
        dict(SELECT, name="select_prefill", batch=1, queries=4096, index_heads=64, context=32768, topk=2048,
             first=28672),
        # A prompt's new cache rows written as fp8.
        dict(op="kv_write", name="kv_write_8k", batch=1, queries=8192, pow2=True),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    """One more case of the listed ones' ranges: decode batches of 1 to 64
    sequences with 1 to 4 tokens each and prefill chunks of up to 4096 tokens,
    16 to 128 heads, contexts of 1024 to 65536 tokens, 256 to 2048 slots."""
    op = rng.choices(["attend", "select", "layer", "kv_write"], [11, 4, 2, 3])[0]
    if op == "kv_write":
        return dict(op=op, batch=1, queries=_log_int(rng, 1, 65536), pow2=rng.random() < 0.8)
    decode = op == "layer" or rng.random() < 0.5
    if decode:
        batch, queries = _log_int(rng, 1, 64), rng.choice([1, 1, 2, 3, 4])
    else:
        batch, queries = rng.choice([1, 1, 1, 2, 3]), _log_int(rng, 8, 4096)
    context = _log_int(rng, 1024, 65536)
    topk = rng.choice([512, 1024, 2048, rng.randint(256, 2048)])
    case = dict(op=op, batch=batch, queries=queries, topk=topk, ragged=decode and rng.random() < 0.5)
    if op != "select":
        case.update(heads=rng.choice([16, 32, 48, 64, 96, 128]), cache=rng.choice(["bf16", "bf16", "fp8"]),
                    block=rng.choice([0, 0, 16, 64]), value_dim=rng.choice([0, 0, 128]),
                    model_scale=rng.random() < 0.5)
        if case["block"]:
            context -= context % case["block"]
    if op == "attend":
        case["order"] = rng.choice(["any", "ascending"])
    if op != "attend":
        case["index_heads"] = rng.choice([32, 64])
    if not decode:  # a chunk lies inside the context, at its start, its end or between
        case["queries"] = queries = min(queries, context, 4096 // batch)
    case["context"] = context
    case["first"] = context - queries if decode else rng.choice([0, rng.randint(0, context - queries),
                                                                 context - queries])
    if op != "attend":  # more keys than slots, so that there is something to select
        case["topk"] = min(topk, context // 3)
        case["first"] = context - queries
    while work(case)["flops"] > MAX_FLOPS:
        case["queries"] = max(1, case["queries"] // 2)
    return case


# ------------------------------------------------------------------ inputs

def _normal(gen, *dims):
    return torch.randn(dims, generator=gen, device=DEVICE, dtype=torch.float32)


def _normal_bf16(gen, *dims):
    """N(0, 1) in bf16, drawn in slices of the first dimension to bound the fp32 temporaries."""
    out = torch.empty(dims, device=DEVICE, dtype=torch.bfloat16)
    flat = out.view(dims[0], -1)
    step = max(1, (1 << 28) // flat.shape[1])
    for i in range(0, dims[0], step):
        flat[i:i + step] = _normal(gen, *flat[i:i + step].shape)
    return out


def _visible(case, gen):
    """Keys each query sees, int32 [B, SQ]: its position plus one; with
    ``ragged``, sequence b's context ends somewhere in the upper half."""
    row = torch.arange(case["queries"], device=DEVICE) + case["first"] + 1
    seen = row.expand(case["batch"], -1)
    if case["ragged"]:
        cut = torch.rand((case["batch"], 1), generator=gen, device=DEVICE) * (case["context"] // 2)
        seen = (seen - cut.long()).clamp_min(1)
    return seen.clamp_max(case["context"]).int().contiguous()


def _pick(seen, topk, context, ascending, gen):
    """int32 [rows, topk]: distinct slots uniform over [0, seen), -1 where a row has fewer keys."""
    ids = torch.empty((seen.numel(), topk), device=DEVICE, dtype=torch.int32)
    seen = seen.reshape(-1, 1)
    width = max(context, topk)
    columns = torch.arange(width, device=DEVICE)
    step = max(1, (1 << 27) // width)
    for i in range(0, ids.shape[0], step):
        keys = torch.rand((min(step, ids.shape[0] - i), width), generator=gen, device=DEVICE)
        keys.masked_fill_(columns >= seen[i:i + step], 2.0)
        value, slot = keys.topk(topk, dim=1, largest=False)
        slot = slot.int().masked_fill_(value > 1.0, context)
        if ascending:
            slot = slot.sort(dim=1).values
        ids[i:i + step] = slot.masked_fill_(slot == context, -1)
    return ids


def _fp8_rows(kv, k_rope, pow2=True):
    """bf16 rows as 656 bytes: 512 e4m3 codes, four fp32 scales (with ``pow2``
    the least power of two that keeps a 128-wide block within 448), 64 bf16
    rope values."""
    x = kv.float().unflatten(-1, (4, 128))
    scale = x.abs().amax(-1, keepdim=True) / 448.0
    scale = torch.where(scale > 0, scale, torch.ones_like(scale))
    if pow2:
        mantissa, exponent = torch.frexp(scale)
        scale = torch.ldexp(torch.ones_like(scale), exponent - (mantissa == 0.5).int())
    codes = (x / scale).clamp(-448.0, 448.0).to(torch.float8_e4m3fn).flatten(-2)
    return torch.cat([codes.view(torch.uint8), scale.flatten(-2).view(torch.uint8),
                      k_rope.contiguous().view(torch.uint8)], -1)


def _cache(case, gen, state):
    """The kv cache: ``kv``/``k_rope`` bf16 or ``kv`` fp8 rows, as [B, L, 1, .]
    or as a pool of blocks under a random block table."""
    batch, context, block = case["batch"], case["context"], case["block"]
    lead = (batch, context, 1)
    if block:
        per = context // block
        lead = (batch * per, block, 1)
        state["block_table"] = torch.randperm(batch * per, generator=gen,
                                              device=DEVICE).int().reshape(batch, per)
    if case["cache"] == "bf16":
        state["kv"] = _normal_bf16(gen, *lead, LATENT)
        state["k_rope"] = _normal_bf16(gen, *lead, ROPE)
        return
    rows = torch.empty((*lead, FP8_ROW), device=DEVICE, dtype=torch.uint8)
    flat = rows.view(-1, FP8_ROW)
    for i in range(0, flat.shape[0], 1 << 18):
        n = min(1 << 18, flat.shape[0] - i)
        flat[i:i + n] = _fp8_rows(_normal_bf16(gen, n, LATENT), _normal_bf16(gen, n, ROPE))
    state["kv"], state["k_rope"] = rows, None


def prepare(case, seed):
    gen = torch.Generator(device=DEVICE).manual_seed(seed)
    batch, queries = case["batch"], case["queries"]
    state = {"case": case, "block_table": None, "scale": None, "w_uv": None}
    if case["op"] == "kv_write":
        # normalised latents: channels of unlike magnitude
        gain = torch.exp(_normal(gen, LATENT))
        state["kv"] = (_normal(gen, batch, queries, 1, LATENT) * gain).bfloat16()
        state["k_rope"] = _normal_bf16(gen, batch, queries, 1, ROPE)
        return state
    state["lengths"] = _visible(case, gen)
    if case["op"] != "attend":
        heads = case["index_heads"]
        state["q_idx"] = _normal_bf16(gen, batch, queries, heads, INDEX_DIM)
        state["k_idx"] = _normal_bf16(gen, batch, case["context"], INDEX_DIM)
        state["weights"] = _normal(gen, batch, queries, heads) * 0.1
    if case["op"] != "select":
        heads = case["heads"]
        state["q"] = _normal_bf16(gen, batch, queries, heads, LATENT)
        state["q_rope"] = _normal_bf16(gen, batch, queries, heads, ROPE)
        _cache(case, gen, state)
        if case["model_scale"]:
            state["scale"] = MODEL_SCALE
        if case["value_dim"]:
            state["w_uv"] = (_normal(gen, heads, case["value_dim"], LATENT) * LATENT ** -0.5).bfloat16()
    if case["op"] == "attend":
        ids = _pick(state["lengths"], case["topk"], case["context"], case["order"] == "ascending", gen)
        state["indices"] = ids.reshape(batch, queries, 1, case["topk"])
    return state


# ------------------------------------------------------------------ one pass

def _forward(state, indices):
    options = {k: state[k] for k in ("scale", "block_table", "w_uv") if state[k] is not None}
    return dsa_amd.forward(state["q"], state["kv"], state["q_rope"], state["k_rope"], indices, **options)


def _whole_logits(case):
    """Every logit of the case is defined (each query sees the whole context)."""
    return case["queries"] == 1 and case["first"] == case["context"] - 1 and not case["ragged"]


def run(state):
    case = state["case"]
    if case["op"] == "kv_write":
        return dsa_amd.quantize_kv_fp8(state["kv"], state["k_rope"], pow2_scales=case["pow2"])
    if case["op"] == "attend":
        return _forward(state, state["indices"])
    inputs = (state["q_idx"], state["k_idx"], state["weights"], state["lengths"])
    if case["op"] == "select" and _whole_logits(case):
        logits = dsa_amd.indexer_logits(*inputs)
        return logits, dsa_amd.indexer_topk(logits, state["lengths"], case["topk"])
    indices = dsa_amd.indexer(*inputs, case["topk"])
    if case["op"] == "select":
        return indices
    return (indices, *_forward(state, indices))


# ------------------------------------------------------------------ bounds

def _seen_sums(case):
    """(keys seen, slots used) summed over the queries; ragged contexts end at three quarters on average."""
    cut = case["context"] // 4 if case["ragged"] else 0
    seen = [max(1, min(case["first"] + i + 1, case["context"]) - cut) for i in range(case["queries"])]
    return case["batch"] * sum(seen), case["batch"] * sum(min(s, case["topk"]) for s in seen)


def work(case):
    """Bytes and operations of one pass: each input that the result depends on
    read once, each output written once."""
    tokens = case["batch"] * case["queries"]
    if case["op"] == "kv_write":
        return {"bytes": tokens * (2 * (LATENT + ROPE) + FP8_ROW), "flops": 2 * tokens * LATENT}
    seen, slots = _seen_sums(case)
    nbytes = 4 * tokens * case["topk"]
    flops = 0
    if case["op"] != "attend":
        heads = case["index_heads"]
        reach = min(case["context"], case["first"] + case["queries"])
        nbytes += case["batch"] * reach * INDEX_DIM * 2 + tokens * heads * (INDEX_DIM * 2 + 4)
        flops += 2 * seen * heads * INDEX_DIM
        if _whole_logits(case):
            nbytes += 4 * seen
    if case["op"] != "select":
        heads, width = case["heads"], case["value_dim"] or LATENT
        rows = min(slots, case["batch"] * min(case["context"], case["first"] + case["queries"]))
        nbytes += rows * (FP8_ROW if case["cache"] == "fp8" else 2 * (LATENT + ROPE))
        nbytes += tokens * heads * (2 * (LATENT + ROPE) + 2 * width + 8) + 2 * heads * case["value_dim"] * LATENT
        flops += 2 * slots * heads * (2 * LATENT + ROPE) + 2 * tokens * heads * case["value_dim"] * LATENT
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["op"] == "kv_write":
        return "exact"
    if case["op"] == "select":
        # fp32 logits; a key whose logit ties the last selected one to within
        # rounding may be exchanged, which shifts the ascending row between the two
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.02}
    limits = {"rel": 1e-2, "max": 0.1}  # bf16 probabilities and results
    if case["op"] == "layer":
        limits["differ"] = 0.02
    return limits


# ------------------------------------------------------------------ 64 bits

def _physical(state, ids, first_token):
    """Rows of the flattened cache behind slots ``ids`` [n, K] of tokens from ``first_token`` on."""
    case = state["case"]
    token = torch.arange(first_token, first_token + ids.shape[0], device=DEVICE)
    seq = (token // case["queries"])[:, None]
    if state["block_table"] is None:
        return seq * case["context"] + ids
    block = case["block"]
    return state["block_table"].long()[seq, ids // block] * block + ids % block


def _rows64(state, flat_rows):
    """Cache rows as float64 [n, K, 576]."""
    kv = state["kv"].view(-1, state["kv"].shape[-1])[flat_rows]
    if state["k_rope"] is not None:
        return torch.cat([kv, state["k_rope"].view(-1, ROPE)[flat_rows]], -1).double()
    codes = kv[..., :LATENT].contiguous().view(torch.float8_e4m3fn).double()
    scale = kv[..., LATENT:LATENT + 16].contiguous().view(torch.float32).double()
    latent = codes.unflatten(-1, (4, 128)) * scale[..., None]
    return torch.cat([latent.flatten(-2), kv[..., LATENT + 16:].contiguous().view(torch.bfloat16).double()], -1)


def _attend64(state, indices):
    case = state["case"]
    batch, queries, heads = case["batch"], case["queries"], case["heads"]
    tokens = batch * queries
    q = torch.cat([state["q"], state["q_rope"]], -1).view(tokens, heads, LATENT + ROPE)
    ids = indices.view(tokens, -1).long()
    scale = DEFAULT_SCALE if state["scale"] is None else state["scale"]
    out, peak, total = [], [], []
    step = max(1, (1 << 28) // (ids.shape[1] * (LATENT + ROPE)))
    for i in range(0, tokens, step):
        part = ids[i:i + step]
        rows = _rows64(state, _physical(state, part.clamp_min(0), i))
        score = torch.bmm(q[i:i + step].double(), rows.transpose(1, 2).contiguous()) * scale
        score.masked_fill_((part < 0)[:, None, :], -math.inf)
        top = score.amax(-1, keepdim=True)
        weight = torch.exp(score - top)
        norm = weight.sum(-1, keepdim=True)
        latent = torch.bmm(weight, rows[..., :LATENT].contiguous()) / norm
        if state["w_uv"] is not None:
            w = state["w_uv"].double().transpose(1, 2).contiguous()
            latent = torch.bmm(latent.transpose(0, 1).contiguous(), w).transpose(0, 1)
        out.append(latent)
        peak.append(top.squeeze(-1))
        total.append(norm.squeeze(-1))
    shape = (batch, queries, heads, -1)
    return (torch.cat(out).reshape(shape), torch.cat(peak).view(batch, 1, queries, heads),
            torch.cat(total).view(batch, 1, queries, heads))


def _logits64(state, seq, first, last):
    """float64 logits [last - first, L] of queries [first, last) of one sequence."""
    q = state["q_idx"][seq, first:last].double()
    score = torch.matmul(q.flatten(0, 1), state["k_idx"][seq].double().t().contiguous()).clamp_min_(0)
    weights = state["weights"][seq, first:last].double()
    return torch.bmm(weights[:, None, :], score.view(*weights.shape, -1)).squeeze(1)


def _select64(state):
    case = state["case"]
    batch, queries, context, topk = case["batch"], case["queries"], case["context"], case["topk"]
    ids = torch.full((batch, queries, 1, topk), -1, device=DEVICE, dtype=torch.int32)
    logits = []
    columns = torch.arange(context, device=DEVICE)
    step = max(1, (1 << 28) // (context * case["index_heads"]))
    for seq in range(batch):
        for i in range(0, queries, step):
            last = min(i + step, queries)
            part = _logits64(state, seq, i, last)
            if _whole_logits(case):
                logits.append(part)
            unseen = columns >= state["lengths"][seq, i:last, None]
            value, slot = part.masked_fill(unseen, -math.inf).sort(dim=1, descending=True, stable=True)
            keep = min(topk, context)
            slot = slot[:, :keep].masked_fill(value[:, :keep] == -math.inf, context).sort(dim=1).values
            ids[seq, i:last, 0, :keep] = slot.masked_fill(slot == context, -1).int()
    if _whole_logits(case):
        return torch.stack(logits).view(batch, queries, context), ids
    return ids


def exact(case, seed):
    state = prepare(case, seed)
    if case["op"] == "kv_write":
        return _fp8_rows(state["kv"], state["k_rope"], case["pow2"])
    if case["op"] == "attend":
        return _attend64(state, state["indices"])
    picked = _select64(state)
    if case["op"] == "select":
        return picked
    ids = picked[1] if isinstance(picked, tuple) else picked
    return (ids, *_attend64(state, ids))
