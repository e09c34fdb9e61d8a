"""The calls whose speed matters to a user of this package, as measurable cases.

A case is a dict of plain values; ``prepare`` makes what a serving program
holds before the call (inputs, pools, plans, captured graphs) from a seed,
``run`` makes one pass through the public entry points and returns its
outputs, ``work`` counts the bytes and operations the pass cannot do without,
``exact`` gives the outputs in 64 bits from plain torch, and ``tolerance``
says how far two correct implementations may differ.

Kinds of cases:

* ``decode``   decode attention of one layer step (``PreparedDecode``), eager
               for launches of tens of microseconds, and as a captured graph
               of several layers' launches for the small ones, as a serving
               loop issues them;
* ``score``    block scores and tier labels from attention probabilities;
* ``migrate``  a policy step's demotions and promotions;
* ``prefill``  block scores of a prompt without materialised probabilities;
* ``serve``    the batched runtime: prompts into their tiers, decode steps
               replayed as a graph, one policy step.
"""

from __future__ import annotations

import math

import torch

from paged_tierkv_amd import kernels
from paged_tierkv_amd.runtime import BatchedTieredKVRuntime, prefill_states, recency_scores
from paged_tierkv_amd.tierkv_hip import PreparedDecode

HOT, WARM, COLD = 0, 1, 2
BS = 16                    # tokens per block, in every configuration of this package
RECENT = 8                 # most recent blocks, always HOT beside block 0
DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}


def _decode(name, batch, ctx, heads, kv_heads, head_dim, hot, warm, fmt="absmax_i8", cold="masked", dtype="fp16",
            scores=False, det=False, ragged=False, layers=1):
    return dict(name=name, kind="decode", batch=batch, ctx=ctx, heads=heads, kv_heads=kv_heads, head_dim=head_dim,
                hot=hot, warm=warm, fmt=fmt, cold=cold, dtype=dtype, scores=scores, det=det, ragged=ragged,
                layers=layers)


def listed():
    return [
        # One short conversation on a small model (TinyLlama's attention, 512
        # tokens): launch and round-trip latency; captured, as a decode loop is.
        _decode("decode_tiny_b1_512", 1, 512, 32, 4, 64, 0.25, 0.5, layers=8),
        # The headline batch: Llama-3-8B attention, 32 sequences of 4096.
        _decode("decode_b32_4k", 32, 4096, 32, 8, 128, 0.10, 0.60),
        # The batched runtime's decode step at 2304 tokens (its tier fractions
        # and its reproducible hand-out; replayed, as its decode loop does).
        _decode("decode_b16_2304_det", 16, 2304, 32, 8, 128, 0.15, 0.55, det=True, layers=4),
        # An odd, ragged batch in the reference's WARM format and COLD rule
        # with a bf16 model of 64-wide heads.
        _decode("decode_b7_ragged_ref_bf16", 7, 3001, 32, 4, 64, 0.2, 0.5, fmt="ref_u8", cold="zero_logit",
                dtype="bf16", ragged=True, layers=8),
        # A policy step over long contexts: the same launch with score sums.
        _decode("decode_scores_b4_32k", 4, 32768, 32, 8, 128, 0.05, 0.45, scores=True),
        # A large batch in the reference's WARM format: the biggest launch.
        _decode("decode_b128_8k_ref", 128, 8192, 32, 8, 128, 0.10, 0.60, fmt="ref_u8", cold="zero_logit"),
        # Block scores and tier labels of a policy step from probabilities.
        dict(name="score_labels_b32_4k", kind="score", batch=32, heads=32, tokens=4096, hot=0.10, warm=0.60),
        # A small policy step's migrations (a few dozen blocks), and a large
        # one's (half of a 4096-block pool each way) in the other format.
        dict(name="migrate_48", kind="migrate", blocks=48, kv_heads=8, head_dim=128, fmt="absmax_i8"),
        dict(name="migrate_2048_ref", kind="migrate", blocks=2048, kv_heads=8, head_dim=128, fmt="ref_u8"),
        # Prompt block scores: a batch of 2048-token prompts, and an odd small
        # batch of a bf16 model with 64-wide heads.
        dict(name="prefill_scores_b16_2k", kind="prefill", batch=16, tokens=2048, heads=32, kv_heads=8, head_dim=128,
             dtype="fp16"),
        dict(name="prefill_scores_b3_1001_bf16", kind="prefill", batch=3, tokens=1001, heads=32, kv_heads=4,
             head_dim=64, dtype="bf16"),
        # A batch served by the runtime: prompts tiered into the pools, one
        # policy interval of decode steps, the policy step.
        dict(name="serve_b16_2k", kind="serve", batch=16, prompt=2048, steps=64, layers=4, heads=32, kv_heads=8,
             head_dim=128, hot=0.15, warm=0.55, fmt="absmax_i8"),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 6 + ["score", "migrate", "prefill", "prefill", "serve"])
    if kind == "decode":
        head_dim = rng.choice([64, 128, 128])
        kv_heads = rng.choice([2, 4, 8, 8])
        group = rng.choice([1, 4, 4, 8])
        ctx = _log(rng, 130, 32768)
        batch = min(_log(rng, 1, 128), max(1, (128 * 8192) // ctx))
        hot = rng.uniform(0.04, 0.3)
        tokens = batch * ctx
        return {k: v for k, v in _decode(
            "", batch, ctx, kv_heads * group, kv_heads, head_dim, round(hot, 3), round(rng.uniform(0.4, 0.65), 3),
            fmt=rng.choice(["absmax_i8", "ref_u8"]), cold=rng.choice(["masked", "zero_logit"]),
            dtype=rng.choice(["fp16", "fp16", "bf16"]), scores=rng.random() < 0.25, det=rng.random() < 0.3,
            ragged=rng.random() < 0.4, layers=8 if tokens <= 24000 else 4 if tokens <= 48000 else 1).items() if k != "name"}
    if kind == "score":
        blocks = _log(rng, 8, 512)
        return dict(kind="score", batch=min(_log(rng, 1, 64), 8192 // blocks), heads=rng.choice([8, 16, 32, 32]),
                    tokens=blocks * BS, hot=round(rng.uniform(0.05, 0.3), 3), warm=round(rng.uniform(0.4, 0.65), 3))
    if kind == "migrate":
        return dict(kind="migrate", blocks=_log(rng, 5, 2048), kv_heads=rng.choice([4, 8]),
                    head_dim=rng.choice([64, 128]), fmt=rng.choice(["absmax_i8", "ref_u8"]))
    if kind == "prefill":
        tokens = _log(rng, 100, 8192)
        batch = min(_log(rng, 1, 16), max(1, (16 * 2048 * 2048) // (tokens * tokens)))
        kv_heads, group = rng.choice([(8, 1), (4, 4), (8, 4), (8, 4), (4, 8)])
        return dict(kind="prefill", batch=batch, tokens=tokens, heads=kv_heads * group, kv_heads=kv_heads,
                    head_dim=rng.choice([64, 128]), dtype=rng.choice(["fp16", "bf16"]))
    return dict(kind="serve", batch=_log(rng, 1, 16), prompt=_log(rng, 60, 2048), steps=rng.choice([16, 32, 64]),
                layers=2, heads=32, kv_heads=rng.choice([4, 8]), head_dim=rng.choice([64, 128]),
                hot=round(rng.uniform(0.1, 0.25), 3), warm=round(rng.uniform(0.4, 0.6), 3),
                fmt=rng.choice(["absmax_i8", "ref_u8"]))


# -- inputs -------------------------------------------------------------------


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn(gen, shape, dtype=torch.float16):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32).to(dtype)


def _quant_absmax(x):
    """fp16 tiles [S, H, bs, D] -> int8 codes and fp32 scales [S, H]."""
    f = x.float()
    s = f.abs().amax(dim=(2, 3)) / 127.0
    q = torch.round(f / torch.where(s == 0, torch.ones_like(s), s)[:, :, None, None]).clamp_(-127, 127)
    return q.to(torch.int8), s


def _quant_ref(x):
    """fp16 tiles -> uint8 codes, fp16 scale and zero point per token, in the
    half-precision op sequence of the reference codec."""
    mn, mx = x.amin(-1, keepdim=True), x.amax(-1, keepdim=True)
    s = (mx - mn) / 255.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    z = -torch.round(mn / s)
    q = (torch.round(x / s) + z).clamp_(0, 255)
    return q.to(torch.uint8), s, z


def _quant(x, fmt):
    """Codes, scale, zero of fp16 tiles, quantized in slices (bounded memory)."""
    parts = [(_quant_absmax(c) + (None,)) if fmt == "absmax_i8" else _quant_ref(c) for c in x.split(4096)]
    q, s = (torch.cat([p[i] for p in parts]) for i in (0, 1))
    return q, s, (None if fmt == "absmax_i8" else torch.cat([p[2] for p in parts]))


def _decode_inputs(c, seed):
    """Tables, pools and query of one layer's decode launch."""
    gen = _gen(seed)
    B, kv, D = c["batch"], c["kv_heads"], c["head_dim"]
    nb = -(-c["ctx"] // BS)
    if c["ragged"]:
        toks = torch.randint(max(1, c["ctx"] // 3), c["ctx"] + 1, (B,), generator=gen, device="cuda")
    else:
        toks = torch.full((B,), c["ctx"], device="cuda")
    nblk = (toks + BS - 1) // BS
    idx = torch.arange(nb, device="cuda")[None]
    lengths = (toks[:, None] - idx * BS).clamp(0, BS).to(torch.int32)
    # Block 0 and the most recent blocks HOT, the others shuffled into tiers.
    key = torch.rand((B, nb), generator=gen, device="cuda")
    key = torch.where((idx == 0) | (idx >= nblk[:, None] - RECENT), key + 2.0, key)
    key = torch.where(idx < nblk[:, None], key, key - 8.0)
    rank = key.argsort(dim=1, descending=True).argsort(dim=1)
    n_hot = torch.maximum((nblk * c["hot"]).round(), torch.minimum(nblk, torch.full_like(nblk, RECENT + 1)))
    n_warm = (nblk * c["warm"]).round()
    states = torch.where(rank < n_hot[:, None], HOT, torch.where(rank < (n_hot + n_warm)[:, None], WARM, COLD))
    states = torch.where(idx < nblk[:, None], states, COLD).to(torch.int32)
    table = torch.full((B, nb), -1, dtype=torch.int32, device="cuda")
    pools = []
    for tier in (HOT, WARM):
        at = (states == tier).nonzero()
        n = max(1, at.shape[0])
        slot = torch.randperm(n, generator=gen, device="cuda")[: at.shape[0]]
        table[at[:, 0], at[:, 1]] = slot.to(torch.int32)
        k, v = (_randn(gen, (n, kv, BS, D)) for _ in range(2))
        first = slot[at[:, 1] == 0]              # attention sinks: the first four tokens are large
        heavy = slot[torch.rand(at.shape[0], generator=gen, device="cuda") < 0.02]
        for t in (k, v):
            t[first, :, :4] *= 4.0
            t[heavy] *= 2.0
        pools.append((k, v))
    (hk, hv), (wk, wv) = pools
    wk, ks, kz = _quant(wk, c["fmt"])
    wv, vs, vz = _quant(wv, c["fmt"])
    q = _randn(gen, (B, c["heads"], 1, D)).to(DTYPES[c["dtype"]])
    return dict(query=q, table=table, states=states, lengths=lengths, hot_k=hk, hot_v=hv, warm_k=wk, warm_v=wv,
                k_scale=ks, k_zero=kz, v_scale=vs, v_zero=vz, num_blocks=nb,
                nblk=nblk.to(torch.int32) if c["ragged"] else None)


def _score_inputs(c, seed):
    gen = _gen(seed)
    logits = torch.randn((c["batch"], c["heads"], c["tokens"]), generator=gen, device="cuda") * 3.0
    probs = torch.softmax(logits, dim=-1)
    n = c["tokens"] // BS
    states = torch.randint(0, 10, (c["batch"], n), generator=gen, device="cuda")
    states = torch.where(states < 2, HOT, torch.where(states < 8, WARM, COLD)).to(torch.int32)
    return probs, states


def _migrate_inputs(c, seed):
    """A HOT pool (first half demoted, second half the promotions' targets) and
    a WARM pool (first half the demotions' targets, second half promoted)."""
    gen = _gen(seed)
    n, shape = c["blocks"], (c["blocks"], c["kv_heads"], BS, c["head_dim"])
    src_k, src_v, wk, wv = (_randn(gen, shape) for _ in range(4))
    order = [torch.randperm(n, generator=gen, device="cuda").to(torch.int32) for _ in range(4)]
    lengths = torch.full((n,), BS, dtype=torch.int32, device="cuda")
    lengths[torch.rand((n,), generator=gen, device="cuda") < 0.02] = 7   # open blocks, partly filled
    return src_k, src_v, wk, wv, order, lengths


def _prefill_inputs(c, seed):
    gen = _gen(seed)
    dt = DTYPES[c["dtype"]]
    # As the projections leave them: [batch, tokens, heads, head_dim] in memory.
    q = _randn(gen, (c["batch"], c["tokens"], c["heads"], c["head_dim"]), dt).transpose(1, 2)
    k = _randn(gen, (c["batch"], c["tokens"], c["kv_heads"], c["head_dim"]), dt).transpose(1, 2)
    return q, k


def _serve_inputs(c, seed):
    gen = _gen(seed)
    B, kv, D = c["batch"], c["kv_heads"], c["head_dim"]
    layers = []
    for _ in range(c["layers"]):
        pk, pv = (_randn(gen, (B, kv, c["prompt"], D)) for _ in range(2))
        q = _randn(gen, (B, c["heads"], 1, D))
        k, v = (_randn(gen, (B, kv, 1, D)) for _ in range(2))
        layers.append((pk, pv, q, k, v))
    ang = c["prompt"] * 10000.0 ** (-torch.arange(0, D, 2, device="cuda").double() / D)
    ang = torch.cat([ang, ang])[None, None]
    return layers, (ang.cos().half(), ang.sin().half())


# -- state and passes ---------------------------------------------------------


def prepare(case, seed):
    return _PREPARE[case["kind"]](case, seed)


def _prepare_decode(c, seed):
    plans = []
    for layer in range(c["layers"]):
        i = _decode_inputs(c, seed * 64 + layer)
        plans.append(PreparedDecode(
            i["query"], i["table"], i["states"], i["lengths"], i["hot_k"], i["hot_v"], i["warm_k"], i["warm_v"],
            i["k_scale"], i["k_zero"], i["v_scale"], i["v_zero"], i["num_blocks"], c["heads"] // c["kv_heads"],
            c["head_dim"] ** -0.5, return_scores=c["scores"], cold_mode=c["cold"], seq_num_blocks=i["nblk"],
            deterministic=c["det"]))
    state = dict(case=c, plans=plans, graph=None)
    if c["layers"] > 1:
        for p in plans:
            p.launch()
        torch.cuda.synchronize()
        state["graph"] = torch.cuda.CUDAGraph()
        with torch.cuda.graph(state["graph"]):
            for p in plans:
                p.launch()
    return state


def _run_decode(s):
    if s["graph"] is not None:
        s["graph"].replay()
    else:
        for p in s["plans"]:
            p.launch()
    return [(p.out, p.score_sums) if s["case"]["scores"] else p.out for p in s["plans"]]


def _prepare_score(c, seed):
    probs, states = _score_inputs(c, seed)
    n = c["tokens"] // BS
    return dict(case=c, probs=probs, states=states, hot=max(2, round(n * c["hot"])), warm=round(n * c["warm"]))


def _run_score(s):
    mass = kernels.block_mass_from_probs(s["probs"], BS)
    return mass, kernels.tier_labels(mass, s["states"], s["hot"], s["warm"], mode="hot_warm_cold")


def _prepare_migrate(c, seed):
    src_k, src_v, wk, wv, order, lengths = _migrate_inputs(c, seed)
    n = c["blocks"]
    hot = [torch.cat([x, torch.zeros_like(x)]) for x in (src_k, src_v)]
    warm, scale, zero = [], [], []
    for x in (wk, wv):
        q, s, z = _quant(x, c["fmt"])
        warm.append(torch.cat([torch.zeros_like(q), q]))
        scale.append(torch.cat([torch.zeros_like(s), s]))
        zero.append(None if z is None else torch.cat([torch.zeros_like(z), z]))
    table = torch.cat([order[0], n + order[2]])[None].contiguous()
    states = torch.cat([torch.full((n,), HOT), torch.full((n,), WARM)]).to(torch.int32).cuda()[None].contiguous()
    pos = torch.arange(2 * n, dtype=torch.int32, device="cuda")
    return dict(case=c, hot=hot, warm=warm, scale=scale, zero=zero, table=table, states=states, lengths=lengths,
                dem=(order[0], order[1], pos[:n]), pro=(n + order[2], n + order[3], pos[n:]))


def _run_migrate(s):
    fmt, (hk, hv), (wk, wv), (ks, vs), (kz, vz) = s["case"]["fmt"], s["hot"], s["warm"], s["scale"], s["zero"]
    src, dst, pos = s["dem"]
    kernels.demote_to_warm(hk, hv, src, dst, s["lengths"], wk, wv, ks, kz, vs, vz, warm_format=fmt, pad_tail=True,
                           block_table=s["table"], block_states=s["states"], table_pos=pos)
    src, dst, pos = s["pro"]
    kernels.promote_to_hot(wk, wv, ks, kz, vs, vz, src, dst, s["lengths"], hk, hv, warm_format=fmt,
                           block_table=s["table"], block_states=s["states"], table_pos=pos)
    return [wk, wv, ks, vs] + ([] if kz is None else [kz, vz]) + [hk, hv, s["table"], s["states"]]


def _prepare_prefill(c, seed):
    q, k = _prefill_inputs(c, seed)
    return dict(case=c, q=q, k=k)


def _run_prefill(s):
    return kernels.prefill_block_mass(s["q"], s["k"], BS, s["case"]["head_dim"] ** -0.5)


def _prepare_serve(c, seed):
    layers, rope = _serve_inputs(c, seed)
    rt = BatchedTieredKVRuntime(c["layers"], c["batch"], c["kv_heads"], c["head_dim"], c["prompt"] + c["steps"] + BS,
                                block_size=BS, hot_fraction=c["hot"], warm_fraction=c["warm"],
                                policy_interval=c["steps"], warm_format=c["fmt"], device="cuda:0")
    rt.fixed_launch_bound = True
    rt.reserve_decode_workspace(c["heads"])
    state = dict(case=c, rt=rt, layers=layers, rope=rope, graph=None)
    # One eager step loads every kernel; the next one is captured.
    _serve_prompts(state)
    _serve_step(state)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        state["outs"] = _serve_step(state)
    state["graph"] = graph
    rt.decode_step = 0
    return state


def _serve_prompts(s):
    for i, (pk, pv, _, _, _) in enumerate(s["layers"]):
        s["rt"].prefill_layer(i, pk, pv)


def _serve_step(s, policy=False):
    rt, c = s["rt"], s["case"]
    return [rt.decode_layer(i, q, k, v, c["heads"] // c["kv_heads"], c["head_dim"] ** -0.5, policy_step=policy,
                            rope=s["rope"]) for i, (_, _, q, k, v) in enumerate(s["layers"])]


def _run_serve(s):
    """Prompts, then a policy interval of decode steps: the first eagerly, the
    others replayed, the policy step (the last) eagerly."""
    rt, c = s["rt"], s["case"]
    _serve_prompts(s)
    first = last = None
    for step in range(c["steps"]):
        rt.begin_forward(1)
        if rt.policy_tick_this_forward or step == 0:
            last = _serve_step(s, policy=rt.policy_tick_this_forward)
            first = first or last
        else:
            for layer in range(rt.num_layers):
                rt._advance_blocks(layer, 1)
            s["graph"].replay()
        rt.finish_forward()
    return first, last, [torch.stack([st.table, st.states, st.lengths]) for st in rt.layers]


_PREPARE = {"decode": _prepare_decode, "score": _prepare_score, "migrate": _prepare_migrate,
            "prefill": _prepare_prefill, "serve": _prepare_serve}
_RUN = {"decode": _run_decode, "score": _run_score, "migrate": _run_migrate, "prefill": _run_prefill,
        "serve": _run_serve}


def run(state):
    return _RUN[state["case"]["kind"]](state)


# -- work and tolerance -------------------------------------------------------


def _tier_bytes(n_hot, n_warm, kv, D, fmt):
    meta = 2 * kv * 4 if fmt == "absmax_i8" else 2 * 2 * kv * BS * 2
    return n_hot * 2 * kv * BS * D * 2 + n_warm * (2 * kv * BS * D + meta)


def work(case):
    c, kind = case, case["kind"]
    if kind == "score":
        n = c["batch"] * c["tokens"] // BS
        return {"bytes": c["batch"] * c["heads"] * c["tokens"] * 4 + n * 12, "flops": c["batch"] * c["heads"] * c["tokens"]}
    if kind == "migrate":
        return {"bytes": _tier_bytes(2 * c["blocks"], 2 * c["blocks"], c["kv_heads"], c["head_dim"], c["fmt"]) +
                2 * c["blocks"] * 24, "flops": 0}
    if kind == "prefill":
        B, T, D = c["batch"], c["tokens"], c["head_dim"]
        return {"bytes": B * T * (c["heads"] + c["kv_heads"]) * D * 2 + B * -(-T // BS) * 4,
                "flops": B * c["heads"] * T * (T + 1) * D}
    B, kv, D, H = c["batch"], c["kv_heads"], c["head_dim"], c["heads"]
    if kind == "decode":
        nb = -(-c["ctx"] // BS) * (2.0 / 3.0 if c["ragged"] else 1.0)
        n_hot, n_warm = max(RECENT + 1, nb * c["hot"]), nb * c["warm"]
        one = B * (_tier_bytes(n_hot, n_warm, kv, D, c["fmt"]) + nb * 12 + 2 * H * D * 2 + (H * nb * 4 if c["scores"] else 0))
        return {"bytes": c["layers"] * one, "flops": c["layers"] * B * H * (n_hot + n_warm) * BS * D * 4}
    # serve: the prompt's resident tokens read and written once, then each
    # step's decode over the growing row (half of the interval on average).
    nb = -(-c["prompt"] // BS)
    n_hot, n_warm = max(2, nb * c["hot"]), nb * c["warm"]
    step = _tier_bytes(n_hot + c["steps"] / BS / 2, n_warm, kv, D, c["fmt"]) + nb * 12 + 2 * H * D * 2 + 8 * kv * D
    prompt = (n_hot + n_warm) * 2 * kv * BS * D * 2 + _tier_bytes(n_hot, n_warm, kv, D, c["fmt"]) + nb * 12
    return {"bytes": c["layers"] * B * (prompt + c["steps"] * step),
            "flops": c["layers"] * c["steps"] * B * H * (n_hot + n_warm) * BS * D * 4}


def tolerance(case):
    kind = case["kind"]
    if kind == "decode":
        # Probabilities enter the product in fp16, outputs are rounded to the
        # query's type; score sums are sums of 32-bit probabilities.
        return {"rel": 4e-3 if case["dtype"] == "bf16" else 1e-3}
    if kind == "score":
        return {"rel": 2e-6, "differ": 2e-3}      # 32-bit sums; labels may differ where two scores tie
    if kind == "prefill":
        return {"rel": 4e-6}                      # 32-bit logits, exponentials and sums
    if kind == "migrate":
        return "exact"
    return {"rel": 1.5e-3, "differ": 5e-3}        # as decode; a tie in the policy step moves two blocks


# -- 64-bit outputs -----------------------------------------------------------


def exact(case, seed):
    return _EXACT[case["kind"]](case, seed)


def _dequant(q, s, z, fmt):
    if fmt == "absmax_i8":
        return q.double() * s.double()[..., None, None]
    return (q.double() - z.double()) * s.double()


def _attend(q, k, v, ok, cold, scale):
    """q [H, D], k / v [kv, T, D], ok [T]: softmax attention over the valid
    tokens and ``cold`` further tokens of logit 0 and value 0."""
    H, (kv, _, D) = q.shape[0], k.shape
    x = (q.double().view(kv, H // kv, D) @ k.transpose(1, 2).contiguous()) * scale
    x = x.masked_fill(~ok, float("-inf"))
    m = x.amax(-1, keepdim=True)
    if cold:
        m = m.clamp_min(0.0)
    e = torch.exp(x - m)
    tail = torch.exp(-m) * cold
    p = e / (e.sum(-1, keepdim=True) + tail)
    return (p @ v).view(H, D), p.view(H, -1), (torch.exp(-m) / (e.sum(-1, keepdim=True) + tail)).view(H)


def _exact_decode_layer(c, i):
    outs, sums = [], []
    D, kv = c["head_dim"], c["kv_heads"]
    for b in range(c["batch"]):
        st, ln, tb = i["states"][b], i["lengths"][b], i["table"][b].long()
        hot, warm = (st == HOT).nonzero()[:, 0], (st == WARM).nonzero()[:, 0]
        ids = torch.cat([hot, warm])
        sel = lambda t: None if t is None else t[tb[warm]]  # noqa: E731
        kk = torch.cat([i["hot_k"][tb[hot]].double(), _dequant(sel(i["warm_k"]), sel(i["k_scale"]), sel(i["k_zero"]), c["fmt"])])
        vv = torch.cat([i["hot_v"][tb[hot]].double(), _dequant(sel(i["warm_v"]), sel(i["v_scale"]), sel(i["v_zero"]), c["fmt"])])
        kk, vv = (t.transpose(0, 1).reshape(kv, -1, D) for t in (kk, vv))
        ok = (torch.arange(BS, device="cuda")[None] < ln[ids][:, None]).reshape(-1)
        cold_len = torch.where(st == COLD, ln, 0)
        cold = int(cold_len.sum()) if c["cold"] == "zero_logit" else 0
        o, p, cold_p = _attend(i["query"][b, :, 0], kk, vv, ok, cold, D ** -0.5)
        outs.append(o[None])
        row = torch.zeros((c["heads"], i["num_blocks"]), dtype=torch.float64, device="cuda")
        row[:, ids] = p.view(c["heads"], -1, BS).sum(-1)
        if cold:
            row += cold_p[:, None] * cold_len
        sums.append(row)
    out = torch.stack(outs)
    return (out, torch.stack(sums)) if c["scores"] else out


def _exact_decode(c, seed):
    return [_exact_decode_layer(c, _decode_inputs(c, seed * 64 + layer)) for layer in range(c["layers"])]


def _exact_score(c, seed):
    probs, _ = _score_inputs(c, seed)
    return probs.double().view(c["batch"], c["heads"], -1, BS).sum((1, 3)) / c["heads"] / BS, None


def _exact_migrate(c, seed):
    src_k, src_v, wk, wv, order, lengths = _migrate_inputs(c, seed)
    n, ln = c["blocks"], lengths.long()
    valid = (torch.arange(BS, device="cuda")[None] < ln[:, None])[:, None, :, None]
    hot, scales = [], []
    for src, warm in ((src_k, wk), (src_v, wv)):
        q, s, z = _quant(warm, c["fmt"])
        got = torch.zeros((n,) + tuple(src.shape[1:]), dtype=torch.float64, device="cuda")
        got[order[3].long()] = _dequant(q, s, z, c["fmt"])[order[2].long()] * valid
        hot.append(torch.cat([src.double(), got]))
        x = src[order[0].long()].double()
        if c["fmt"] == "absmax_i8":
            new = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
            new[order[1].long()] = (x.abs() * valid).amax((2, 3)) / 127.0
            scales.append(torch.cat([new, s.double()]))
        else:
            step = torch.where(valid, (x.amax(-1, keepdim=True) - x.amin(-1, keepdim=True)) / 255.0, 1.0)
            new = torch.zeros(s.shape, dtype=torch.float64, device="cuda")
            new[order[1].long()] = step
            scales.append(torch.cat([new, s.double()]))
    codes = [None, None]
    zeros = [] if c["fmt"] == "absmax_i8" else [None, None]
    return codes + scales + zeros + hot + [None, None]


def _exact_prefill(c, seed):
    q, k = _prefill_inputs(c, seed)
    B, H, T, D = q.shape
    G = H // k.shape[1]
    nblk = -(-T // BS)
    out = torch.zeros((B, nblk * BS), dtype=torch.float64, device="cuda")
    for b in range(B):
        for h in range(k.shape[1]):
            kk = k[b, h].double().t().contiguous()
            for t0 in range(0, T, 2048):
                qq = q[b, h * G:(h + 1) * G, t0:t0 + 2048].double()
                x = (qq.reshape(-1, D) @ kk).view(G, -1, T) * D ** -0.5
                later = torch.arange(T, device="cuda")[None] > torch.arange(t0, t0 + qq.shape[1], device="cuda")[:, None]
                out[b, :T] += torch.softmax(x.masked_fill_(later, float("-inf")), dim=-1).sum((0, 1))
    size = (T - torch.arange(nblk, device="cuda") * BS).clamp_max(BS)
    return out.view(B, nblk, BS).sum(-1) / (H * T) / size


def _exact_serve(c, seed):
    """The first decode step's outputs; the rest depends on ranks of rounded scores."""
    layers, (cos, sin) = _serve_inputs(c, seed)
    nb = -(-c["prompt"] // BS)
    tiers = torch.tensor(prefill_states(nb, recency_scores(nb), max(2, round(c["hot"] * nb)), round(c["warm"] * nb),
                                        "hot_warm_cold"), device="cuda")

    def rotate(x):
        half = torch.cat([-x[..., c["head_dim"] // 2:], x[..., : c["head_dim"] // 2]], dim=-1)
        return (x * cos + half * sin).double()

    first = []
    for pk, pv, q, k, v in layers:
        B, kv, T, D = pk.shape
        pad = torch.nn.functional.pad
        kt, vt = (pad(t, (0, 0, 0, nb * BS - T)).view(B, kv, nb, BS, D).transpose(1, 2) for t in (pk, pv))
        both = []
        for t in (kt, vt):
            codes = _quant(t.reshape(B * nb, kv, BS, D), c["fmt"])
            deq = _dequant(*codes, c["fmt"]).view(B, nb, kv, BS, D)
            x = torch.where((tiers == WARM)[None, :, None, None, None], deq, t.double())
            both.append(x.transpose(1, 2).reshape(B, kv, nb * BS, D))
        ok = (tiers != COLD).repeat_interleave(BS) & (torch.arange(nb * BS, device="cuda") < T)
        ok = torch.cat([ok, torch.ones(1, dtype=torch.bool, device="cuda")])
        kk, vv = (torch.cat([x, new], dim=2) for x, new in zip(both, (rotate(k), v.double())))
        qr = rotate(q)
        first.append(torch.stack([_attend(qr[b, :, 0], kk[b], vv[b], ok, 0, D ** -0.5)[0][None] for b in range(B)]))
    return first, [None] * len(layers), [None] * len(layers)


_EXACT = {"decode": _exact_decode, "score": _exact_score, "migrate": _exact_migrate, "prefill": _exact_prefill,
          "serve": _exact_serve}
