"""Workloads of the paged KV path, as the programs that use it call it.

A case is one pass through public entry points of kavor_amd on inputs that are resident
on the GPU:

  decode     one query token per sequence over paged K/V.  entry "call": paged_decode;
             "module": Attention.forward (append, then decode); "step": the one-launch
             paged_decode_fused (q/k norm, RoPE, append, decode), `layers` of them.
             captured: the program replays a graph, as the engine's decode does.
  prefill    Attention.forward on packed new tokens: append, then varlen attention, over
             the fresh k / v (no cached prefix) or over the pages (prefix-cached).
  layer_ops  the kernels beside attention: q/k norm + RoPE + append, RMSNorm, SiLU * up.
  sample     next tokens of [rows, vocab] logits: Gumbel-max above temperature 0, else
             greedy.
  model      a captured decode step of a small-depth Qwen3 with its LM head: logits.

Lengths are evenly spaced over the stated range, so that the work of a case does not
depend on the seed; their order, the page ids and all values come from the seed.
"""

from __future__ import annotations

import math
import random

import torch

from kavor_amd.engine.cache_pool import CachePool
from kavor_amd.engine.qwen3 import Qwen3ForCausalLM, Qwen3Spec
from kavor_amd.layers import fused
from kavor_amd.layers.attention import Attention, paged_decode, paged_decode_fused
from kavor_amd.utils.context import reset_context, set_context

D = 128
EPS = 1e-6
BF16 = torch.bfloat16


# ----------------------------------------------------------------------------- the cases

def _decode(name, entry, seqs, q_heads, kv_heads, ctx_min, ctx_max, layers=1, captured=False, block=256):
    return dict(name=name, kind="decode", entry=entry, seqs=seqs, q_heads=q_heads, kv_heads=kv_heads,
                ctx_min=ctx_min, ctx_max=ctx_max, layers=layers, captured=captured, block=block)


def _prefill(name, seqs, q_heads, kv_heads, new_min, new_max, prefix_min=0, prefix_max=0, share=1, block=256):
    return dict(name=name, kind="prefill", seqs=seqs, q_heads=q_heads, kv_heads=kv_heads, new_min=new_min,
                new_max=new_max, prefix_min=prefix_min, prefix_max=prefix_max, share=share, block=block)


def listed():
    return [
        # one user generating: the attention of a whole 28-layer decode step, latency only
        _decode("decode_one", "step", 1, 16, 8, 611, 611, layers=28, captured=True),
        # the tail of a batch job: a few sequences left
        _decode("decode_few", "step", 8, 16, 8, 600, 3000, layers=4, captured=True),
        # the engine's full batch through the reference's own attention module
        _decode("decode_batch", "module", 256, 16, 8, 100, 2048),
        # long contexts, four query heads per kv head
        _decode("decode_long", "call", 128, 32, 8, 1024, 32768),
        # eight query heads per kv head (a 64-head model), mid-size contexts
        _decode("decode_wide", "step", 64, 64, 8, 1000, 9000, captured=True),
        # a first batch of prompts: no cached prefix, dense k / v
        _prefill("prefill_dense", 32, 16, 8, 100, 1024),
        # prompts that share cached prefixes in groups of four
        _prefill("prefill_prefix", 32, 16, 8, 100, 1024, 0, 4096, share=4),
        # the next turns of three chats: little new text on a long cached history
        _prefill("prefill_turn", 3, 32, 8, 17, 300, 2048, 8192),
        # one token budget (16384) spent on two long prompts
        _prefill("prefill_long", 2, 32, 8, 8100, 8192),
        # the other kernels of a layer over a full prefill budget
        dict(name="layer_ops", kind="layer_ops", tokens=16384, q_heads=16, kv_heads=8, hidden=1024, inter=3072,
             captured=False),
        # a full batch's next tokens; half the rows as flat as random weights make them,
        # half peaked as a trained model's
        dict(name="sample", kind="sample", rows=256, vocab=151936, temp_min=0.6, temp_max=1.2, peaked=0.5,
             greedy=0.0),
        # whole decode steps at a middling batch, LM head included
        dict(name="model_decode", kind="model", seqs=48, layers=4, ctx_min=100, ctx_max=2048),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "decode", "prefill", "prefill", "prefill", "layer_ops", "sample"])
    q_heads, kv_heads = rng.choice([(16, 8), (16, 8), (32, 8), (40, 8), (64, 8), (8, 8)])
    block = rng.choice([256, 256, 64])
    if kind == "decode":
        entry = rng.choice(["call", "module", "step", "step"])
        captured = entry == "step"
        ctx_max = _log_int(rng, 33, 32768)
        ctx_min = max(1, int(ctx_max * rng.uniform(0.03, 1.0)))
        seqs = _log_int(rng, 1, 256)
        seqs = max(1, min(seqs, 1_000_000 // ctx_max))
        layers = max(1, min(4, 200_000 // (seqs * ctx_max))) if captured else 1
        case = _decode("", entry, seqs, q_heads, kv_heads, ctx_min, ctx_max, layers, captured, block)
    elif kind == "prefill":
        total = _log_int(rng, 16, 16000)
        seqs = min(total, rng.choice([1, 1, 2, 3, 5, 8, 13, 32]))
        new_max = max(1, min(8192, int(1.4 * total / seqs)))
        new_min = max(1, int(new_max * rng.uniform(0.1, 1.0)))
        prefix_max = 0
        if rng.random() < 0.6:
            prefix_max = max(block, _log_int(rng, 256, 32768))
        share = rng.choice([1, 1, 4]) if prefix_max else 1
        case = _prefill("", seqs, q_heads, kv_heads, new_min, new_max, prefix_max // 4, prefix_max, share, block)
        while work(case)["flops"] > 1e12:  # no more than the largest listed one
            for key in ("new_min", "new_max", "prefix_min", "prefix_max"):
                case[key] = case[key] * 3 // 4
    elif kind == "layer_ops":
        tokens = _log_int(rng, 1, 16384)
        hidden, inter = rng.choice([(1024, 3072), (2048, 6144), (4096, 12288), (5120, 17408)])
        tokens = max(1, min(tokens, 16384 * 4096 // hidden))
        case = dict(kind="layer_ops", tokens=tokens, q_heads=q_heads, kv_heads=kv_heads, hidden=hidden, inter=inter,
                    captured=tokens <= 512)
    else:
        case = dict(kind="sample", rows=_log_int(rng, 1, 384), vocab=rng.choice([151936, 151643, 32000]),
                    temp_min=round(rng.uniform(0.3, 1.0), 2), temp_max=round(rng.uniform(1.0, 1.5), 2),
                    peaked=rng.choice([0.0, 0.5, 1.0]), greedy=rng.choice([0.0, 0.0, 0.3, 1.0]))
    case.pop("name", None)
    return case


# ----------------------------------------------------------------------------- lengths

def _spaced(lo, hi, n):
    return [lo + (hi - lo) * i // max(1, n - 1) for i in range(n)] if n > 1 else [(lo + hi) // 2]


def _decode_lens(case):
    return _spaced(case["ctx_min"], case["ctx_max"], case["seqs"])


def _prefill_lens(case):
    """[(new tokens, cached tokens, group)]: whole blocks are cached, per group."""
    n, share, bs = case["seqs"], case["share"], case["block"]
    new = _spaced(case["new_min"], case["new_max"], n)
    random.Random(n).shuffle(new)
    groups = -(-n // share)
    prefix = [p // bs * bs for p in _spaced(case["prefix_min"], case["prefix_max"], groups)]
    return [(new[i], prefix[i // share], i // share) for i in range(n)]


# ----------------------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return torch.empty(*shape, dtype=BF16, device="cuda").normal_(0.0, std, generator=g)


def _ints(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _pool(g, layers, blocks, block, kv_heads):
    """Pages as the engine's pool holds them (K, then V, of one block) and their views."""
    pool = _randn(g, layers, blocks, 2 * block * kv_heads * D)
    shape = (blocks, block, kv_heads, D)
    strides = (2 * block * kv_heads * D, kv_heads * D, D, 1)
    half = block * kv_heads * D
    k = [pool[i].as_strided(shape, strides, pool[i].storage_offset()) for i in range(layers)]
    v = [pool[i].as_strided(shape, strides, pool[i].storage_offset() + half) for i in range(layers)]
    return pool, k, v


def _rope_table(positions):
    inv = 1.0 / (1_000_000.0 ** (torch.arange(0, D, 2, dtype=torch.float64, device="cuda") / D))
    f = torch.outer(torch.arange(positions, dtype=torch.float64, device="cuda"), inv)
    return torch.cat((f.cos(), f.sin()), dim=-1).float().contiguous()


def _norm_weight(g, size):
    return (1.0 + 0.1 * torch.randn(size, generator=g, device="cuda")).to(BF16)


def _pages(rng, lens, bs, spare=8):
    """A shuffled pool of page ids and each sequence's table of them."""
    need = [-(-n // bs) for n in lens]
    blocks = sum(need) + spare
    ids = list(range(blocks))
    rng.shuffle(ids)
    tables, at = [], 0
    for n in need:
        tables.append(ids[at:at + n])
        at += n
    return blocks, tables


def _table_tensor(tables):
    width = max(1, max(len(t) for t in tables))
    return _ints([t + [-1] * (width - len(t)) for t in tables])


def _decode_inputs(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    hq, hkv, bs, L = case["q_heads"], case["kv_heads"], case["block"], case["layers"]
    lens = _decode_lens(case)
    rng.shuffle(lens)
    B = len(lens)
    blocks, tables = _pages(rng, lens, bs)
    x = {"lens": lens, "tables": tables, "ctx": _ints(lens), "bt": _table_tensor(tables)}
    x["slots"] = _ints([t[(n - 1) // bs] * bs + (n - 1) % bs for t, n in zip(tables, lens)])
    x["pool"], x["k"], x["v"] = _pool(g, L, blocks, bs, hkv)
    x["qkv"] = _randn(g, L, B, (hq + 2 * hkv) * D)
    if case["entry"] == "step":
        x["qw"], x["kw"] = _norm_weight(g, D), _norm_weight(g, D)
        x["rope"] = _rope_table(max(lens))
    return x


def _prefill_inputs(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    hq, hkv, bs = case["q_heads"], case["kv_heads"], case["block"]
    seqs = _prefill_lens(case)
    rng.shuffle(seqs)
    prefixes = {grp: p for _, p, grp in seqs}
    order = sorted(prefixes)
    blocks, own = _pages(rng, [prefixes[grp] for grp in order] + [n for n, _, _ in seqs], bs)
    shared = dict(zip(order, own))
    tables = [shared[grp] + own[len(order) + i] for i, (_, _, grp) in enumerate(seqs)]
    cu_q, cu_k, slots = [0], [0], []
    for (new, pre, _), t in zip(seqs, tables):
        cu_q.append(cu_q[-1] + new)
        cu_k.append(cu_k[-1] + pre + new)
        slots += [t[p // bs] * bs + p % bs for p in range(pre, pre + new)]
    x = {"seqs": seqs, "tables": tables, "cu_q": _ints(cu_q), "cu_k": _ints(cu_k), "slots": _ints(slots),
         "bt": _table_tensor(tables) if any(p for _, p, _ in seqs) else None,
         "max_q": max(s[0] for s in seqs), "max_k": max(s[0] + s[1] for s in seqs)}
    x["pool"], x["k"], x["v"] = _pool(g, 1, blocks, bs, hkv)
    T = cu_q[-1]
    # q and k as the norm and RoPE leave them, v a view of the qkv rows
    x["q"], x["new_k"] = _randn(g, T, hq, D), _randn(g, T, hkv, D)
    x["qkv"] = _randn(g, T, (hq + 2 * hkv) * D)
    x["new_v"] = x["qkv"][:, (hq + hkv) * D:].view(T, hkv, D)
    return x


def _layer_inputs(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    T, hq, hkv = case["tokens"], case["q_heads"], case["kv_heads"]
    ids = list(range(-(-T // 256) + 4))
    rng.shuffle(ids)
    x = {"slots": _ints([ids[i // 256] * 256 + i % 256 for i in range(T)]),
         "positions": _ints([i % 4096 for i in range(T)]), "rope": _rope_table(4096)}
    x["pool"], x["k"], x["v"] = _pool(g, 1, len(ids), 256, hkv)
    x["qkv"] = _randn(g, T, (hq + 2 * hkv) * D)
    x["qw"], x["kw"], x["w"] = _norm_weight(g, D), _norm_weight(g, D), _norm_weight(g, case["hidden"])
    x["hidden"] = _randn(g, T, case["hidden"])
    x["gate_up"] = _randn(g, T, 2 * case["inter"])
    return x


def _sample_inputs(case, seed):
    g, rng = _gen(seed), random.Random(seed)
    R, V = case["rows"], case["vocab"]
    logits = torch.empty(R, -(-V // 8) * 8, device="cuda", dtype=BF16)[:, :V]
    peaked = round(case["peaked"] * R)
    flat = torch.randn(R, V, generator=g, device="cuda")
    order = list(range(R))
    rng.shuffle(order)
    for j, r in enumerate(order):  # the last `peaked` of the order have a trained model's shape
        logits[r] = (0.64 * flat[r]).to(BF16) if j < R - peaked else (2.2 * flat[r]).to(BF16)
    tops = torch.randint(0, V, (R, 40), generator=g, device="cuda")
    lift = 9.0 * torch.rand(R, 40, generator=g, device="cuda") + 8.0
    for r in order[R - peaked:]:
        logits[r, tops[r]] = lift[r].to(BF16)
    temps = torch.tensor(_spaced(0, 1000, R), dtype=torch.float32, device="cuda") / 1000
    temps = case["temp_min"] + (case["temp_max"] - case["temp_min"]) * temps
    cold = rng.sample(range(R), round(case["greedy"] * R))
    if cold:
        temps[torch.tensor(cold, device="cuda")] = 0.0
    return {"logits": logits, "temps": temps, "seed": torch.full((1,), seed % 100_000, dtype=torch.int32, device="cuda")}


def _model_spec(case):
    return Qwen3Spec(num_hidden_layers=case["layers"], max_position_embeddings=4096)


def _model_inputs(case, seed):
    """A checkpoint's tensors (Hugging Face names) and a batch in the middle of decoding."""
    g, rng = _gen(seed), random.Random(seed)
    H, I, hq, hkv, V = 1024, 3072, 16, 8, 151936
    w = {"model.embed_tokens.weight": _randn(g, V, H, std=0.02), "model.norm.weight": _norm_weight(g, H)}
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        for name, shape in (("self_attn.q_proj", (hq * D, H)), ("self_attn.k_proj", (hkv * D, H)),
                            ("self_attn.v_proj", (hkv * D, H)), ("self_attn.o_proj", (H, hq * D)),
                            ("mlp.gate_proj", (I, H)), ("mlp.up_proj", (I, H)), ("mlp.down_proj", (H, I))):
            w[p + name + ".weight"] = _randn(g, *shape, std=0.02)
        for name, size in (("self_attn.q_norm", D), ("self_attn.k_norm", D), ("input_layernorm", H),
                           ("post_attention_layernorm", H)):
            w[p + name + ".weight"] = _norm_weight(g, size)
    lens = _decode_lens(case)
    rng.shuffle(lens)
    blocks, tables = _pages(rng, lens, 256)
    return {"weights": w, "lens": lens, "tables": tables, "blocks": blocks,
            "pages": _randn(g, case["layers"], blocks, 2 * 256 * hkv * D),
            "ids": torch.randint(0, V, (len(lens),), generator=g, device="cuda", dtype=torch.int32),
            "positions": _ints([n - 1 for n in lens]), "ctx": _ints(lens), "bt": _table_tensor(tables),
            "slots": _ints([t[(n - 1) // 256] * 256 + (n - 1) % 256 for t, n in zip(tables, lens)])}


# ----------------------------------------------------------------------------- prepare and run

def _capture(step):
    """The graph a serving program replays: one eager pass, then the capture."""
    step()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        step()
    torch.cuda.synchronize()
    return graph


def _module(case, x):
    attn = Attention(case["q_heads"], D, D ** -0.5, case["kv_heads"])
    attn.k_cache[0], attn.v_cache[0] = x["k"][0], x["v"][0]
    return attn


@torch.inference_mode()
def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode":
        x = _decode_inputs(case, seed)
        hq, hkv, B = case["q_heads"], case["kv_heads"], case["seqs"]
        if case["entry"] == "step":
            out = torch.empty(case["layers"], B, hq, D, dtype=BF16, device="cuda")

            def step():
                for i in range(case["layers"]):
                    paged_decode_fused(x["qkv"][i], x["rope"], x["qw"], x["kw"], EPS, hq, hkv, x["k"][i], x["v"][i],
                                       x["slots"], x["ctx"], x["bt"], D ** -0.5, out=out[i])
                return out, x["pool"]

            return {"step": step, "outs": (out, x["pool"]), "graph": _capture(step) if case["captured"] else None}
        rows = x["qkv"][0]
        q = rows[:, :hq * D].reshape(B, hq, D)
        if case["entry"] == "call":
            return {"step": lambda: paged_decode(q, x["k"][0], x["v"][0], x["ctx"], x["bt"], D ** -0.5), "graph": None}
        k = rows[:, hq * D:(hq + hkv) * D].reshape(B, hkv, D)
        v = rows[:, (hq + hkv) * D:].view(B, hkv, D)
        attn = _module(case, x)

        def forward():
            set_context(False, slot_mapping=x["slots"], context_lens=x["ctx"], block_tables=x["bt"])
            o = attn(q, k, v)
            reset_context()
            return o, x["pool"]

        return {"step": forward, "graph": None}
    if kind == "prefill":
        x = _prefill_inputs(case, seed)
        attn = _module(case, x)

        def forward():
            set_context(True, x["cu_q"], x["cu_k"], x["max_q"], x["max_k"], x["slots"], None, x["bt"])
            o = attn(x["q"], x["new_k"], x["new_v"])
            reset_context()
            return o, x["pool"]

        return {"step": forward, "graph": None}
    if kind == "layer_ops":
        x = _layer_inputs(case, seed)
        T, hq, hkv = case["tokens"], case["q_heads"], case["kv_heads"]
        outs = None
        if case["captured"]:
            outs = [torch.empty(T, hq, D, dtype=BF16, device="cuda"), torch.empty_like(x["hidden"]),
                    torch.empty(T, case["inter"], dtype=BF16, device="cuda")]

        def ops():
            o = outs or [None] * 3
            q = fused.qk_norm_rope_append(x["qkv"], x["positions"], x["rope"], x["qw"], x["kw"], EPS, hq, hkv,
                                          x["k"][0], x["v"][0], x["slots"], q_out=o[0])
            h = fused.rms_norm(x["hidden"], x["w"], EPS, out=o[1])
            a = fused.silu_and_mul(x["gate_up"], out=o[2])
            return q, h, a, x["pool"]

        if case["captured"]:
            return {"step": ops, "outs": (*outs, x["pool"]), "graph": _capture(ops)}
        return {"step": ops, "graph": None}
    if kind == "sample":
        x = _sample_inputs(case, seed)
        if case["greedy"] == 1.0:
            return {"step": lambda: fused.greedy_argmax(x["logits"]), "graph": None}
        return {"step": lambda: fused.sample(x["logits"], x["temps"], x["seed"]), "graph": None}
    x = _model_inputs(case, seed)
    model = Qwen3ForCausalLM(_model_spec(case), torch.device("cuda"))
    model.load_hf_state(x["weights"])
    pool = CachePool(model, 8, D, 256)
    pool.allocate(x["blocks"], torch.device("cuda"))
    pool.pools.view(BF16).copy_(x["pages"])
    logits = torch.empty(case["seqs"], 151936, dtype=BF16, device="cuda")

    def step():
        set_context(False, slot_mapping=x["slots"], context_lens=x["ctx"], block_tables=x["bt"])
        model.compute_logits(model(x["ids"], x["positions"]), out=logits)
        reset_context()

    keep = {k: x[k] for k in ("ids", "positions", "slots", "ctx", "bt")}
    return {"step": step, "outs": (logits,), "graph": _capture(step), "keep": (model, pool, keep)}


@torch.inference_mode()
def run(state):
    if state["graph"] is not None:
        state["graph"].replay()
        return state["outs"]
    return state["step"]()


# ----------------------------------------------------------------------------- work and tolerance

def work(case):
    kind = case["kind"]
    if kind == "decode":
        lens = _decode_lens(case)
        hq, hkv, L = case["q_heads"], case["kv_heads"], case["layers"]
        tables = 4 * sum(2 - (-n // case["block"]) for n in lens)
        new = len(lens) * 2 * hkv * D * 2  # each sequence's own k and v
        kv, qo = sum(lens) * 2 * hkv * D * 2, 2 * len(lens) * hq * D * 2
        extra = 0 if case["entry"] == "call" else new  # read from the rows, written to the page
        return {"bytes": L * (kv + qo + extra) + tables, "flops": L * 4 * hq * D * sum(lens)}
    if kind == "prefill":
        seqs, hq, hkv = _prefill_lens(case), case["q_heads"], case["kv_heads"]
        new = sum(s[0] for s in seqs)
        cached = sum({grp: p for _, p, grp in seqs}.values())
        pairs = sum(n * p + n * (n + 1) // 2 for n, p, _ in seqs)
        return {"bytes": 2 * new * hq * D * 2 + (2 * new + cached) * 2 * hkv * D * 2, "flops": 4 * hq * D * pairs}
    if kind == "layer_ops":
        T, hq, hkv = case["tokens"], case["q_heads"], case["kv_heads"]
        return {"bytes": T * 2 * (2 * (hq + 2 * hkv) * D + 2 * case["hidden"] + 3 * case["inter"]),
                "flops": T * (10 * (hq + hkv) * D + 4 * case["hidden"] + 6 * case["inter"])}
    if kind == "sample":
        return {"bytes": case["rows"] * (2 * case["vocab"] + 12), "flops": 2 * case["rows"] * case["vocab"]}
    lens, H, I, V, hq, hkv = _decode_lens(case), 1024, 3072, 151936, 16, 8
    weights = case["layers"] * (H * (hq + 2 * hkv) * D + hq * D * H + 3 * H * I) + V * H
    kv = case["layers"] * sum(lens) * 2 * hkv * D
    return {"bytes": 2 * (weights + kv) + 2 * len(lens) * V,
            "flops": 2 * len(lens) * weights + case["layers"] * 4 * hq * D * sum(lens)}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    if kind == "model":
        return {"rel": 0.03, "max": 0.5}
    if kind == "layer_ops":
        return {"rel": 4e-3, "max": 0.02}
    # bf16 outputs; weights of the softmax in bf16 in prefill
    return {"rel": 8e-3, "max": 0.25}


# ----------------------------------------------------------------------------- 64-bit results

def _rms64(x, w):
    x = x.double()
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope64(x, rows):
    """x [T, H, D] rotated by the table rows [T, D]."""
    c, s = rows.double()[:, None, :D // 2], rows.double()[:, None, D // 2:]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat((a * c - b * s, b * c + a * s), -1)


def _attend64(q, k, v, offset):
    """q [n, Hq, D] over k / v [m, Hkv, D]; query i sees keys up to i + offset."""
    n, hq, _ = q.shape
    m, hkv, _ = k.shape
    out = torch.empty(n, hq, D, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 26) // m)
    for h in range(hq):
        kh = k[:, h * hkv // hq].double().t().contiguous()
        vh = v[:, h * hkv // hq].double().contiguous()
        for i in range(0, n, step):
            s = torch.mm(q[i:i + step, h].double().contiguous(), kh) * D ** -0.5
            rows = torch.arange(i, min(n, i + step), device=q.device)[:, None]
            s.masked_fill_(torch.arange(m, device=q.device)[None, :] > rows + offset, -math.inf)
            out[i:i + step, h] = torch.mm(torch.softmax(s, -1), vh)
    return out


def _gather(cache, table, n):
    return cache[torch.tensor(table, device="cuda")].reshape(-1, *cache.shape[2:])[:n]


def _append64(k_cache, v_cache, slots, k, v):
    bs = k_cache.shape[1]
    k_cache[slots.long() // bs, slots.long() % bs] = k
    v_cache[slots.long() // bs, slots.long() % bs] = v


def _views64(pool, block, kv_heads):
    pages = pool.double().view(pool.shape[0], pool.shape[1], 2, block, kv_heads, D)
    return pages, [p[:, 0] for p in pages], [p[:, 1] for p in pages]


def _pool64(x, case, layers_k, layers_v):
    """The pool after the appends in 64 bits, where that is small enough to write down."""
    if x["pool"].numel() > 1 << 28:
        return None
    pages, k, v = _views64(x["pool"], case.get("block", 256), case["kv_heads"])
    for i, (kn, vn) in enumerate(zip(layers_k, layers_v)):
        _append64(k[i], v[i], x["slots"], kn.double(), vn.double())
    return pages.view(x["pool"].shape)


def _decode64(q, kn, vn, x, i):
    """Layer i's attention of one token per sequence; kn / vn: its own new k and v, or None."""
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    for b, (n, t) in enumerate(zip(x["lens"], x["tables"])):
        k, v = _gather(x["k"][i], t, n), _gather(x["v"][i], t, n)
        if kn is not None:
            k, v = k.double(), v.double()
            k[-1], v[-1] = kn[b], vn[b]
        G = q.shape[1] // k.shape[1]
        for h in range(k.shape[1]):
            s = torch.mm(q[b, G * h:G * h + G].double(), k[:, h].double().t().contiguous()) * D ** -0.5
            out[b, G * h:G * h + G] = torch.mm(torch.softmax(s, -1), v[:, h].double().contiguous())
    return out


@torch.inference_mode()
def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return None
    if kind == "decode":
        x = _decode_inputs(case, seed)
        hq, hkv, B = case["q_heads"], case["kv_heads"], case["seqs"]
        outs, ks, vs = [], [], []
        for i in range(case["layers"]):
            r = x["qkv"][i]
            q = r[:, :hq * D].reshape(B, hq, D)
            k, v = r[:, hq * D:(hq + hkv) * D].reshape(B, hkv, D), r[:, (hq + hkv) * D:].reshape(B, hkv, D)
            if case["entry"] == "step":
                rows = x["rope"][x["ctx"].long() - 1]
                q, k = _rope64(_rms64(q, x["qw"]), rows), _rope64(_rms64(k, x["kw"]), rows)
            new = case["entry"] != "call"
            outs.append(_decode64(q, k if new else None, v if new else None, x, i))
            ks.append(k)
            vs.append(v)
        if case["entry"] == "call":
            return outs[0]
        pool = _pool64(x, case, ks, vs)
        return (torch.stack(outs) if case["entry"] == "step" else outs[0]), pool
    if kind == "prefill":
        x = _prefill_inputs(case, seed)
        out = torch.empty(x["q"].shape, dtype=torch.float64, device="cuda")
        at = 0
        for (new, pre, _), t in zip(x["seqs"], x["tables"]):
            rows = slice(at, at + new)
            k, v = x["new_k"][rows], x["new_v"][rows]
            if pre:
                k = torch.cat((_gather(x["k"][0], t, pre), k))
                v = torch.cat((_gather(x["v"][0], t, pre), v))
            out[rows] = _attend64(x["q"][rows], k, v, pre)
            at += new
        return out, _pool64(x, case, [x["new_k"]], [x["new_v"]])
    if kind == "layer_ops":
        x = _layer_inputs(case, seed)
        T, hq, hkv = case["tokens"], case["q_heads"], case["kv_heads"]
        rows = x["rope"][x["positions"].long()]
        r = x["qkv"].view(T, hq + 2 * hkv, D)
        k = _rope64(_rms64(r[:, hq:hq + hkv], x["kw"]), rows)
        gate, up = x["gate_up"].double().chunk(2, -1)
        return (_rope64(_rms64(r[:, :hq], x["qw"]), rows), _rms64(x["hidden"], x["w"]),
                gate * torch.sigmoid(gate) * up, _pool64(x, case, [k], [r[:, hq + hkv:]]))
    x = _model_inputs(case, seed)
    w = {n: t.double() for n, t in x["weights"].items()}
    rows = _rope_table(4096)[x["positions"].long()]
    B, hq, hkv = case["seqs"], 16, 8
    pages = x["pages"].view(case["layers"], x["blocks"], 2, 256, hkv, D)
    x["k"], x["v"] = [p[:, 0] for p in pages], [p[:, 1] for p in pages]
    h = w["model.embed_tokens.weight"][x["ids"].long()]
    for i in range(case["layers"]):
        p = f"model.layers.{i}."
        n = _rms64(h, w[p + "input_layernorm.weight"])
        q, k, v = (torch.mm(n, w[p + f"self_attn.{s}_proj.weight"].t().contiguous()).view(B, -1, D) for s in "qkv")
        q = _rope64(_rms64(q, w[p + "self_attn.q_norm.weight"]), rows)
        k = _rope64(_rms64(k, w[p + "self_attn.k_norm.weight"]), rows)
        o = _decode64(q, k, v, x, i).reshape(B, hq * D)
        h = h + torch.mm(o, w[p + "self_attn.o_proj.weight"].t().contiguous())
        n = _rms64(h, w[p + "post_attention_layernorm.weight"])
        gate, up = (torch.mm(n, w[p + f"mlp.{s}_proj.weight"].t().contiguous()) for s in ("gate", "up"))
        h = h + torch.mm(gate * torch.sigmoid(gate) * up, w[p + "mlp.down_proj.weight"].t().contiguous())
    h = _rms64(h, w["model.norm.weight"])
    return (torch.mm(h, w["model.embed_tokens.weight"].t().contiguous()),)
