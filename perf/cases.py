"""Performance cases of the paged-KV framework: what a serving engine asks of it.

Every case is one pass through the public entry points, on inputs made from a
seed: the single calls of a layer (store, gather, fused store + gather, decode
attention, prefill attention) and one whole decode step as a captured graph
replays it.  Head layouts, block size and context laws are those of
nanokv.workloads and the benchmark: 8 x 128, 4 x 128 and 2 x 128 kv rows,
256-token blocks, contexts log-uniform up to 16k.

``listed()`` is the fixed list, ``draw(rng)`` one more case of the same
ranges.  A case names its kind and sizes; the sequence lengths follow from the
case alone (``lengths`` seeds them), so ``work`` knows them; block tables and
values follow from the seed given to ``prepare``.
"""
from __future__ import annotations

import math
import random
import sys
from pathlib import Path

import torch

_PACKAGE = str(Path(__file__).resolve().parents[1] / "nano-vllm-multimodal_amd")
if _PACKAGE not in sys.path:
    sys.path.insert(0, _PACKAGE)

HEAD_DIM = 128
BLOCK = 256
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
DEVICE = "cuda"


def listed() -> list[dict]:
    return [
        # One layer's store of a decode step's new rows, 64 sequences: the
        # smallest call of a step, made once per layer.
        {"name": "store_decode", "kind": "store", "tokens": 64, "kv": 8, "q": 16, "dtype": "bf16"},
        # The reference op as SDPA attention calls it: K, then V, of one
        # request (text and one image span) from narrow rows.
        {"name": "gather_request", "kind": "gather", "tokens": 1429, "kv": 2, "dtype": "fp16"},
        # A full prefill chunk: the layer's store and the gather of every
        # request's context, half the requests continuing earlier chunks.
        {"name": "chunk_store_gather", "kind": "store_gather", "seqs": 16, "new": 8192,
         "cached": 2048, "kv": 8, "q": 16, "dtype": "bf16", "lengths": 18},
        # One layer of a 256-sequence decode step that gathers: store, then K
        # and V of every context in one launch (the headline step's layer).
        {"name": "step_gather", "kind": "step_gather", "seqs": 256, "low": 256, "high": 16384,
         "kv": 8, "q": 16, "dtype": "bf16", "lengths": 21},
        # Decode attention of a single user's conversation: latency.
        {"name": "decode_single", "kind": "decode", "seqs": 1, "low": 5003, "high": 5003,
         "kv": 8, "q": 16, "dtype": "bf16", "lengths": 1},
        # Decode attention of a lightly loaded server, 7 query heads per kv head.
        {"name": "decode_small", "kind": "decode", "seqs": 8, "low": 256, "high": 16384,
         "kv": 4, "q": 28, "dtype": "fp16", "lengths": 5},
        # Decode attention of the headline step's layer, the chip full.
        {"name": "decode_full", "kind": "decode", "seqs": 256, "low": 256, "high": 16384,
         "kv": 8, "q": 16, "dtype": "bf16", "lengths": 21},
        # First prefill of one multimodal prompt (text, one image span, text):
        # nothing cached, so keys come straight from the projection.
        {"name": "prefill_prompt", "kind": "prefill", "paged": False, "seqs": 1, "new": 1511,
         "cached": 0, "kv": 2, "q": 16, "dtype": "bf16", "lengths": 3},
        # A full prefill chunk of 16 requests through the paged cache, half of
        # them continuing.
        {"name": "prefill_chunk", "kind": "prefill", "paged": True, "seqs": 16, "new": 8192,
         "cached": 2048, "kv": 8, "q": 16, "dtype": "bf16", "lengths": 18},
        # One long prompt that fills the chunk by itself.
        {"name": "prefill_long", "kind": "prefill", "paged": False, "seqs": 1, "new": 8192,
         "cached": 0, "kv": 4, "q": 28, "dtype": "bf16", "lengths": 2},
        # The next turn of 4 conversations: short questions over long
        # contexts found in the prefix cache.
        {"name": "prefill_followup", "kind": "prefill", "paged": True, "seqs": 4, "new": 391,
         "cached": 12288, "kv": 8, "q": 16, "dtype": "bf16", "lengths": 7},
        # A whole decode step as the engine replays it: metadata packed into
        # the graph's buffers, then a captured graph of 12 layers of store and
        # decode attention, 30 sequences in a bucket of 32.
        {"name": "decode_graph", "kind": "graph", "seqs": 30, "bucket": 32, "low": 256,
         "high": 8192, "kv": 8, "q": 32, "dtype": "bf16", "layers": 12, "lengths": 11},
    ]


def _log_int(rng: random.Random, low: int, high: int) -> int:
    return max(low, min(high, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(("store", "gather", "store_gather", "step_gather", "decode", "decode",
                       "decode", "prefill", "prefill", "prefill", "prefill", "graph"))
    kv, q = rng.choice(((8, 16), (8, 32), (4, 28), (2, 16)))
    half = rng.choice(("bf16", "bf16", "fp16"))
    lengths = rng.randrange(1 << 20)
    if kind == "store":
        return {"kind": kind, "tokens": _log_int(rng, 1, 8192), "kv": kv, "q": q,
                "dtype": rng.choice(("bf16", "fp16", "fp32"))}
    if kind == "gather":
        return {"kind": kind, "tokens": _log_int(rng, 1, 32768), "kv": kv,
                "dtype": rng.choice(("bf16", "fp16", "fp32"))}
    if kind == "store_gather":
        seqs = _log_int(rng, 1, 24)
        return {"kind": kind, "seqs": seqs, "new": _log_int(rng, 64 * seqs, 8192),
                "cached": rng.choice((0, 1024, 2048, 4096)), "kv": kv, "q": q,
                "dtype": rng.choice(("bf16", "fp16", "fp32")), "lengths": lengths}
    if kind == "step_gather":
        return {"kind": kind, "seqs": _log_int(rng, 2, 128), "low": 256, "high": 16384, "kv": kv,
                "q": q, "dtype": half, "lengths": lengths}
    if kind == "decode":
        return {"kind": kind, "seqs": _log_int(rng, 1, 256), "low": _log_int(rng, 17, 1024),
                "high": _log_int(rng, 2048, 16384), "kv": kv, "q": q, "dtype": half,
                "lengths": lengths}
    if kind == "prefill":
        seqs = _log_int(rng, 1, 16)
        new = _log_int(rng, 16 * seqs, 8192)
        paged = rng.random() < 0.6
        cached = _log_int(rng, 256, 16384) if paged else 0
        return {"kind": kind, "paged": paged, "seqs": seqs, "new": new, "cached": cached, "kv": kv,
                "q": q, "dtype": half, "lengths": lengths}
    seqs = _log_int(rng, 1, 48)
    return {"kind": "graph", "seqs": seqs, "bucket": max(1, -(-seqs // 8) * 8), "low": 256,
            "high": _log_int(rng, 1024, 8192), "kv": kv, "q": q, "dtype": half,
            "layers": rng.choice((4, 8, 12)), "lengths": lengths}


# ------------------------------------------------------------------ lengths

def _lengths(case: dict) -> tuple[list[int], list[int]]:
    """(cached, new) tokens of every sequence."""
    rng = random.Random(int(case.get("lengths", 0)))
    kind = case["kind"]
    if kind in ("decode", "step_gather", "graph"):
        ctx = [_log_int(rng, case["low"], case["high"]) for _ in range(case["seqs"])]
        return [c - 1 for c in ctx], [1] * len(ctx)
    seqs, total = case["seqs"], case["new"]
    # Uneven shares of the chunk, at least one token each.
    shares = [rng.uniform(1.0, 8.0) for _ in range(seqs)]
    new = [max(1, int(total * s / sum(shares))) for s in shares]
    new[-1] += total - sum(new)
    if new[-1] < 1:
        new = [total // seqs] * (seqs - 1) + [total - (seqs - 1) * (total // seqs)]
    # Cached prefixes are whole blocks; every second request of a store +
    # gather or paged prefill step has none, unless the case is a follow-up
    # turn (few new tokens over a long context), where all have one.
    cached = [0] * seqs
    if case["cached"]:
        most = max(1, case["cached"] // BLOCK)
        follow_up = total <= case["cached"] // 4
        for i in range(seqs):
            if follow_up or i % 2 == 0:
                cached[i] = BLOCK * rng.randint((most + 1) // 2 if follow_up else 1, most)
    return cached, new


def _contexts(case: dict) -> list[int]:
    cached, new = _lengths(case)
    return [c + n for c, n in zip(cached, new)]


# ------------------------------------------------------------------- inputs

def _normal(shape, dtype, gen) -> torch.Tensor:
    return torch.randn(shape, dtype=dtype, device=DEVICE, generator=gen)


def _qkv(tokens: int, case: dict, gen):
    """q, k, v as views of one fused projection output, as attention gets them."""
    kv, q = case["kv"], case.get("q", case["kv"])
    fused = _normal((tokens, (q + 2 * kv) * HEAD_DIM), DTYPES[case["dtype"]], gen)
    parts = fused.split([q * HEAD_DIM, kv * HEAD_DIM, kv * HEAD_DIM], dim=1)
    return [p.view(tokens, -1, HEAD_DIM) for p in parts]


def _int32(values) -> torch.Tensor:
    return torch.tensor(values, dtype=torch.int32, device=DEVICE)


def _cu(lens) -> torch.Tensor:
    out = [0]
    for n in lens:
        out.append(out[-1] + n)
    return _int32(out)


def _block_lists(ctx: list[int], seed: int, headroom: float = 1.1):
    """Distinct physical blocks per sequence in random order, as a free list
    that has seen traffic hands them out; returns (lists, num_blocks)."""
    need = [-(-c // BLOCK) for c in ctx]
    num_blocks = max(8, math.ceil(sum(need) * headroom))
    order = list(range(num_blocks))
    random.Random(seed).shuffle(order)
    lists, at = [], 0
    for n in need:
        lists.append(order[at: at + n])
        at += n
    return lists, num_blocks


def _padded(lists, width=None) -> torch.Tensor:
    width = max(1, max(len(t) for t in lists)) if width is None else width
    return _int32([t + [-1] * (width - len(t)) for t in lists])


def _slots(lists, cached, new) -> list[int]:
    return [t[p // BLOCK] * BLOCK + p % BLOCK
            for t, c, n in zip(lists, cached, new) for p in range(c, c + n)]


def _inputs(case: dict, seed: int) -> dict:
    """Everything of a case that is plain data."""
    gen = torch.Generator(device=DEVICE)
    gen.manual_seed(int(seed))
    kind, dtype, kv = case["kind"], DTYPES[case["dtype"]], case["kv"]
    s: dict = {"case": dict(case), "scale": HEAD_DIM ** -0.5}
    if kind == "store":
        tokens = case["tokens"]
        blocks = max(64, -(-2 * tokens // BLOCK))
        s["k_cache"] = _normal((blocks, BLOCK, kv, HEAD_DIM), dtype, gen)
        s["v_cache"] = _normal((blocks, BLOCK, kv, HEAD_DIM), dtype, gen)
        s["q"], s["k"], s["v"] = _qkv(tokens, case, gen)
        slots = random.Random(seed).sample(range(blocks * BLOCK), tokens)
        for i in range(15, tokens, 16):  # padding rows of a graph bucket
            slots[i] = -1
        s["slots"] = _int32(slots)
        return s
    if kind == "gather":
        lists, blocks = _block_lists([case["tokens"]] * 2, seed, 4.0)
        s["k_cache"] = _normal((blocks, BLOCK, kv, HEAD_DIM), dtype, gen)
        s["v_cache"] = _normal((blocks, BLOCK, kv, HEAD_DIM), dtype, gen)
        s["table"] = _int32(lists[0])
        return s
    cached, new = _lengths(case)
    ctx = [c + n for c, n in zip(cached, new)]
    s["cu_q"], s["cu_k"], s["total"] = _cu(new), _cu(ctx), sum(ctx)
    s["max_q"], s["max_k"] = max(new), max(ctx)
    s["q"], s["k"], s["v"] = _qkv(sum(new), case, gen)
    if kind == "prefill" and not case["paged"]:
        return s
    lists, blocks = _block_lists(ctx, seed)
    s["lists"], s["ctx"] = lists, ctx
    layers = case["layers"] if kind == "graph" else 1
    cache = _normal((2, layers, blocks, BLOCK, kv, HEAD_DIM), dtype, gen)
    s["cache"], s["k_cache"], s["v_cache"] = cache, cache[0, 0], cache[1, 0]
    s["tables"] = _padded(lists)
    s["slots"] = _int32(_slots(lists, cached, new))
    if kind == "graph":
        pad = case["bucket"]
        s["layer_qkv"] = [_qkv(pad, case, gen) for _ in range(layers)]
    if kind == "prefill":  # the step's rows are in the cache before attention runs
        s["k_cache"].view(-1, kv, HEAD_DIM)[s["slots"].long()] = s["k"]
        s["v_cache"].view(-1, kv, HEAD_DIM)[s["slots"].long()] = s["v"]
    return s


def prepare(case: dict, seed: int) -> dict:
    from nanokv.paged_kv import create_paged_kv_backend

    s = _inputs(case, seed)
    backend = s["backend"] = create_paged_kv_backend("hip")
    kind = case["kind"]
    # Plans are built once per step and serve all of its layers.
    if kind == "store_gather":
        s["plan"] = backend.build_store_gather_plan(s["k_cache"], s["tables"], s["cu_q"], s["cu_k"],
                                                    s["k"].shape[0], s["total"])
    if kind == "step_gather":
        s["plan"] = backend.build_gather_plan(s["k_cache"], s["tables"], s["cu_k"], s["total"])
    if kind in ("store_gather", "step_gather"):
        out = torch.empty((s["total"], case["kv"], HEAD_DIM), dtype=s["k"].dtype, device=DEVICE)
        s["out"] = (out, torch.empty_like(out))
    if kind == "decode":
        s["plan"] = backend.build_attention_plan(s["k_cache"], s["cu_k"], s["total"])
    if kind == "prefill" and case["paged"]:
        s["plan"] = backend.build_prefill_plan(s["q"], s["k_cache"], s["cu_q"], s["cu_k"])
    if kind == "graph":
        _capture(s)
    return s


def _capture(s: dict) -> None:
    """The decode graph of the engine: per layer, store and decode attention
    on the fixed buffers of one batch bucket."""
    from nanokv.flash import flash_attn_with_kvcache
    from nanokv.packing import DecodeGraphBuffers, DevicePacker, SequenceBatch

    case, cache, bucket = s["case"], s["cache"], s["case"]["bucket"]
    s["packer"] = DevicePacker(DEVICE, BLOCK)
    buffers = s["buffers"] = DecodeGraphBuffers.allocate(DEVICE, bucket, -(-case["high"] // BLOCK))
    s["batch_of"] = lambda: SequenceBatch.from_block_lists(s["ctx"], s["lists"])
    s["packer"].pack_decode_into(s["batch_of"](), buffers)

    def layers():
        outs = []
        for i, (q, k, v) in enumerate(s["layer_qkv"]):
            s["backend"].store(k, v, cache[0, i], cache[1, i], buffers.slot_mapping)
            outs.append(flash_attn_with_kvcache(
                q.unsqueeze(1), cache[0, i], cache[1, i], cache_seqlens=buffers.context_lens,
                block_table=buffers.block_tables, softmax_scale=s["scale"], causal=True))
        return outs

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        layers()
    torch.cuda.current_stream().wait_stream(side)
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        s["outs"] = layers()


def run(s: dict):
    kind, backend = s["case"]["kind"], s["backend"]
    if kind == "store":
        backend.store(s["k"], s["v"], s["k_cache"], s["v_cache"], s["slots"])
        return s["k_cache"], s["v_cache"]
    if kind == "gather":
        length = s["case"]["tokens"]
        return (backend.gather(s["k_cache"], s["table"], length),
                backend.gather(s["v_cache"], s["table"], length))
    if kind == "store_gather":
        out = backend.store_gather(s["k"], s["v"], s["k_cache"], s["v_cache"], s["slots"],
                                   s["tables"], s["cu_q"], s["cu_k"], s["total"], plan=s["plan"],
                                   out=s["out"])
        return s["k_cache"], s["v_cache"], out
    if kind == "step_gather":
        backend.store(s["k"], s["v"], s["k_cache"], s["v_cache"], s["slots"])
        out = backend.gather_varlen(s["k_cache"], s["v_cache"], s["tables"], s["cu_k"], s["total"],
                                    plan=s["plan"], out=s["out"])
        return s["k_cache"], s["v_cache"], out
    if kind == "decode":
        return backend.paged_attention_decode(s["q"], s["k_cache"], s["v_cache"], s["tables"],
                                              s["cu_k"], s["total"], s["scale"], plan=s["plan"])
    if kind == "prefill" and s["case"]["paged"]:
        return backend.paged_attention_prefill(s["q"], s["k_cache"], s["v_cache"], s["tables"],
                                               s["cu_q"], s["cu_k"], s["scale"],
                                               total_context_tokens=s["total"], plan=s["plan"])
    if kind == "prefill":
        from nanokv.flash import flash_attn_varlen_func

        return flash_attn_varlen_func(s["q"], s["k"], s["v"], max_seqlen_q=s["max_q"],
                                      cu_seqlens_q=s["cu_q"], max_seqlen_k=s["max_k"],
                                      cu_seqlens_k=s["cu_k"], softmax_scale=s["scale"], causal=True)
    s["packer"].pack_decode_into(s["batch_of"](), s["buffers"])
    s["graph"].replay()
    return [o[: s["case"]["seqs"]] for o in s["outs"]], s["cache"]


# ----------------------------------------------------------------- the rest

def work(case: dict) -> dict:
    size = torch.empty((), dtype=DTYPES[case["dtype"]]).element_size()
    row, kind = case["kv"] * HEAD_DIM * size, case["kind"]
    if kind == "store":
        tokens = case["tokens"] - case["tokens"] // 16
        return {"bytes": 4 * tokens * row + 4 * case["tokens"], "flops": 0}
    if kind == "gather":
        return {"bytes": 4 * case["tokens"] * row + 8 * -(-case["tokens"] // BLOCK), "flops": 0}
    cached, new = _lengths(case)
    ctx = [c + n for c, n in zip(cached, new)]
    q_row = case["q"] * HEAD_DIM * size
    if kind == "store_gather":
        return {"bytes": 2 * row * (sum(new) + sum(cached) + sum(new) + sum(ctx)), "flops": 0}
    if kind == "step_gather":
        return {"bytes": 4 * row * (sum(new) + sum(ctx)), "flops": 0}
    pairs = sum(n * c + n * (n + 1) // 2 for c, n in zip(cached, new))
    bytes_ = 2 * row * sum(ctx) + 2 * q_row * sum(new)
    flops = 4 * HEAD_DIM * case["q"] * pairs
    if kind == "graph":
        return {"bytes": case["layers"] * (bytes_ + 4 * row * sum(new)),
                "flops": case["layers"] * flops}
    return {"bytes": bytes_, "flops": flops}


def tolerance(case: dict):
    if case["kind"] in ("store", "gather", "store_gather", "step_gather"):
        return "exact"  # bytes are moved, never converted
    # The softmax weights and the result are rounded to the element type:
    # 2.3e-3 (bf16) and 3.5e-4 (fp16) from 64 bits as measured, times four.
    if case["dtype"] == "fp16":
        return {"rel": 1.5e-3, "max": 1.5e-2}
    return {"rel": 1e-2, "max": 8e-2}


def _attend(q, k, v, cached: int, scale: float) -> torch.Tensor:
    """Causal attention of one sequence in 64 bits: q [n, Hq, D], k and v
    [cached + n, Hkv, D]; query j sees keys [0, cached + j]."""
    n, heads, kv = q.shape[0], q.shape[1], k.shape[1]
    out = torch.empty((n, heads, HEAD_DIM), dtype=torch.float64, device=DEVICE)
    group = heads // kv
    step = max(1, min(n, (1 << 27) // max(1, k.shape[0])))
    for h in range(heads):
        kh = k[:, h // group].double().t().contiguous()
        vh = v[:, h // group].double().contiguous()
        for a in range(0, n, step):
            scores = (q[a: a + step, h].double() @ kh) * scale
            seen = torch.arange(k.shape[0], device=DEVICE)[None, :]
            at = torch.arange(a, min(n, a + step), device=DEVICE)[:, None] + cached
            out[a: a + step, h] = scores.masked_fill_(seen > at, -math.inf).softmax(1) @ vh
    return out


def _attend_one(q, k, v, scale: float) -> torch.Tensor:
    """Decode attention of one sequence in 64 bits: q [Hq, D], k and v [L, Hkv, D]."""
    kv, group = k.shape[1], q.shape[0] // k.shape[1]
    kd = k.double().permute(1, 2, 0).contiguous()  # [Hkv, D, L]
    vd = v.double().permute(1, 0, 2).contiguous()  # [Hkv, L, D]
    weights = torch.bmm(q.double().view(kv, group, HEAD_DIM) * scale, kd).softmax(2)
    return torch.bmm(weights, vd).reshape(kv * group, HEAD_DIM)


def exact(case: dict, seed: int):
    kind = case["kind"]
    if kind not in ("decode", "prefill", "graph"):
        return None
    s = _inputs(case, seed)
    cached, new = _lengths(case)

    def context(cache, i):
        rows = cache[torch.tensor(s["lists"][i], device=DEVICE)]
        return rows.reshape(-1, *rows.shape[2:])[: s["ctx"][i]]

    if kind == "decode":
        return torch.stack([_attend_one(s["q"][i], context(s["k_cache"], i),
                                        context(s["v_cache"], i), s["scale"])
                            for i in range(case["seqs"])])
    if kind == "graph":
        outs = []
        for layer, (q, k, v) in enumerate(s["layer_qkv"]):
            rows = []
            for i in range(case["seqs"]):
                kc, vc = context(s["cache"][0, layer], i), context(s["cache"][1, layer], i)
                kc[-1], vc[-1] = k[i], v[i]  # the step's store (context() copies)
                rows.append(_attend_one(q[i], kc, vc, s["scale"]))
            outs.append(torch.stack(rows).unsqueeze(1))
        return outs, None
    out, at = [], 0
    for i, (c, n) in enumerate(zip(cached, new)):
        if case["paged"]:
            k, v = context(s["k_cache"], i), context(s["v_cache"], i)
        else:
            k, v = s["k"][at: at + n], s["v"][at: at + n]
        out.append(_attend(s["q"][at: at + n], k, v, c, s["scale"]))
        at += n
    return torch.cat(out)
