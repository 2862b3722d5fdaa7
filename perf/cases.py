"""Performance cases: the work a serving program has this library do.

A pass is what one engine step does with the entry point in question. Decode
work is replayed from a hipGraph, as the engine replays it; prefill work is
launched eagerly, as the engine launches it, with the step's metadata made in
the pass. The attention cases run several layers on one step's metadata, each
layer over a cache of its own. Shapes are the two head configurations of
``microinfer_amd.workloads`` (16 / 8 and 32 / 8 heads, head_dim 128, block 16)
and the Qwen3-0.6B dimensions of ``microinfer_amd.engine.model``.

Lengths come from the case alone (``lens`` seeds them), values and block
placement from the seed.
"""

from __future__ import annotations

import math
import random

import torch

HEAD_DIM = 128
BLOCK = 16
EPS = 1e-6
ROPE_BASE = 1e6
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
# Qwen3-0.6B (microinfer_amd.engine.model.QwenConfig), fewer layers.
HIDDEN, INTER, VOCAB, HQ, HKV = 1024, 3072, 151936, 16, 8


def listed():
    return [
        # Whole decode steps of the engine: one stream alone (interactive use,
        # the smallest step there is) and the engine benchmark's 64 requests.
        dict(name="decode_step_1", kind="decode_step", seqs=1, lo=300, hi=300, lens=1, layers=4),
        dict(name="decode_step_64", kind="decode_step", seqs=64, lo=128, hi=144, lens=2, layers=4),
        # A chunked-prefill step of the engine: 512 scheduled tokens, one chunk
        # continuing a cached prefix, ragged prompts beside it.
        dict(name="prefill_step", kind="prefill_step", chunks=4, chunk_lo=60, chunk_hi=200,
             prefix_hi=700, lens=3, layers=4),
        # Decode attention of a full batch, the append fused in (bench.py's
        # default workload).
        dict(name="decode_attn_batch", kind="decode_attn", dtype="bf16", hq=16, hkv=8, seqs=32,
             lo=128, hi=2048, lens=0, layers=8, how="fused"),
        # One long conversation: all of the context belongs to one sequence.
        dict(name="decode_attn_long", kind="decode_attn", dtype="bf16", hq=32, hkv=8, seqs=1,
             lo=16384, hi=16384, lens=0, layers=8, how="meta"),
        # Full-precision decode (debugging and parity runs), append and attend.
        dict(name="decode_attn_f32", kind="decode_attn", dtype="f32", hq=16, hkv=8, seqs=8,
             lo=64, hi=512, lens=0, layers=8, how="cached"),
        # The mixed step of chunked prefill: 8 chunks of 512 on cached prefixes
        # and 24 decode rows in one launch per layer. The largest case.
        dict(name="prefill_mixed", kind="prefill_attn", dtype="bf16", hq=32, hkv=8, chunks=8,
             chunk_lo=512, chunk_hi=512, prefix_hi=3072, decodes=24, paged=True, lens=0,
             layers=4),
        # New prompts without a cached prefix, of odd lengths, in half precision.
        dict(name="prefill_direct_f16", kind="prefill_attn", dtype="f16", hq=16, hkv=8, chunks=6,
             chunk_lo=150, chunk_hi=1300, prefix_hi=0, decodes=0, paged=False, lens=5, layers=4),
        # Full-precision prefill (parity runs): a few chunks on short prefixes.
        dict(name="prefill_f32", kind="prefill_attn", dtype="f32", hq=16, hkv=8, chunks=3,
             chunk_lo=77, chunk_hi=333, prefix_hi=700, decodes=0, paged=True, lens=6, layers=4),
        # The feed-forward half of decode layers at an odd batch.
        dict(name="mlp_decode", kind="mlp_decode", dtype="bf16", rows=37, hidden=1024, inter=3072,
             layers=8),
        # Q/K norm + RoPE + append of the mixed step's tokens.
        dict(name="qk_norm_rope", kind="qk_norm_rope", dtype="bf16", hq=32, hkv=8, tokens=4120),
        # Block-table gather of the long-prompt path.
        dict(name="gather_kv", kind="gather", dtype="bf16", hkv=8, seqs=6, lo=500, hi=6000,
             lens=7),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case, at most as much work as the largest listed one."""
    most = max(map(_cost, listed()))
    while True:
        case = _draw(rng)
        if _cost(case) <= most:
            return case


def _cost(case):
    w = work(case)
    return max(w["bytes"], w["flops"] / 50)


def _draw(rng):
    kind = rng.choice(["decode_step", "decode_step", "prefill_step", "decode_attn", "decode_attn",
                       "decode_attn", "prefill_attn", "prefill_attn", "prefill_attn",
                       "mlp_decode", "qk_norm_rope", "gather"])
    lens = rng.randrange(1 << 20)
    half = rng.choice(["bf16", "bf16", "f16"])
    hq = rng.choice([16, 32])
    if kind == "decode_step":
        lo = _log(rng, 16, 1000)
        return dict(kind=kind, seqs=_log(rng, 1, 64), lo=lo, hi=_log(rng, lo, 2 * lo), lens=lens,
                    layers=4)
    if kind == "prefill_step":
        lo = _log(rng, 8, 128)
        return dict(kind=kind, chunks=rng.randint(1, 6), chunk_lo=lo, chunk_hi=_log(rng, lo, 340),
                    prefix_hi=rng.choice([0, _log(rng, 16, 2000)]), lens=lens, layers=4)
    if kind == "decode_attn":
        dtype = rng.choice([half, half, half, "f32"])
        seqs = _log(rng, 1, 64)
        top = min(32768, 65536 // seqs) if dtype != "f32" else min(4096, 16384 // seqs)
        lo = _log(rng, min(64, top), top)
        return dict(kind=kind, dtype=dtype, hq=hq, hkv=8, seqs=seqs, lo=lo,
                    hi=_log(rng, lo, top), lens=lens, layers=8,
                    how=rng.choice(["fused", "meta", "cached"]))
    if kind == "prefill_attn":
        dtype = rng.choice([half, half, half, "f32"])
        chunks = rng.randint(1, 8)
        most = (4096 if dtype != "f32" else 1000) // chunks
        hi = _log(rng, 16, most)
        paged = rng.random() < 0.65
        return dict(kind=kind, dtype=dtype, hq=hq, hkv=8, chunks=chunks,
                    chunk_lo=_log(rng, max(1, hi // 4), hi), chunk_hi=hi,
                    prefix_hi=_log(rng, 16, 3000 if dtype != "f32" else 700) if paged else 0,
                    decodes=rng.choice([0, rng.randint(1, 32)]) if paged and dtype != "f32" else 0,
                    paged=paged, lens=lens, layers=4)
    if kind == "mlp_decode":
        hidden = rng.choice([1024, 1024, 2048, 4096])
        return dict(kind=kind, dtype=half, rows=_log(rng, 1, 64), hidden=hidden, inter=3 * hidden,
                    layers=8 if hidden == 1024 else 4)
    if kind == "qk_norm_rope":
        return dict(kind=kind, dtype=rng.choice([half, half, "f32"]), hq=hq, hkv=8,
                    tokens=_log(rng, 64, 8192))
    lo = _log(rng, 64, 4000)
    return dict(kind=kind, dtype=half, hkv=8, seqs=rng.randint(1, 8), lo=lo,
                hi=_log(rng, lo, 8000), lens=lens)


# ---------------------------------------------------------------------------
# Lengths (from the case) and inputs (from the seed).
# ---------------------------------------------------------------------------
def _contexts(case):
    """Context lengths of the sequences of a decode or gather case."""
    r = random.Random(case["lens"])
    return [r.randint(case["lo"], case["hi"]) for _ in range(case["seqs"])]


def _chunks(case):
    """(query lengths, context lengths): chunks on prefixes, then decode rows."""
    r = random.Random(case["lens"])
    q = [r.randint(case["chunk_lo"], case["chunk_hi"]) for _ in range(case["chunks"])]
    c = [n + r.randint(0, case["prefix_hi"]) for n in q]
    for _ in range(case.get("decodes", 0)):
        q.append(1)
        c.append(r.randint(256, 2048))
    return q, c


def _blocks(tokens):
    return -(-tokens // BLOCK)


def _gen(seed, salt):
    return torch.Generator(device="cuda").manual_seed(1000003 * int(seed) + salt)


def _randn(gen, dtype, *shape):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _tables(contexts, seed):
    """Block ids of each sequence: disjoint, in random order over the pool."""
    need = [_blocks(c) for c in contexts]
    ids = list(range(sum(need)))
    random.Random(seed).shuffle(ids)
    rows, at = [], 0
    for n in need:
        rows.append(ids[at:at + n])
        at += n
    return rows


def _table_tensor(rows):
    width = max(len(r) for r in rows)
    return torch.tensor([r + [-1] * (width - len(r)) for r in rows], dtype=torch.int32,
                        device="cuda")


def _cu(lengths):
    ends = [0]
    for n in lengths:
        ends.append(ends[-1] + n)
    return torch.tensor(ends, dtype=torch.int32, device="cuda")


def _slots(rows, contexts):
    return torch.tensor([row[(c - 1) // BLOCK] * BLOCK + (c - 1) % BLOCK
                         for row, c in zip(rows, contexts)], dtype=torch.int32, device="cuda")


def _pool(case, gen, blocks, heads, dtype):
    """One layer's cached K or V: what earlier steps left in the pool."""
    return _randn(gen, dtype, blocks, BLOCK, heads, HEAD_DIM)


def _caches(case, seed, layers, blocks, heads, dtype):
    """The bound cache of every layer, filled."""
    from microinfer_amd.worker.kv_cache import KVCache

    cache = KVCache(layers, blocks, BLOCK, heads, HEAD_DIM, dtype=dtype, device="cuda")
    for i in range(layers):
        gen = _gen(seed, 100 + i)
        cache.keys[i].copy_(_pool(case, gen, blocks, heads, dtype))
        cache.values[i].copy_(_pool(case, gen, blocks, heads, dtype))
    return [cache.layer(i) for i in range(layers)]


def _rows(case, seed, layer, count, heads, dtype, salt=0):
    return _randn(_gen(seed, 10000 + 100 * layer + salt), dtype, count, heads, HEAD_DIM)


def _model_weights(case, seed):
    """Random weights of the decoder, named as the model's fields."""
    gen = _gen(seed, 1)
    bf = torch.bfloat16

    def normal(*shape):
        return (0.02 * torch.randn(shape, generator=gen, device="cuda")).to(bf)

    def scale(n):
        return (1 + 0.1 * torch.randn(n, generator=gen, device="cuda")).to(bf)

    rows = (HQ + 2 * HKV) * HEAD_DIM
    w = {"embedding": normal(VOCAB, HIDDEN), "lm_head": normal(VOCAB, HIDDEN),
         "final_norm": scale(HIDDEN), "layers": []}
    for _ in range(case["layers"]):
        w["layers"].append({
            "pre_norm": scale(HIDDEN), "qkv": normal(rows, HIDDEN), "q_norm": scale(HEAD_DIM),
            "k_norm": scale(HEAD_DIM), "out": normal(HIDDEN, HQ * HEAD_DIM),
            "post_norm": scale(HIDDEN), "gate_up": normal(2 * INTER, HIDDEN),
            "down": normal(HIDDEN, INTER)})
    return w


def _token_ids(contexts, seed):
    r = random.Random(seed + 17)
    return [[r.randrange(VOCAB) for _ in range(c)] for c in contexts]


def _mlp_weights(case, seed, layer):
    gen, dtype = _gen(seed, 300 + layer), DTYPES[case["dtype"]]
    h, i = case["hidden"], case["inter"]

    def normal(*shape):
        return (0.02 * torch.randn(shape, generator=gen, device="cuda")).to(dtype)

    return ((1 + 0.1 * torch.randn(h, generator=gen, device="cuda")).to(dtype), normal(2 * i, h),
            normal(h, i))


def _qk_inputs(case, seed):
    gen, dtype, t = _gen(seed, 5), DTYPES[case["dtype"]], case["tokens"]
    qkv = _randn(gen, dtype, t, (case["hq"] + 2 * case["hkv"]) * HEAD_DIM)
    qw = (1 + 0.1 * torch.randn(HEAD_DIM, generator=gen, device="cuda")).to(dtype)
    kw = (1 + 0.1 * torch.randn(HEAD_DIM, generator=gen, device="cuda")).to(dtype)
    positions = torch.randint(0, 40960, (t,), generator=gen, device="cuda")
    blocks = 2 * _blocks(t)
    slots = torch.randperm(blocks * BLOCK, generator=gen, device="cuda")[:t].to(torch.int32)
    return qkv, qw, kw, positions, slots, blocks


# ---------------------------------------------------------------------------
# prepare
# ---------------------------------------------------------------------------
def _capture(step):
    """``step`` in a graph, as the engine captures a decode bucket."""
    from microinfer_amd.runner import capture_graph

    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side), torch.inference_mode():
        step()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with capture_graph(graph, stream=side), torch.inference_mode():
        out = step()
    torch.cuda.synchronize()
    return graph, out


def _model_runner(case, seed, contexts, graphs):
    from microinfer_amd.engine.config import EngineConfig
    from microinfer_amd.engine.model import QwenConfig, Qwen3Model
    from microinfer_amd.engine.model_runner import ModelRunner
    from microinfer_amd.engine.sequence import Sequence

    model = Qwen3Model(QwenConfig(num_hidden_layer=case["layers"]), dtype=torch.bfloat16,
                       device="cuda", seed=0)
    w = _model_weights(case, seed)
    for name in ("embedding", "lm_head", "final_norm"):
        getattr(model, name).copy_(w[name])
    for layer, values in zip(model.layers, w["layers"]):
        for name, value in values.items():
            getattr(layer, name).copy_(value)
    del w
    rows = _tables(contexts, seed)
    blocks = sum(len(r) for r in rows)
    runner = ModelRunner(model, EngineConfig(max_num_seqs=len(contexts), use_cuda_graph=graphs),
                         num_blocks=blocks, block_size=BLOCK)
    for i in range(case["layers"]):
        gen = _gen(seed, 100 + i)
        cache = runner.kv_cache.layer(i)
        cache.keys[:blocks].copy_(_pool(case, gen, blocks, HKV, torch.bfloat16))
        cache.values[:blocks].copy_(_pool(case, gen, blocks, HKV, torch.bfloat16))
    seqs = []
    for ids, row in zip(_token_ids(contexts, seed), rows):
        seq = Sequence(ids)
        seq.block_table = list(row)
        seqs.append(seq)
    return runner, seqs


def prepare(case, seed):
    kind = case["kind"]
    if kind == "decode_step":
        runner, seqs = _model_runner(case, seed, _contexts(case), True)
        return dict(kind=kind, runner=runner, seqs=seqs)
    if kind == "prefill_step":
        q, contexts = _chunks(case)
        runner, seqs = _model_runner(case, seed, contexts, False)
        for seq, n, c in zip(seqs, q, contexts):
            seq.num_cached_tokens, seq.num_scheduled_tokens = c - n, n
        return dict(kind=kind, runner=runner, seqs=seqs)
    dtype = DTYPES[case["dtype"]]
    if kind == "decode_attn":
        return _prepare_decode_attn(case, seed, dtype)
    if kind == "prefill_attn":
        q, contexts = _chunks(case)
        layers = case["layers"]
        state = dict(kind=kind, paged=case["paged"], max_q=max(q), max_k=max(contexts),
                     cu_q=_cu(q), cu_k=_cu(contexts),
                     query=[_rows(case, seed, i, sum(q), case["hq"], dtype)
                            for i in range(layers)])
        if case["paged"]:
            rows = _tables(contexts, seed)
            blocks = sum(len(r) for r in rows)
            state["tables"] = _table_tensor(rows)
            state["kv"] = [(c.keys, c.values) for c in _caches(case, seed, layers, blocks,
                                                              case["hkv"], dtype)]
        else:
            state["tables"] = None
            state["kv"] = [tuple(_rows(case, seed, i, sum(q), case["hkv"], dtype, salt)
                                 for salt in (1, 2)) for i in range(layers)]
        return state
    if kind == "mlp_decode":
        from microinfer_amd.layer.hip_dense import (hip_linear, hip_linear_swiglu,
                                                    hip_rms_norm_residual)

        gen = _gen(seed, 7)
        x = _randn(gen, dtype, case["rows"], case["hidden"])
        res = _randn(gen, dtype, case["rows"], case["hidden"])
        weights = [_mlp_weights(case, seed, i) for i in range(case["layers"])]

        def step():
            hidden, residual, outs = x, res, []
            for norm, gate_up, down in weights:
                normed, residual = hip_rms_norm_residual(hidden, residual, norm, EPS)
                hidden = hip_linear(hip_linear_swiglu(normed, gate_up), down)
                outs.append(hidden)
            return outs, residual

        graph, out = _capture(step)
        return dict(kind=kind, graph=graph, out=out, keep=(x, res, weights))
    if kind == "qk_norm_rope":
        from microinfer_amd.layer.hip_qk_norm_rope import rope_tables

        qkv, qw, kw, positions, slots, blocks = _qk_inputs(case, seed)
        cos, sin = rope_tables(40960, HEAD_DIM, ROPE_BASE, device="cuda")
        cache = _caches(case, seed, 1, blocks, case["hkv"], dtype)[0]
        return dict(kind=kind, qkv=qkv, qw=qw, kw=kw, positions=positions, slots=slots, cos=cos,
                    sin=sin, cache=cache, hq=case["hq"], hkv=case["hkv"])
    contexts = _contexts(case)
    rows = _tables(contexts, seed)
    cache = _caches(case, seed, 1, sum(len(r) for r in rows), case["hkv"], dtype)[0]
    return dict(kind=kind, cache=cache, tables=_table_tensor(rows), contexts=contexts)


def _prepare_decode_attn(case, seed, dtype):
    from microinfer_amd.layer.cached_attention import CachedAttention
    from microinfer_amd.layer.hip_paged_attention import hip_paged_decode
    from microinfer_amd.layer.metadata import AttentionMetadata
    from microinfer_amd.layer.paged_attention import paged_attention_meta

    contexts = _contexts(case)
    rows = _tables(contexts, seed)
    blocks = sum(len(r) for r in rows)
    n, layers, hq, hkv = case["seqs"], case["layers"], case["hq"], case["hkv"]
    caches = _caches(case, seed, layers, blocks, hkv, dtype)
    q = [_rows(case, seed, i, n, hq, dtype) for i in range(layers)]
    k = [_rows(case, seed, i, n, hkv, dtype, 1) for i in range(layers)]
    v = [_rows(case, seed, i, n, hkv, dtype, 2) for i in range(layers)]
    tables, slots = _table_tensor(rows), _slots(rows, contexts)
    lens = torch.tensor(contexts, dtype=torch.int32, device="cuda")
    attns = []
    for cache in caches:
        attns.append(CachedAttention())
        attns[-1].bind_cache(cache)

    def step():
        meta = AttentionMetadata.build(is_prefill=False, slot_mapping=slots, context_lens=lens,
                                       block_tables=tables, validate_cache_write=False)
        outs = []
        for i, cache in enumerate(caches):
            if case["how"] == "fused":
                outs.append(hip_paged_decode(
                    q[i], cache.keys, cache.values, tables, lens,
                    plan=meta.decode_plan(hkv, BLOCK), new_keys=k[i], new_values=v[i]))
            elif case["how"] == "cached":
                outs.append(attns[i](q[i], k[i], v[i], meta))
            else:
                outs.append(paged_attention_meta(q[i], cache.keys, cache.values, meta))
        return outs

    graph, outs = _capture(step)
    if case["how"] != "meta":  # the appended caches are results too
        outs = outs + [t for c in caches for t in (c.keys, c.values)]
    return dict(kind="decode_attn", graph=graph, out=outs, keep=(q, k, v, caches, tables, slots,
                                                                lens))


# ---------------------------------------------------------------------------
# run: one pass
# ---------------------------------------------------------------------------
def run(state):
    kind = state["kind"]
    if kind in ("decode_attn", "mlp_decode"):
        state["graph"].replay()
        return state["out"]
    if kind == "decode_step":
        # The step selects tokens too; over random weights they are near ties.
        return state["runner"].graphs.run(state["seqs"])[0]
    if kind == "prefill_step":
        runner = state["runner"]
        with torch.inference_mode():
            return runner.run_model(*runner.builder.prepare_prefill(state["seqs"]))
    if kind == "prefill_attn":
        from microinfer_amd.layer.metadata import AttentionMetadata
        from microinfer_amd.layer.paged_attention import paged_attention_meta, varlen_attention

        meta = AttentionMetadata.build(is_prefill=True, cu_seqlens_q=state["cu_q"],
                                       cu_seqlens_k=state["cu_k"], max_seqlen_q=state["max_q"],
                                       max_seqlen_k=state["max_k"], block_tables=state["tables"])
        attend = paged_attention_meta if state["paged"] else varlen_attention
        return [attend(q, k, v, meta) for q, (k, v) in zip(state["query"], state["kv"])]
    if kind == "qk_norm_rope":
        from microinfer_amd.layer.hip_qk_norm_rope import qk_norm_rope_append

        s, cache = state, state["cache"]
        q = qk_norm_rope_append(s["qkv"], q_weight=s["qw"], k_weight=s["kw"], eps=EPS,
                                cos_table=s["cos"], sin_table=s["sin"], positions=s["positions"],
                                num_q_heads=s["hq"], num_kv_heads=s["hkv"], head_dim=HEAD_DIM,
                                slot_mapping=s["slots"], key_cache=cache.keys,
                                value_cache=cache.values)
        return q, cache.keys, cache.values
    from microinfer_amd.layer.paged_attention import gather_paged_kv

    cache = state["cache"]
    return gather_paged_kv(cache.keys, cache.values, state["tables"], state["contexts"], BLOCK)


# ---------------------------------------------------------------------------
# work: bytes and operations a pass cannot do without
# ---------------------------------------------------------------------------
def _attn_flops(q, c, hq):
    return sum(4 * hq * HEAD_DIM * (n * (t - n) + n * (n + 1) // 2) for n, t in zip(q, c))


def _layer_weights():
    return ((HQ + 2 * HKV) * HEAD_DIM * HIDDEN + HIDDEN * HQ * HEAD_DIM + 3 * INTER * HIDDEN)


def work(case):
    kind = case["kind"]
    if kind in ("decode_step", "prefill_step"):
        if kind == "decode_step":
            c, q = _contexts(case), [1] * case["seqs"]
        else:
            q, c = _chunks(case)
        tokens, heads = sum(q), case["seqs"] if kind == "decode_step" else case["chunks"]
        kv = 4 * HKV * HEAD_DIM * (sum(c) + tokens)
        return dict(bytes=case["layers"] * (2 * _layer_weights() + kv) + 2 * VOCAB * HIDDEN
                    + 2 * tokens * HIDDEN + 2 * heads * VOCAB,
                    flops=case["layers"] * (2 * tokens * _layer_weights() + _attn_flops(q, c, HQ))
                    + 2 * heads * VOCAB * HIDDEN)
    es = 4 if case["dtype"] == "f32" else 2
    if kind == "decode_attn":
        c, n, hq, hkv = _contexts(case), case["seqs"], case["hq"], case["hkv"]
        append = 0 if case["how"] == "meta" else 4 * n * hkv * HEAD_DIM * es
        return dict(bytes=case["layers"] * (2 * sum(c) * hkv * HEAD_DIM * es + append
                                            + 2 * n * hq * HEAD_DIM * es
                                            + 4 * sum(map(_blocks, c)) + 8 * n),
                    flops=case["layers"] * 4 * hq * HEAD_DIM * sum(c))
    if kind == "prefill_attn":
        q, c = _chunks(case)
        return dict(bytes=case["layers"] * es * HEAD_DIM * (2 * sum(q) * case["hq"]
                                                            + 2 * sum(c) * case["hkv"]),
                    flops=case["layers"] * _attn_flops(q, c, case["hq"]))
    if kind == "mlp_decode":
        m, h, i = case["rows"], case["hidden"], case["inter"]
        return dict(bytes=case["layers"] * (6 * h * i + 4 * m * h) + 4 * m * h,
                    flops=case["layers"] * 6 * m * h * i)
    if kind == "qk_norm_rope":
        t, row = case["tokens"], HEAD_DIM * es
        return dict(bytes=t * (2 * (case["hq"] + 2 * case["hkv"]) * row + 4 * HEAD_DIM + 12),
                    flops=t * 10 * (case["hq"] + case["hkv"]) * HEAD_DIM)
    c = _contexts(case)
    return dict(bytes=4 * sum(c) * case["hkv"] * HEAD_DIM * es + 4 * sum(map(_blocks, c)), flops=0)


def tolerance(case):
    kind = case["kind"]
    if kind == "gather":
        return "exact"
    if kind in ("decode_step", "prefill_step"):
        # Four layers of bf16 roundings on the way to the logits: 1.6e-2 off 64 bits.
        return {"rel": 3e-2, "max": 0.3}
    if kind == "mlp_decode":
        return {"rel": 3e-2 if case["dtype"] == "bf16" else 4e-3, "max": 0.2}
    return {"bf16": {"rel": 1e-2, "max": 0.05}, "f16": {"rel": 1.5e-3, "max": 1e-2},
            "f32": {"rel": 4e-6, "max": 1e-4}}[case["dtype"]]


# ---------------------------------------------------------------------------
# exact: the same in 64 bits, plain torch
# ---------------------------------------------------------------------------
def _attend(q, k, v):
    """q [n, Hq, D] at the last n of the c positions of k, v [c, Hkv, D]."""
    n, hq, d = q.shape
    c, hkv, _ = k.shape
    g = hq // hkv
    qh = q.double().view(n, hkv, g, d).permute(1, 2, 0, 3).reshape(hkv, g * n, d)
    s = torch.matmul(qh, k.double().permute(1, 2, 0).contiguous()) / math.sqrt(d)
    seen = torch.arange(c, device=q.device)[None, :] <= torch.arange(c - n, c,
                                                                     device=q.device)[:, None]
    s = s.masked_fill(~seen.repeat(g, 1), -math.inf)
    o = torch.matmul(torch.softmax(s, -1), v.double().permute(1, 0, 2).contiguous())
    return o.view(hkv, g, n, d).permute(2, 0, 1, 3).reshape(n, hq, d)


def _gathered(pool, row, c):
    ids = torch.tensor(row, device=pool.device)
    return pool[ids].reshape(-1, *pool.shape[2:])[:c]


def _put(pool, slots, rows):
    pool.view(-1, *pool.shape[2:])[slots.long()] = rows
    return pool


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x, positions):
    half = HEAD_DIM // 2
    # The rotation takes float32 angle tables as its input.
    inv = ROPE_BASE ** (-torch.arange(0, HEAD_DIM, 2, device="cuda", dtype=torch.float32)
                        / HEAD_DIM)
    angle = torch.outer(torch.arange(40960, device="cuda", dtype=torch.float32), inv)
    cos = angle.cos()[positions].double()[:, None]
    sin = angle.sin()[positions].double()[:, None]
    a, b = x[..., :half], x[..., half:]
    return torch.cat([a * cos - b * sin, b * cos + a * sin], -1)


def _exact_model(case, seed, q, contexts):
    w = _model_weights(case, seed)
    rows = _tables(contexts, seed)
    blocks = sum(len(r) for r in rows)
    ids = _token_ids(contexts, seed)
    tokens = torch.tensor([t for s, n, c in zip(ids, q, contexts) for t in s[c - n:c]],
                          device="cuda")
    positions = torch.tensor([p for n, c in zip(q, contexts) for p in range(c - n, c)],
                             device="cuda")
    slots = torch.tensor([row[p // BLOCK] * BLOCK + p % BLOCK
                          for row, n, c in zip(rows, q, contexts) for p in range(c - n, c)],
                         device="cuda")
    x, qw, kvw = w["embedding"][tokens].double(), HQ * HEAD_DIM, HKV * HEAD_DIM
    for i, layer in enumerate(w["layers"]):
        gen = _gen(seed, 100 + i)
        keys = _pool(case, gen, blocks, HKV, torch.bfloat16).double()
        values = _pool(case, gen, blocks, HKV, torch.bfloat16).double()
        qkv = _rms(x, layer["pre_norm"]) @ layer["qkv"].double().T
        heads = qkv.view(len(tokens), -1, HEAD_DIM)
        query = _rope(_rms(heads[:, :HQ], layer["q_norm"]), positions)
        _put(keys, slots, _rope(_rms(heads[:, HQ:HQ + HKV], layer["k_norm"]), positions))
        _put(values, slots, heads[:, HQ + HKV:])
        outs, at = [], 0
        for row, n, c in zip(rows, q, contexts):
            outs.append(_attend(query[at:at + n], _gathered(keys, row, c),
                                _gathered(values, row, c)))
            at += n
        x = x + torch.cat(outs).view(-1, qw) @ layer["out"].double().T
        gate_up = _rms(x, layer["post_norm"]) @ layer["gate_up"].double().T
        x = x + (torch.nn.functional.silu(gate_up[:, :INTER]) * gate_up[:, INTER:]
                 ) @ layer["down"].double().T
    last = torch.tensor([sum(q[:i + 1]) - 1 for i in range(len(q))], device="cuda")
    return _rms(x, w["final_norm"])[last] @ w["lm_head"].double().T


def exact(case, seed):
    kind = case["kind"]
    if kind == "decode_step":
        contexts = _contexts(case)
        return _exact_model(case, seed, [1] * len(contexts), contexts)
    if kind == "prefill_step":
        return _exact_model(case, seed, *_chunks(case))
    dtype = DTYPES[case["dtype"]]
    if kind == "decode_attn":
        contexts = _contexts(case)
        rows = _tables(contexts, seed)
        blocks = sum(len(r) for r in rows)
        slots, outs, caches = _slots(rows, contexts), [], []
        for i in range(case["layers"]):
            gen = _gen(seed, 100 + i)
            keys = _pool(case, gen, blocks, case["hkv"], dtype)
            values = _pool(case, gen, blocks, case["hkv"], dtype)
            q = _rows(case, seed, i, len(contexts), case["hq"], dtype)
            if case["how"] != "meta":
                _put(keys, slots, _rows(case, seed, i, len(contexts), case["hkv"], dtype, 1))
                _put(values, slots, _rows(case, seed, i, len(contexts), case["hkv"], dtype, 2))
                caches += [keys, values]
            outs.append(torch.cat([_attend(q[s:s + 1], _gathered(keys, row, c),
                                           _gathered(values, row, c))
                                   for s, (row, c) in enumerate(zip(rows, contexts))]))
        return outs + caches
    if kind == "prefill_attn":
        q, contexts = _chunks(case)
        rows = _tables(contexts, seed) if case["paged"] else None
        outs = []
        for i in range(case["layers"]):
            query, parts, at = _rows(case, seed, i, sum(q), case["hq"], dtype), [], 0
            if case["paged"]:
                gen = _gen(seed, 100 + i)
                blocks = sum(len(r) for r in rows)
                keys = _pool(case, gen, blocks, case["hkv"], dtype)
                values = _pool(case, gen, blocks, case["hkv"], dtype)
            else:
                keys, values = (_rows(case, seed, i, sum(q), case["hkv"], dtype, salt)
                                for salt in (1, 2))
            for r, (n, c) in enumerate(zip(q, contexts)):
                k = _gathered(keys, rows[r], c) if case["paged"] else keys[at:at + n]
                v = _gathered(values, rows[r], c) if case["paged"] else values[at:at + n]
                parts.append(_attend(query[at:at + n], k, v))
                at += n
            outs.append(torch.cat(parts))
        return outs
    if kind == "mlp_decode":
        gen = _gen(seed, 7)
        hidden = _randn(gen, dtype, case["rows"], case["hidden"]).double()
        residual = _randn(gen, dtype, case["rows"], case["hidden"]).double()
        outs = []
        for i in range(case["layers"]):
            norm, gate_up, down = _mlp_weights(case, seed, i)
            residual = residual + hidden
            both = _rms(residual, norm) @ gate_up.double().T
            gate, up = both.chunk(2, -1)
            hidden = (torch.nn.functional.silu(gate) * up) @ down.double().T
            outs.append(hidden)
        return outs, residual
    if kind == "qk_norm_rope":
        qkv, qw, kw, positions, slots, blocks = _qk_inputs(case, seed)
        hq, hkv = case["hq"], case["hkv"]
        heads = qkv.double().view(case["tokens"], -1, HEAD_DIM)
        gen = _gen(seed, 100)
        keys = _pool(case, gen, blocks, hkv, dtype).double()
        values = _pool(case, gen, blocks, hkv, dtype).double()
        _put(keys, slots, _rope(_rms(heads[:, hq:hq + hkv], kw), positions))
        _put(values, slots, heads[:, hq + hkv:])
        return _rope(_rms(heads[:, :hq], qw), positions), keys, values
    contexts = _contexts(case)
    rows = _tables(contexts, seed)
    gen, blocks = _gen(seed, 100), sum(len(r) for r in rows)
    keys = _pool(case, gen, blocks, case["hkv"], dtype)
    values = _pool(case, gen, blocks, case["hkv"], dtype)
    return tuple(torch.cat([_gathered(p, row, c) for row, c in zip(rows, contexts)])
                 for p in (keys, values))
