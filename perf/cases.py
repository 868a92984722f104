"""The work this framework does for its users, as timed cases over its public entry points.

Kinds of case (`case["kind"]`), each a call or a short run of calls as an engine makes them:

* request: attention.attention_for_request, one request at a time (the latency of a single call).
* batch:   attention.paged_decode_batch with the new rows' page write (the backend contract of
           the batched decode: int64 tables, positions, active mask).
* step:    the attention of one decode step over several layers: one plan, then per layer
           the decode with the fused page write.  float32 caches and pages below 16 tokens have
           no plan and go without.
* shared:  one layer's decode for groups of rows that share a prompt prefix.
* prefill: the attention of one ragged prefill step: the step's plan, then per layer the
           page write of the chunks and the causal attention over cached + new tokens.
* block:   decoder layers of a decode step (projections, norms, RoPE, attention, MLP) replayed
           from a HIP graph, as the engine's captured buckets run.
* model:   a whole decode step through GraphDecodeStep (buckets 1/2/4/8): logits and pools.
* forward: a whole ragged forward through Qwen2Model.forward: last-token logits and pools.

Head shapes, block sizes and length ranges are those of the repository's workloads, tests and
benchmark (12/2/128, 14/2/64) and a generic 32/8/128.  Values are N(0, 1), tables are random
permutations of the pool, and what the context lengths are follows from the case alone, so that
work() can count them.
"""
from __future__ import annotations

import math
import random

import torch

from flexengine_amd import attention, ops
from flexengine_amd.decode_step import GraphDecodeStep
from flexengine_amd.kv_cache import CacheLayout, PagedKVCache
from flexengine_amd.model import Chunk, Qwen2Config, Qwen2Model

DEV = "cuda:0"
HEADS = ((12, 2, 128), (14, 2, 64), (32, 8, 128))
# decoder sizes of the two models whose head shapes the workloads use
DECODERS = {
    "1.5b": dict(hidden_size=1536, intermediate_size=8960, num_attention_heads=12,
                 num_key_value_heads=2, head_dim=128),
    "0.5b": dict(hidden_size=896, intermediate_size=4864, num_attention_heads=14,
                 num_key_value_heads=2, head_dim=64),
}


def listed():
    return [
        # one chat request's next token through the per-request route: the smallest call
        dict(name="request_token", kind="request", new=1, cached=512, hq=12, hkv=2, d=128,
             dtype="float16", block=16, sizes=1),
        # a small server's decode batch, short contexts, head_dim 64
        dict(name="batch_small", kind="batch", rows=8, lo=16, hi=512, hq=14, hkv=2, d=64,
             dtype="float16", block=16, sizes=2),
        # a busy server's decode step: 64 rows, mixed contexts up to 4096
        dict(name="step_mixed", kind="step", layers=4, rows=64, lo=128, hi=4096, hq=12, hkv=2,
             d=128, dtype="float16", block=16, sizes=3),
        # long-context decode, bfloat16, larger pages: the most K/V that one step reads here
        dict(name="step_long", kind="step", layers=2, rows=37, lo=2048, hi=16384, hq=32, hkv=8,
             d=128, dtype="bfloat16", block=32, sizes=4),
        # the reference's default cache type
        dict(name="step_float32", kind="step", layers=2, rows=48, lo=128, hi=4096, hq=12, hkv=2,
             d=128, dtype="float32", block=16, sizes=5),
        # many users behind a few system prompts
        dict(name="shared_prefix", kind="shared", groups=8, members=32, prefix=2048, lo=16,
             hi=2048, hq=12, hkv=2, d=128, dtype="float16", block=16, sizes=6),
        # continuous batching: four prompt chunks over cached contexts
        dict(name="chunks", kind="prefill", layers=2, chunks=4, new_lo=256, new_hi=500,
             cached_hi=3072, hq=12, hkv=2, d=128, dtype="float16", block=16, sizes=7),
        # one long prompt at once, odd length, bfloat16
        dict(name="prompt_long", kind="prefill", layers=1, chunks=1, new_lo=8191, new_hi=8191,
             cached_hi=0, hq=32, hkv=8, d=128, dtype="bfloat16", block=16, sizes=8),
        # float32 chunks
        dict(name="chunks_float32", kind="prefill", layers=1, chunks=3, new_lo=100, new_hi=700,
             cached_hi=1500, hq=12, hkv=2, d=128, dtype="float32", block=16, sizes=9),
        # three decoder layers at four rows inside a captured step
        dict(name="block_rows4", kind="block", decoder="1.5b", layers=3, rows=4, lo=512, hi=4096,
             block=16, sizes=10),
        # a whole captured decode step of eight requests
        dict(name="model_step8", kind="model", decoder="1.5b", layers=28, vocab=151936, rows=8,
             lo=512, hi=4096, block=16, sizes=11),
        # a whole ragged forward: two fresh prompts and two later chunks
        dict(name="model_forward", kind="forward", decoder="1.5b", layers=28, vocab=151936,
             chunks=4, new_lo=256, new_hi=500, cached_hi=3072, block=16, sizes=12),
    ]


def _log(rng, lo, hi):
    """An integer spread over the logarithm of lo..hi."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(("request", "batch", "step", "step", "shared", "prefill", "prefill", "block",
                       "model"))
    hq, hkv, d = rng.choice(HEADS)
    case = dict(kind=kind, hq=hq, hkv=hkv, d=d, sizes=rng.randrange(1 << 30),
                dtype=rng.choice(("float16", "float16", "bfloat16", "bfloat16", "float32")),
                block=rng.choice((16, 16, 32)))
    if kind == "request":
        case.update(new=rng.choice((1, 1, _log(rng, 2, 600))), cached=_log(rng, 16, 4096))
    elif kind == "batch":
        lo = _log(rng, 16, 1024)
        case.update(rows=_log(rng, 2, 64), lo=lo, hi=_log(rng, lo, 4096))
    elif kind == "step":
        lo = _log(rng, 64, 4096)
        case.update(layers=rng.randint(1, 4), rows=_log(rng, 4, 128), lo=lo,
                    hi=_log(rng, lo, 12288))
        # at most about 3 GB of K and V in all
        token = 2 * hkv * d * (4 if case["dtype"] == "float32" else 2) * case["layers"] * case["rows"]
        case["hi"] = max(lo, min(case["hi"], 3 * 10**9 // token))
    elif kind == "shared":
        lo = _log(rng, 8, 512)
        case.update(groups=rng.randint(1, 10), members=_log(rng, 4, 40),
                    prefix=_log(rng, 256, 6000), lo=lo, hi=_log(rng, lo, 2048))
    elif kind == "prefill":
        lo = _log(rng, 16, 2048)
        case.update(layers=rng.randint(1, 2), chunks=rng.randint(1, 6), new_lo=lo,
                    new_hi=min(_log(rng, lo, 6000), 8 * lo),
                    cached_hi=rng.choice((0, _log(rng, 64, 6000))))
        case["chunks"] = max(1, min(case["chunks"], 12000 // case["new_hi"]))
        if case["dtype"] == "float32":  # the 32-bit matrix rate is a sixteenth of the 16-bit one
            case.update(layers=1, chunks=min(3, case["chunks"]), new_lo=min(lo, 500),
                        new_hi=min(case["new_hi"], 1000), cached_hi=min(case["cached_hi"], 1500))
    else:
        for k in ("hq", "hkv", "d", "dtype"):
            del case[k]
        lo = _log(rng, 64, 2048)
        case.update(decoder=rng.choice(sorted(DECODERS)), lo=lo, hi=_log(rng, lo, 4096))
        if kind == "block":
            case.update(layers=rng.randint(1, 4), rows=_log(rng, 1, 32))
        else:
            case.update(layers=rng.randint(4, 24), rows=rng.randint(1, 8),
                        vocab=_log(rng, 4000, 151936))
    return case


# ---- sizes: from the case alone ---------------------------------------------------------------

def _lengths(case):
    """Context lengths (cached + new) and new tokens of each row or chunk."""
    rng = random.Random(case["sizes"])
    kind = case["kind"]
    if kind == "request":
        return [case["cached"] + case["new"]], [case["new"]]
    if kind == "shared":
        n = case["groups"] * case["members"]
        whole = case["prefix"] // case["block"] * case["block"]
        return [whole + rng.randint(case["lo"], case["hi"]) for _ in range(n)], [1] * n
    if kind in ("prefill", "forward"):
        new = [_log(rng, case["new_lo"], case["new_hi"]) for _ in range(case["chunks"])]
        return [n + rng.randint(0, case["cached_hi"]) for n in new], new
    return [_log(rng, case["lo"], case["hi"]) for _ in range(case["rows"])], [1] * case["rows"]


def _heads(case):
    if "decoder" in case:
        c = DECODERS[case["decoder"]]
        return c["num_attention_heads"], c["num_key_value_heads"], c["head_dim"], torch.float16
    return case["hq"], case["hkv"], case["d"], getattr(torch, case["dtype"])


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(seed)


def _randn(gen, shape, dtype, std=1.0):
    out = torch.empty(shape, dtype=dtype, device=DEV)
    return out.normal_(0.0, std, generator=gen)


def _paged(case, seed):
    """Pools [layers, NB, BS, Hkv, D], int32 tables [rows, W] and lengths of a case."""
    ctx, new = _lengths(case)
    hq, hkv, d, dt = _heads(case)
    bs, layers = case["block"], case.get("layers", 1)
    gen, rng = _gen(seed), random.Random(seed)
    shared = 0
    if case["kind"] == "shared":
        shared = case["prefix"] // bs
    pages = [-(-n // bs) for n in ctx]
    need = sum(p - shared for p in pages) + shared * case.get("groups", 0)
    nb = need + max(1, need // 8)
    perm = list(range(nb))
    rng.shuffle(perm)
    at, rows = 0, []
    width = max(pages)
    for b, p in enumerate(pages):
        if shared and b % case["members"] == 0:
            prefix = perm[at:at + shared]
            at += shared
        row = (prefix if shared else []) + perm[at:at + p - shared]
        at += p - shared
        rows.append(row + [row[-1]] * (width - len(row)))
    return dict(
        case=case, ctx=ctx, new=new, bs=bs, layers=layers, hq=hq, hkv=hkv, d=d, dt=dt,
        k=_randn(gen, (layers, nb, bs, hkv, d), dt), v=_randn(gen, (layers, nb, bs, hkv, d), dt),
        tables=torch.tensor(rows, dtype=torch.int32, device=DEV), gen=gen,
        lens=torch.tensor(ctx, dtype=torch.int32, device=DEV))


def _attention_inputs(case, seed):
    s = _paged(case, seed)
    total, gen = sum(s["new"]), s["gen"]
    s["q"] = _randn(gen, (s["layers"], total, s["hq"], s["d"]), s["dt"])
    s["k_new"] = _randn(gen, (s["layers"], total, s["hkv"], s["d"]), s["dt"])
    s["v_new"] = _randn(gen, (s["layers"], total, s["hkv"], s["d"]), s["dt"])
    offs = [0]
    for n in s["new"]:
        offs.append(offs[-1] + n)
    s["offs"] = offs
    return s


# ---- decoder weights --------------------------------------------------------------------------

def _config(case):
    return Qwen2Config(num_hidden_layers=case["layers"], vocab_size=case.get("vocab", 1024),
                       **DECODERS[case["decoder"]])


def _layer_weights(cfg, gen):
    h, i, d = cfg.hidden_size, cfg.intermediate_size, cfg.head_dim
    nq, nqkv = cfg.num_attention_heads * d, (cfg.num_attention_heads + 2 * cfg.num_key_value_heads) * d
    f = torch.float16
    return dict(input_norm=1.0 + _randn(gen, (h,), f, 0.1), post_norm=1.0 + _randn(gen, (h,), f, 0.1),
                w_qkv=_randn(gen, (nqkv, h), f, 0.02), b_qkv=_randn(gen, (nqkv,), f, 0.2),
                w_o=_randn(gen, (h, nq), f, 0.02), w_gate_up=_randn(gen, (2 * i, h), f, 0.02),
                w_down=_randn(gen, (h, i), f, 0.02))


def _inv_freq(cfg):
    return 1.0 / cfg.rope_theta ** (
        torch.arange(0, cfg.head_dim, 2, device=DEV, dtype=torch.float32) / cfg.head_dim)


def _model(case, seed):
    """The model with weights of this file's own drawing, and its cache."""
    cfg = _config(case)
    model = Qwen2Model(cfg, DEV, seed=1)
    gen = _gen(seed + 1)
    for lw in model.layer_weights:
        for name, value in _layer_weights(cfg, gen).items():
            getattr(lw, name).copy_(value)
    model.embed.copy_(_randn(gen, tuple(model.embed.shape), torch.float16, 0.02))
    model.final_norm.copy_(1.0 + _randn(gen, tuple(model.final_norm.shape), torch.float16, 0.1))
    return model


def _model_sizes(case):
    """Context lengths, new tokens, and pool blocks: rows reserve their pages in turn."""
    ctx, new = _lengths(case)
    pages = [-(-n // case["block"]) for n in ctx]
    return ctx, new, pages


def _model_state(case, seed, capture=True):
    ctx, new, pages = _model_sizes(case)
    cfg = _config(case)
    scratch = 8 if case["kind"] == "model" else 0
    layout = CacheLayout(cfg.num_hidden_layers, sum(pages) + scratch, case["block"],
                         cfg.num_key_value_heads, cfg.head_dim)
    cache = PagedKVCache(layout, DEV, torch.float16)
    gen, rng = _gen(seed), random.Random(seed)
    cache.k.normal_(generator=gen)
    cache.v.normal_(generator=gen)
    model = _model(case, seed)
    step = GraphDecodeStep(model, cache, max_model_len=max(ctx)) if scratch else None
    chunks = []
    for b, (n, m) in enumerate(zip(ctx, new)):
        cache.reserve(f"r{b}", n)
        order = list(cache.tables[f"r{b}"])
        rng.shuffle(order)
        cache.tables[f"r{b}"] = order
        ids = [rng.randrange(cfg.vocab_size) for _ in range(m)]
        chunks.append(Chunk(f"r{b}", ids, n - m))
    if step is not None and capture:  # the engine captures its buckets when it starts
        step.manager.capture(step.manager.bucket_for(len(chunks)), step._decode,
                             step.graph_inputs(chunks, step.manager.bucket_for(len(chunks))))
    return dict(case=case, cache=cache, model=model, step=step, chunks=chunks)


def _block_layers(s):
    """The decode step's layers as the model runs them; returns the last (residual, normed)."""
    cfg, scale = s["cfg"], 1.0 / math.sqrt(s["d"])
    plan = ops.paged_decode_plan(s["tables"], s["lens"], s["k"].shape[1], s["hkv"], s["bs"])
    res, h = s["x"], s["h"]
    for layer, w in enumerate(s["weights"]):
        nxt = s["weights"][(layer + 1) % len(s["weights"])]["input_norm"]
        q, k, v = ops.gemm_rope(h, w["w_qkv"], w["b_qkv"], s["positions"], s["inv_freq"], s["hq"],
                                s["hkv"], s["d"])
        attn = ops.paged_decode(q, s["k"][layer], s["v"][layer], s["tables"], s["lens"],
                                scale=scale, k_new=k, v_new=v, plan=plan)
        r1, h2 = ops.gemm_resid_rmsnorm(attn.reshape(len(attn), -1), w["w_o"], res, w["post_norm"],
                                        cfg.rms_norm_eps)
        act = ops.gemm_silu(h2, w["w_gate_up"])
        res, h = ops.gemm_resid_rmsnorm(act, w["w_down"], r1, nxt, cfg.rms_norm_eps)
    return res, h


def _block_inputs(case, seed):
    s = _paged(case, seed)
    cfg, gen = _config(case), s["gen"]
    s.update(cfg=cfg, weights=[_layer_weights(cfg, gen) for _ in range(case["layers"])],
             x=_randn(gen, (case["rows"], cfg.hidden_size), torch.float16),
             h=_randn(gen, (case["rows"], cfg.hidden_size), torch.float16),
             positions=s["lens"].long() - 1, inv_freq=_inv_freq(cfg))
    return s


# ---- prepare and run --------------------------------------------------------------------------

def prepare(case, seed):
    kind = case["kind"]
    if kind in ("model", "forward"):
        return _model_state(case, seed)
    if kind == "block":
        s = _block_inputs(case, seed)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            _block_layers(s)
        torch.cuda.current_stream().wait_stream(side)
        torch.cuda.synchronize()
        s["graph"] = torch.cuda.CUDAGraph()
        with ops.hold_workspaces() as held, torch.cuda.graph(s["graph"]):
            s["out"] = _block_layers(s)
        s["held"] = list(held)
        return s
    s = _attention_inputs(case, seed)
    if kind == "request":
        layout = CacheLayout(1, s["k"].shape[1], s["bs"], s["hkv"], s["d"])
        s["cache"] = cache = PagedKVCache(layout, DEV, s["dt"])
        cache.k.copy_(s["k"])
        cache.v.copy_(s["v"])
        cache.reserve("r", s["ctx"][0])
        order = list(cache.tables["r"])
        random.Random(seed).shuffle(order)
        cache.tables["r"] = order
        s["positions"] = torch.arange(case["cached"], s["ctx"][0], device=DEV)
    elif kind == "batch":
        layout = CacheLayout(1, s["k"].shape[1], s["bs"], s["hkv"], s["d"])
        s["cache"] = cache = PagedKVCache(layout, DEV, s["dt"])
        cache.k, cache.v = s["k"], s["v"]
        s["tables64"] = s["tables"].long()
        s["positions"] = s["lens"].long() - 1
        s["mask"] = torch.ones(case["rows"], device=DEV)
    elif kind == "shared":
        n, m = case["groups"] * case["members"], case["members"]
        s["group_offsets"] = torch.arange(0, n + 1, m, dtype=torch.int32, device=DEV)
        s["prefix_lens"] = torch.full((case["groups"],), case["prefix"], dtype=torch.int32, device=DEV)
    elif kind == "prefill":
        s["q_offsets"] = torch.tensor(s["offs"], dtype=torch.int32, device=DEV)
    return s


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "model":
        return {"logits": s["step"](s["chunks"]), "k": s["cache"].k, "v": s["cache"].v}
    if kind == "forward":
        return {"logits": s["model"].forward(s["chunks"], s["cache"]), "k": s["cache"].k,
                "v": s["cache"].v}
    if kind == "block":
        s["graph"].replay()
        return {"out": s["out"], "k": s["k"], "v": s["v"]}
    if kind == "request":
        return attention.attention_for_request(s["q"][0], s["cache"], 0, "r", s["ctx"][0],
                                               s["positions"])
    if kind == "batch":
        out = attention.paged_decode_batch(s["q"][0], s["cache"], 0, s["tables64"], s["positions"],
                                           s["mask"], k_new=s["k_new"][0], v_new=s["v_new"][0])
        return {"out": out, "k": s["k"], "v": s["v"]}
    if kind == "shared":
        out = ops.paged_decode_shared_prefix(
            s["q"][0], s["k"][0], s["v"][0], s["tables"], s["lens"], s["group_offsets"],
            s["prefix_lens"], k_new=s["k_new"][0], v_new=s["v_new"][0])
        return {"out": out, "k": s["k"], "v": s["v"]}
    planned = s["dt"] != torch.float32
    outs = []
    if kind == "step":
        plan = ops.paged_decode_plan(s["tables"], s["lens"], s["k"].shape[1], s["hkv"],
                                     s["bs"]) if planned else None
        for i in range(s["layers"]):
            outs.append(ops.paged_decode(s["q"][i], s["k"][i], s["v"][i], s["tables"], s["lens"],
                                         k_new=s["k_new"][i], v_new=s["v_new"][i], plan=plan))
        return {"out": outs, "k": s["k"], "v": s["v"]}
    total = s["offs"][-1]
    plan = ops.prefill_paged_plan(s["q_offsets"], s["lens"], total, s["hq"], s["hkv"],
                                  s["tables"].shape[1], s["bs"]) if planned else None
    for i in range(s["layers"]):
        ops.write_kv_ragged(s["k_new"][i], s["v_new"][i], s["k"][i], s["v"][i], s["tables"],
                            s["q_offsets"], s["lens"])
        outs.append(ops.prefill_paged(s["q"][i], s["k"][i], s["v"][i], s["tables"], s["q_offsets"],
                                      s["lens"], max(s["new"]), plan=plan))
    return {"out": outs, "k": s["k"], "v": s["v"]}


# ---- work and tolerance -----------------------------------------------------------------------

def work(case):
    ctx, new = _lengths(case)
    hq, hkv, d, dt = _heads(case)
    e = 4 if dt == torch.float32 else 2
    layers, total = case.get("layers", 1), sum(new)
    pairs = sum(n * (c - n) + n * (n + 1) // 2 for c, n in zip(ctx, new))
    rows = sum(ctx)
    if case["kind"] == "shared":  # a group's prefix is read once
        whole = case["prefix"] // case["block"] * case["block"]
        rows = sum(c - whole for c in ctx) + case["groups"] * whole
    nbytes = rows * 2 * hkv * d * e + 2 * total * hq * d * e + 4 * sum(
        -(-c // case["block"]) for c in ctx)
    if case["kind"] != "request":
        nbytes += total * 2 * hkv * d * e  # the new rows' page write
    flops = 4 * hq * d * pairs
    if "decoder" in case:
        cfg = _config(case)
        h, i = cfg.hidden_size, cfg.intermediate_size
        weights = h * (2 * hq + 2 * hkv) * d + 3 * h * i
        nbytes += 2 * weights
        flops += 2 * total * weights
    nbytes, flops = nbytes * layers, flops * layers
    if "vocab" in case:
        nbytes += 2 * case["vocab"] * cfg.hidden_size + 2 * len(ctx) * case["vocab"]
        flops += 2 * len(ctx) * case["vocab"] * cfg.hidden_size
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # about four times the largest error against exact() over the listed cases: 2.4e-4 to 4.6e-4
    # (float16), 2.0e-3 to 2.3e-3 (bfloat16), 4.0e-7 to 4.4e-7 (float32), 9.4e-4 (block) and
    # 6.2e-3 (a whole model: rounding in 16 bits through 28 layers)
    if "decoder" in case:
        return {"rel": 4e-3} if case["kind"] == "block" else {"rel": 2.4e-2}
    return {"float16": {"rel": 2e-3}, "bfloat16": {"rel": 1e-2}, "float32": {"rel": 2e-6}}[
        case["dtype"]]


# ---- 64-bit values ----------------------------------------------------------------------------

def _attend(q, k, v, start):
    """Causal attention in 64 bits: q [n, Hq, D] at positions start.., k / v [L, Hkv, D]."""
    n, hq, d = q.shape
    group = hq // k.shape[1]
    out = torch.empty((n, hq, d), dtype=torch.float64, device=DEV)
    step = max(1, (1 << 26) // k.shape[0])
    for h in range(hq):
        kh = k[:, h // group].double().t().contiguous()
        vh = v[:, h // group].double().contiguous()
        for lo in range(0, n, step):
            hi = min(n, lo + step)
            s = q[lo:hi, h].double().contiguous() @ kh / math.sqrt(d)
            if n > 1:
                row = torch.arange(start + lo, start + hi, device=DEV)
                s.masked_fill_(torch.arange(k.shape[0], device=DEV)[None] > row[:, None], -math.inf)
            out[lo:hi, h] = torch.softmax(s, -1) @ vh
    return out


def _attend_one(q, k, v):
    """One row: q [Hq, D], k / v [L, Hkv, D]."""
    hq, d = q.shape
    hkv = k.shape[1]
    s = (q.double().reshape(1, hkv, hq // hkv, d) * k.double()[:, :, None]).sum(-1) / math.sqrt(d)
    p = torch.softmax(s, 0)
    return (p[..., None] * v.double()[:, :, None]).sum(0).reshape(hq, d)


def _rows(pool, table, n):
    """The first n rows of a sequence: [n, Hkv, D]."""
    pages = -(-n // pool.shape[1])
    return pool[table[:pages].long()].flatten(0, 1)[:n]


def _norm64(x, w, eps):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _rope64(x, positions, inv_freq):
    a = positions.double()[:, None] * inv_freq.double()[None]
    cos, sin = torch.cat([a.cos()] * 2, -1)[:, None], torch.cat([a.sin()] * 2, -1)[:, None]
    half = x.shape[-1] // 2
    return x * cos + torch.cat([-x[..., half:], x[..., :half]], -1) * sin


def _layer64(cfg, w, h, res, positions, inv_freq, next_norm, attend):
    nq, nk, d = cfg.num_attention_heads, cfg.num_key_value_heads, cfg.head_dim
    qkv = h @ w["w_qkv"].double().t() + w["b_qkv"].double()
    q, k, v = qkv.split([nq * d, nk * d, nk * d], -1)
    q = _rope64(q.reshape(-1, nq, d), positions, inv_freq)
    k = _rope64(k.reshape(-1, nk, d), positions, inv_freq)
    a = attend(q, k, v.reshape(-1, nk, d))
    r1 = res + a.reshape(len(h), -1) @ w["w_o"].double().t()
    h2 = _norm64(r1, w["post_norm"], cfg.rms_norm_eps)
    g, u = (h2 @ w["w_gate_up"].double().t()).chunk(2, -1)
    r2 = r1 + (torch.nn.functional.silu(g) * u) @ w["w_down"].double().t()
    return r2, _norm64(r2, next_norm, cfg.rms_norm_eps)


def _attend_cached(k_pool, v_pool, tables, ctx, new):
    """An attend() of _layer64: each chunk's new K/V rows after the cached ones."""
    def attend(q, k, v):
        out, at = torch.empty_like(q), 0
        for b, (c, n) in enumerate(zip(ctx, new)):
            old = c - n
            kk, vv = k[at:at + n], v[at:at + n]
            if old:
                kk = torch.cat([_rows(k_pool, tables[b], old).double(), kk])
                vv = torch.cat([_rows(v_pool, tables[b], old).double(), vv])
            out[at:at + n] = (_attend_one(q[at], kk, vv)[None] if n == 1
                              else _attend(q[at:at + n], kk, vv, old))
            at += n
        return out
    return attend


def exact(case, seed):
    kind = case["kind"]
    if kind == "block":
        s = _block_inputs(case, seed)
        res, h = s["x"].double(), s["h"].double()
        for i, w in enumerate(s["weights"]):
            nxt = s["weights"][(i + 1) % len(s["weights"])]["input_norm"]
            attend = _attend_cached(s["k"][i], s["v"][i], s["tables"], s["ctx"], s["new"])
            res, h = _layer64(s["cfg"], w, h, res, s["positions"], s["inv_freq"], nxt, attend)
        return {"out": (res, h), "k": None, "v": None}
    if kind in ("model", "forward"):
        s = _model_state(case, seed, capture=False)
        cfg, model, cache, chunks = s["model"].cfg, s["model"], s["cache"], s["chunks"]
        ctx, new, _ = _model_sizes(case)
        tables = [torch.tensor(cache.tables[c.request_id], device=DEV) for c in chunks]
        ids = torch.tensor([t for c in chunks for t in c.input_ids], device=DEV)
        positions = torch.tensor([p for c in chunks for p in range(c.start, c.start + len(c.input_ids))],
                                 device=DEV)
        res = model.embed[ids].double()
        layers = [vars(lw) for lw in model.layer_weights]
        h = _norm64(res, layers[0]["input_norm"], cfg.rms_norm_eps)
        for i, w in enumerate(layers):
            nxt = layers[i + 1]["input_norm"] if i + 1 < len(layers) else model.final_norm
            attend = _attend_cached(cache.k[i], cache.v[i], tables, ctx, new)
            res, h = _layer64(cfg, w, h, res, positions, _inv_freq(cfg), nxt, attend)
        ends = torch.tensor(new, device=DEV).cumsum(0) - 1
        logits = h[ends] @ model.lm_head.double().t()
        return {"logits": list(logits), "k": None, "v": None}
    s = _attention_inputs(case, seed)
    if kind == "request":
        order = list(range(-(-s["ctx"][0] // s["bs"])))
        random.Random(seed).shuffle(order)
        s["tables"] = torch.tensor([order], device=DEV)
    outs = []
    for i in range(s["layers"]):
        k, v = s["k"][i], s["v"][i]
        if kind != "request":
            for b, (c, n) in enumerate(zip(s["ctx"], s["new"])):
                at = torch.arange(c - n, c, device=DEV)
                blk = s["tables"][b].long()[at // s["bs"]]
                k[blk, at % s["bs"]] = s["k_new"][i, s["offs"][b]:s["offs"][b + 1]]
                v[blk, at % s["bs"]] = s["v_new"][i, s["offs"][b]:s["offs"][b + 1]]
        out = torch.empty(s["q"][i].shape, dtype=torch.float64, device=DEV)
        for b, (c, n) in enumerate(zip(s["ctx"], s["new"])):
            lo, hi = s["offs"][b], s["offs"][b + 1]
            kk, vv = _rows(k, s["tables"][b], c), _rows(v, s["tables"][b], c)
            out[lo:hi] = (_attend_one(s["q"][i, lo], kk, vv)[None] if n == 1
                          else _attend(s["q"][i, lo:hi], kk, vv, c - n))
        outs.append(out)
    if kind == "request":
        return outs[0]
    if kind in ("batch", "shared"):
        return {"out": outs[0], "k": None, "v": None}
    return {"out": outs, "k": None, "v": None}
