"""GPU: ragged chunked-prefill attention (fe_prefill_paged) against the oracle."""
from __future__ import annotations

import math

import numpy as np
import pytest
import torch

from flexengine_amd import _lib, attention, ops, workloads
from flexengine_amd.kv_cache import CacheLayout, PagedKVCache
from oracle import paged_ref as R
from tests.parity import assert_attention_close

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _case(seed, n_new, cached, hq=12, hkv=2, d=128, bs=16):
    g = torch.Generator().manual_seed(seed)
    ctx = [c + n for c, n in zip(cached, n_new)]
    pages = [math.ceil(x / bs) for x in ctx]
    nb = sum(pages) + 3
    k_pool = torch.randn(nb, bs, hkv, d, generator=g).half()
    v_pool = torch.randn(nb, bs, hkv, d, generator=g).half()
    perm = torch.randperm(nb, generator=g)
    width = max(pages)
    tables = torch.zeros(len(ctx), width, dtype=torch.int32)
    at = 0
    for i, p in enumerate(pages):
        tables[i, :p] = perm[at:at + p]
        tables[i, p:] = perm[at + p - 1] if p else 0
        at += p
    offs = np.concatenate([[0], np.cumsum(n_new)]).astype(np.int32)
    q = torch.randn(int(offs[-1]), hq, d, generator=g).half()
    return q, torch.tensor(offs), torch.tensor(ctx, dtype=torch.int32), tables, k_pool, v_pool


def _form(q, k, t, new, planned=False):
    """The kernel a prefill of these tensors runs on."""
    return ops.prefill_form(len(new), q.shape[0], max(new), q.shape[1], k.shape[2], k.shape[3],
                            k.shape[1], t.shape[1], q.dtype, planned=planned)


def _run(q, offs, ctx, tables, kp, vp):
    n_new = (offs[1:] - offs[:-1]).tolist()
    out = ops.prefill_paged(q.to(DEV), kp.to(DEV), vp.to(DEV), tables.to(DEV), offs.to(DEV),
                            ctx.to(DEV), max(n_new) if n_new else 0)
    torch.cuda.synchronize()
    return out.cpu().numpy()


@pytest.mark.parametrize("n_new,cached", [([1], [0]), ([5], [0]), ([16], [0]), ([17], [3]),
                                          ([64], [0]), ([65], [100]), ([130, 7, 1], [0, 40, 999]),
                                          ([0, 33], [10, 10])])
def test_ragged_prefill_small(n_new, cached):
    q, offs, ctx, tables, kp, vp = _case(sum(n_new) + 7 * len(n_new), n_new, cached)
    got = _run(q, offs, ctx, tables, kp, vp)
    exp = R.prefill_reference(q.numpy(), offs.numpy(), ctx.numpy(), kp.numpy(), vp.numpy(),
                              tables.numpy(), 16)
    assert_attention_close(got, exp, what=f"n={n_new} c={cached}")


@pytest.mark.parametrize("hq,hkv,d,bs", [(14, 2, 64, 16), (8, 8, 64, 4), (16, 2, 128, 32)])
def test_prefill_shapes(hq, hkv, d, bs):
    q, offs, ctx, tables, kp, vp = _case(hq + d + bs, [70, 3], [25, 200], hq, hkv, d, bs)
    got = _run(q, offs, ctx, tables, kp, vp)
    exp = R.prefill_reference(q.numpy(), offs.numpy(), ctx.numpy(), kp.numpy(), vp.numpy(),
                              tables.numpy(), bs)
    assert_attention_close(got, exp)


@pytest.mark.parametrize("hq,hkv,d,q_scale", [(6, 1, 128, 16.0), (12, 2, 128, 8.0), (14, 2, 64, 16.0)])
def test_prefill_large_scores(hq, hkv, d, q_scale):
    """q scaled up so scores spread over hundreds: the running max must be the true
    max over every key of a block (all four 16-lane rows of the score tile); a max
    taken over part of them lets exp2 and the fp16 probabilities overflow."""
    q, offs, ctx, tables, kp, vp = _case(77 + hq, [40, 130, 1], [300, 20, 64], hq, hkv, d)
    q = (q.float() * q_scale).half()
    got = _run(q, offs, ctx, tables, kp, vp)
    assert np.isfinite(got).all()
    exp = R.prefill_reference(q.numpy(), offs.numpy(), ctx.numpy(), kp.numpy(), vp.numpy(),
                              tables.numpy(), 16)
    assert_attention_close(got, exp, what=f"large scores x{q_scale}")


def test_c4_prefill_chunks_full():
    w = workloads.c4_workload()
    got = _run(w.q, w.q_offsets, w.context_lens, w.block_tables, w.k_pool, w.v_pool)
    exp = R.prefill_reference(w.q.numpy(), w.q_offsets.numpy(), w.context_lens.numpy(),
                              w.k_pool.numpy(), w.v_pool.numpy(), w.block_tables.numpy(), 16)
    assert_attention_close(got, exp, what="C4 prefill")


def test_c4_decode_rows_full():
    """C4's 48 decode rows (L ~ U{256..4096}) in the same pool as the prefill chunks,
    through the decode kernel, against the float64 oracle."""
    w = workloads.c4_workload().decode
    d = w.to(DEV)
    got = ops.paged_decode(d.q, d.k_pool, d.v_pool, d.block_tables, d.context_lens)
    torch.cuda.synchronize()
    exp = R.decode_reference(w.q.numpy(), w.k_pool.numpy(), w.v_pool.numpy(),
                             w.block_tables.numpy(), w.context_lens.numpy(), 16)
    assert_attention_close(got.cpu().numpy(), exp, what="C4 decode rows")


def test_c4_whole_step_prefill_and_decode_share_the_pool():
    """The whole C4 step as the benchmark runs it: the prefill launch over the four
    chunks, then the decode launch over the 48 rows, back to back on one stream."""
    w = workloads.c4_workload()
    d = w.to(DEV)
    pre = ops.prefill_paged(d.q, d.k_pool, d.v_pool, d.block_tables, d.q_offsets,
                            d.context_lens, int(max(w.meta["n_new"])))
    dd = d.decode
    dec = ops.paged_decode(dd.q, d.k_pool, d.v_pool, dd.block_tables, dd.context_lens)
    torch.cuda.synchronize()
    exp_pre = R.prefill_reference(w.q.numpy(), w.q_offsets.numpy(), w.context_lens.numpy(),
                                  w.k_pool.numpy(), w.v_pool.numpy(), w.block_tables.numpy(), 16)
    exp_dec = R.decode_reference(w.decode.q.numpy(), w.k_pool.numpy(), w.v_pool.numpy(),
                                 w.decode.block_tables.numpy(), w.decode.context_lens.numpy(), 16)
    assert_attention_close(pre.cpu().numpy(), exp_pre, what="C4 step: prefill")
    assert_attention_close(dec.cpu().numpy(), exp_dec, what="C4 step: decode rows")


def test_per_request_interface_multi_token_chunk():
    """attention_for_request with Q > 1 takes the prefill kernel (the reference routes it to
    the materialized SDPA, test_triton_paged_attention.py:29-41); compare with the oracle."""
    g = torch.Generator().manual_seed(29)
    cache = PagedKVCache(CacheLayout(1, 8, 4, 1, 64), device=DEV)
    cache.reserve("r", 4)
    keys = torch.randn(4, 1, 64, generator=g).half()
    cache.write(0, "r", 0, keys.to(DEV), keys.to(DEV))
    query = torch.randn(4, 2, 64, generator=g).half()
    positions = torch.arange(4, device=DEV)
    got = attention.attention_for_request(query.to(DEV), cache, 0, "r", 4, positions)
    exp = R.attention_materialized(query.numpy(), keys.numpy(), keys.numpy(), np.arange(4))
    assert_attention_close(got.cpu().numpy(), exp)


def test_prefill_then_decode_consistency():
    """The prefill row at position p equals a decode call with context p + 1."""
    q, offs, ctx, tables, kp, vp = _case(5, [40], [60])
    got = _run(q, offs, ctx, tables, kp, vp)
    j = 23
    pos = 60 + j
    dec = ops.paged_decode(q[j:j + 1].to(DEV), kp.to(DEV), vp.to(DEV), tables.to(DEV),
                           torch.tensor([pos + 1], dtype=torch.int32, device=DEV)).cpu().numpy()
    assert np.abs(got[j] - dec[0].astype(np.float64)).max() <= 2e-3


def test_split_prefill_repeated_calls_and_shapes_share_the_workspace():
    """The key-split merge leaves its tickets at zero: repeated calls of different
    shapes on the shared workspace give the same results each time."""
    a = _case(3, [130, 7, 1], [0, 40, 999])
    b = _case(4, [65], [100])
    first_a, first_b = _run(*a), _run(*b)
    for _ in range(3):
        np.testing.assert_array_equal(_run(*a), first_a)
        np.testing.assert_array_equal(_run(*b), first_b)


def test_stream_k_merge_is_deterministic_whoever_merges():
    """A split unit is merged by whichever contributor draws the last ticket, from its
    registers or from memory: the result must not depend on which (same bits on every
    call), and must match the oracle.  C4 splits nearly every unit; 12 calls on 4
    rotating pool copies vary the timing."""
    w = workloads.c4_workload()
    d = w.to(DEV)
    max_q = int((w.q_offsets[1:] - w.q_offsets[:-1]).max())
    pools = [(d.k_pool, d.v_pool)] + [(d.k_pool.clone(), d.v_pool.clone()) for _ in range(3)]
    outs = []
    for i in range(12):
        kp, vp = pools[i % 4]
        outs.append(ops.prefill_paged(d.q, kp, vp, d.block_tables, d.q_offsets, d.context_lens,
                                      max_q))
    torch.cuda.synchronize()
    for i, o in enumerate(outs[1:], 1):
        assert torch.equal(o, outs[0]), f"call {i} differs from call 0"
    exp = R.prefill_reference(w.q.numpy(), w.q_offsets.numpy(), w.context_lens.numpy(),
                              w.k_pool.numpy(), w.v_pool.numpy(), w.block_tables.numpy(), 16)
    assert_attention_close(outs[0].cpu().numpy(), exp, what="C4 repeated")


# --------------------------------------------------------------------------------------
# prefill plan (fe_prefill_plan / fe_prefill_paged_planned): one plan per model step,
# reused by every layer; results must be bit-identical to the unplanned launch
# --------------------------------------------------------------------------------------

def _planned_prefill_cases():
    w = workloads.c4_workload()
    c4 = (w.q, w.q_offsets, w.context_lens, w.block_tables, w.k_pool, w.v_pool, 16)
    small = _case(61, [130, 7, 1], [0, 40, 999]) + (16,)
    bs32 = _case(62, [70, 3], [25, 200], 16, 2, 128, 32) + (32,)
    d64 = _case(63, [300, 1, 45], [0, 2048, 17], 14, 2, 64, 16) + (16,)
    return {"C4": c4, "small": small, "bs32": bs32, "d64-g7": d64}


@pytest.mark.parametrize("name", ["C4", "small", "bs32", "d64-g7"])
def test_planned_prefill_is_bit_identical_and_reusable(name):
    q, offs, ctx, tables, kp, vp, bs = _planned_prefill_cases()[name]
    print(f"planned prefill case {name}", flush=True)
    hq, hkv = q.shape[1], kp.shape[2]
    offs_d, ctx_d, tables_d = offs.to(DEV), ctx.to(DEV), tables.to(DEV)
    max_q = int((offs[1:] - offs[:-1]).max())
    plan = ops.prefill_paged_plan(offs_d, ctx_d, q.shape[0], hq, hkv, tables.shape[1], bs)
    assert plan is not None
    # three "layers": own pools and queries, the same offsets, lengths and tables
    for layer in range(3):
        g = torch.Generator().manual_seed(200 + layer)
        ql = torch.randn(q.shape, generator=g).half().to(DEV)
        kl = torch.randn(kp.shape, generator=g).half().to(DEV)
        vl = torch.randn(vp.shape, generator=g).half().to(DEV)
        ref = ops.prefill_paged(ql, kl, vl, tables_d, offs_d, ctx_d, max_q)
        got = ops.prefill_paged(ql, kl, vl, tables_d, offs_d, ctx_d, max_q, plan=plan)
        torch.cuda.synchronize()
        assert torch.equal(got, ref), f"{name} layer {layer}: planned output differs"
    got = ops.prefill_paged(q.to(DEV), kp.to(DEV), vp.to(DEV), tables_d, offs_d, ctx_d, max_q,
                            plan=plan)
    exp = R.prefill_reference(q.numpy(), offs.numpy(), ctx.numpy(), kp.numpy(), vp.numpy(),
                              tables.numpy(), bs)
    assert_attention_close(got.cpu().numpy(), exp, what=f"planned {name}")


def test_planned_prefill_bf16_and_refusals():
    """The bf16 planned form matches the bf16 unplanned one bit for bit; a plan for other
    tensors is refused; block sizes the stream-K kernel does not take have no plan."""
    q, offs, ctx, tables, kp, vp, bs = _planned_prefill_cases()["small"]
    qb, kb, vb = (t.float().to(torch.bfloat16).to(DEV) for t in (q, kp, vp))
    offs_d, ctx_d, tables_d = offs.to(DEV), ctx.to(DEV), tables.to(DEV)
    max_q = int((offs[1:] - offs[:-1]).max())
    plan = ops.prefill_paged_plan(offs_d, ctx_d, q.shape[0], q.shape[1], kp.shape[2],
                                  tables.shape[1], bs)
    ref = ops.prefill_paged(qb, kb, vb, tables_d, offs_d, ctx_d, max_q)
    got = ops.prefill_paged(qb, kb, vb, tables_d, offs_d, ctx_d, max_q, plan=plan)
    torch.cuda.synchronize()
    assert got.dtype == torch.bfloat16 and torch.equal(got, ref)
    with pytest.raises(ValueError, match="other q_offsets"):
        ops.prefill_paged(qb, kb, vb, tables_d, offs_d, ctx_d.clone(), max_q, plan=plan)
    q4, offs4, ctx4, tables4, _, _ = _case(64, [20], [7], 8, 8, 64, 4)
    assert ops.prefill_paged_plan(offs4.to(DEV), ctx4.to(DEV), q4.shape[0], 8, 8,
                                  tables4.shape[1], 4) is None
    small = torch.empty(16, dtype=torch.uint8, device=DEV)
    rc = _lib.load().fe_prefill_plan(offs_d.data_ptr(), ctx_d.data_ptr(), ctx.shape[0],
                                     q.shape[0], q.shape[1], kp.shape[2], tables.shape[1], bs,
                                     small.data_ptr(), small.numel(), None)
    assert rc == _lib.FE_ERR_WORKSPACE


def test_planned_prefill_checks_its_plan_and_leaves_tickets_clean():
    """A plan for other tensors (a clone of context_lens, same contents) and a stale plan
    (a length changed in place after the plan call) are not used: every row NaN and the
    error word set, before any split unit's ticket is taken -- so the unplanned and
    freshly planned launches that follow are exact."""
    q, offs, ctx, tables, kp, vp, bs = _planned_prefill_cases()["small"]  # lengths 130, 47, 1000
    hq, hkv, d = q.shape[1], kp.shape[2], q.shape[2]
    qd, kd, vd = q.to(DEV), kp.to(DEV), vp.to(DEV)
    offs_d, ctx_d, tables_d = offs.to(DEV), ctx.to(DEV), tables.to(DEV)
    max_q = int((offs[1:] - offs[:-1]).max())
    plan = ops.prefill_paged_plan(offs_d, ctx_d, q.shape[0], hq, hkv, tables.shape[1], bs)
    need = int(_lib.load().fe_prefill_workspace_size(ctx.shape[0], q.shape[0], hq, hkv, d))
    ws = torch.zeros(need, dtype=torch.uint8, device=DEV)
    out = torch.zeros_like(qd)
    rc = _lib.load().fe_prefill_paged_planned(
        qd.data_ptr(), out.data_ptr(), kd.data_ptr(), vd.data_ptr(), kp.shape[0],
        tables_d.data_ptr(), tables.shape[1], offs_d.data_ptr(), ctx_d.clone().data_ptr(),
        ctx.shape[0], q.shape[0], max_q, hq, hkv, d, bs, 1.0 / math.sqrt(d), ws.data_ptr(),
        need, plan.buffer.data_ptr(), plan.buffer.numel(),
        torch.cuda.current_stream().cuda_stream)
    assert rc == _lib.FE_OK
    torch.cuda.synchronize()
    assert torch.isnan(out).all() and ops.plan_error(plan) == ops.PLAN_ERR_SIZES
    ctx_d[1] += 1                                              # 47 -> 48, same page count
    got = ops.prefill_paged(qd, kd, vd, tables_d, offs_d, ctx_d, max_q, plan=plan)
    torch.cuda.synchronize()
    assert torch.isnan(got).all() and ops.plan_error(plan) == ops.PLAN_ERR_STALE
    ref = ops.prefill_paged(qd, kd, vd, tables_d, offs_d, ctx_d, max_q)
    ops.prefill_paged_plan(offs_d, ctx_d, q.shape[0], hq, hkv, tables.shape[1], bs, out=plan)
    got = ops.prefill_paged(qd, kd, vd, tables_d, offs_d, ctx_d, max_q, plan=plan)
    torch.cuda.synchronize()
    assert ops.plan_error(plan) == 0 and torch.equal(got, ref)
    ctx2 = ctx.clone()
    ctx2[1] += 1
    exp = R.prefill_reference(q.numpy(), offs.numpy(), ctx2.numpy(), kp.numpy(), vp.numpy(),
                              tables.numpy(), bs)
    assert_attention_close(got.cpu().numpy(), exp, what="after a refused plan")


@pytest.mark.parametrize("dtype,max_tol,mean_tol", [(torch.float16, 2e-3, 2e-4),
                                                    (torch.bfloat16, 1.6e-2, 1.6e-3)])
@pytest.mark.parametrize("new,cached,hq,hkv,d,bs", [
    ([1, 2, 31], [0, 3, 0], 12, 2, 128, 16),          # fewer rows than one wave's 32
    ([63, 64, 65, 1], [0, 0, 1, 130], 4, 4, 64, 16),  # block edges, one head a group
    ([300], [17], 32, 8, 128, 32),                    # waves whose rows end before others'
    ([43, 0, 44], [0, 50, 5], 12, 2, 128, 16),        # 258 rows: a second row block of two
    ([1500, 700], [0, 40], 14, 2, 64, 64),            # several row blocks, group 7
    ([4200], [0], 16, 2, 128, 16),                    # more than 64 key blocks: ids reloaded
    ([260], [0], 71, 1, 64, 16),                      # a group above a wave's rows
])
def test_prefill_rows_of_fresh_prompts_match_float64(dtype, max_tol, mean_tol, new, cached, hq, hkv,
                                                     d, bs):
    """Short and fresh prefills (the wide kernel), unplanned and planned, against float64;
    the plan changes no bit."""
    g = torch.Generator().manual_seed(sum(new) + hq)
    ctx = [n + c for n, c in zip(new, cached)]
    pages = [-(-c // bs) for c in ctx]
    nb, width = sum(pages) + 2, max(pages)
    perm = torch.randperm(nb, generator=g).to(torch.int32)
    tables, at = torch.zeros((len(new), width), dtype=torch.int32), 0
    for s, p in enumerate(pages):
        tables[s, :p] = perm[at:at + p]
        at += p
    k = torch.randn(nb, bs, hkv, d, generator=g).to(dtype).to(DEV)
    v = torch.randn(nb, bs, hkv, d, generator=g).to(dtype).to(DEV)
    q = torch.randn(sum(new), hq, d, generator=g).to(dtype).to(DEV)
    offs = [0]
    for n in new:
        offs.append(offs[-1] + n)
    o = torch.tensor(offs, dtype=torch.int32, device=DEV)
    c = torch.tensor(ctx, dtype=torch.int32, device=DEV)
    t = tables.to(DEV)
    assert _form(q, k, t, new) == "wide"
    got = ops.prefill_paged(q, k, v, t, o, c, max(new))
    plan = ops.prefill_paged_plan(o, c, sum(new), hq, hkv, width, bs)
    assert torch.equal(ops.prefill_paged(q, k, v, t, o, c, max(new), plan=plan), got)
    assert ops.plan_error(plan) == 0
    for s, (n, x) in enumerate(zip(new, ctx)):
        kk = k[tables[s, :pages[s]].long()].flatten(0, 1)[:x].double()
        vv = v[tables[s, :pages[s]].long()].flatten(0, 1)[:x].double()
        for h in sorted({0, hq // 2, hq - 1}):
            kh, vh = kk[:, h * hkv // hq].t().contiguous(), vv[:, h * hkv // hq].contiguous()
            sc = q[offs[s]:offs[s + 1], h].double().contiguous() @ kh / d ** 0.5
            sc.masked_fill_(torch.arange(x, device=DEV)[None] >
                            torch.arange(x - n, x, device=DEV)[:, None], float("-inf"))
            err = (got[offs[s]:offs[s + 1], h].double() - torch.softmax(sc, -1) @ vh).abs()
            assert n == 0 or (err.max() <= max_tol and err.mean() <= mean_tol), (s, h, err.max())


def test_wide_prefill_counts_probabilities_below_the_smallest_normal():
    """One key far above thousands of equal ones: their probabilities (5.8e-5) are subnormal in
    fp16 and carry a fifth of the row's sum.  An error bound: probabilities to half a step of
    2^-24 (5.2e-4) in the numerator and the sum, the output to 2^-11."""
    bs, hq, hkv, d, n, gap = 16, 12, 2, 128, 4096, 9.75
    q = torch.zeros(n, hq, d)
    q[..., 0] = d ** 0.5
    k, v = torch.zeros(n // bs, bs, hkv, d), torch.ones(n // bs, bs, hkv, d)
    k[0, 0, :, 0], v[0, 0] = gap, 0.0
    q, k, v = (x.half().to(DEV) for x in (q, k, v))
    t = torch.arange(n // bs, dtype=torch.int32, device=DEV)[None].contiguous()
    o = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    c = torch.tensor([n], dtype=torch.int32, device=DEV)
    assert _form(q, k, t, [n]) == "wide"
    got = ops.prefill_paged(q, k, v, t, o, c, n).double()
    top = float(q[0, 0, 0].double() * k[0, 0, 0, 0].double()) / d ** 0.5
    tail = torch.arange(n, device=DEV).double()[:, None, None] * math.exp(-top)
    exp = tail / (1.0 + tail)
    assert ((got - exp).abs() <= (2 * 5.2e-4 + 2.0 ** -11) * exp + 2.0 ** -25).all()


@pytest.mark.parametrize("d,dtype", [(128, torch.float16), (64, torch.bfloat16)])
def test_wide_prefill_never_uses_rows_past_a_context(d, dtype):
    """NaN in every pool row past the contexts (the last page's tail, unused pages) leaves
    the wide kernel's result as it is, bit for bit."""
    bs, hq, hkv, new = 16, 12, 2, [700, 75]
    pages = [-(-n // bs) for n in new]
    g = torch.Generator().manual_seed(d)
    k = torch.randn(sum(pages) + 3, bs, hkv, d, generator=g).to(dtype).to(DEV)
    v = torch.randn(sum(pages) + 3, bs, hkv, d, generator=g).to(dtype).to(DEV)
    q = torch.randn(sum(new), hq, d, generator=g).to(dtype).to(DEV)
    t = torch.full((2, pages[0] + 1), sum(pages) + 2, dtype=torch.int32)
    t[0, :pages[0]] = torch.arange(pages[0])
    t[1, :pages[1]] = pages[0] + torch.arange(pages[1])
    t = t.to(DEV)
    o = torch.tensor([0, new[0], sum(new)], dtype=torch.int32, device=DEV)
    c = torch.tensor(new, dtype=torch.int32, device=DEV)
    assert _form(q, k, t, new) == "wide"
    good = ops.prefill_paged(q, k, v, t, o, c, max(new))
    for pool in (k, v):
        pool[sum(pages):] = float("nan")
        pool[pages[0] - 1, new[0] % bs:] = float("nan")
        pool[sum(pages) - 1, new[1] % bs:] = float("nan")
    assert torch.equal(ops.prefill_paged(q, k, v, t, o, c, max(new)), good)
    assert good.isfinite().all()


def test_wide_prefill_refuses_a_stale_plan():
    """The wide kernel checks a plan as the stream-K kernel does: changed lengths give NaN in
    the whole output and the stale word, other sizes the sizes word."""
    bs, hq, hkv, d, n = 16, 12, 2, 128, 700
    pages = n // bs + 1
    k = torch.randn(pages, bs, hkv, d, device=DEV).half()
    v, q = torch.randn_like(k), torch.randn(n, hq, d, device=DEV).half()
    t = torch.arange(pages, dtype=torch.int32, device=DEV)[None].contiguous()
    o = torch.tensor([0, n], dtype=torch.int32, device=DEV)
    c = torch.tensor([n], dtype=torch.int32, device=DEV)
    assert _form(q, k, t, [n], planned=True) == "wide"
    plan = ops.prefill_paged_plan(o, c, n, hq, hkv, pages, bs)
    good = ops.prefill_paged(q, k, v, t, o, c, n, plan=plan)
    c.add_(1)
    bad = ops.prefill_paged(q, k, v, t, o, c, n, plan=plan)
    assert bad.isnan().all() and ops.plan_error(plan) == ops.PLAN_ERR_STALE
    c.sub_(1)
    plan.buffer[64:68].zero_()   # the key's low word
    bad = ops.prefill_paged(q, k, v, t, o, c, n, plan=plan)
    assert bad.isnan().all() and ops.plan_error(plan) == ops.PLAN_ERR_SIZES
    plan = ops.prefill_paged_plan(o, c, n, hq, hkv, pages, bs)
    assert torch.equal(ops.prefill_paged(q, k, v, t, o, c, n, plan=plan), good)


def _device_case(new, cached, hq, hkv, d, bs, dtype, seed, width=None):
    """q, pools, tables (width pages, the longest context's by default), offsets and lengths of
    a ragged prefill on the GPU, and its offsets and lengths as lists."""
    g = torch.Generator().manual_seed(seed)
    ctx = [n + c for n, c in zip(new, cached)]
    pages = [-(-c // bs) for c in ctx]
    nb = sum(pages) + 2
    perm = torch.randperm(nb, generator=g).to(torch.int32)
    tables, at = torch.full((len(new), width or max(pages)), int(perm[-1]), dtype=torch.int32), 0
    for s, p in enumerate(pages):
        tables[s, :p] = perm[at:at + p]
        at += p
    k, v = (torch.randn(nb, bs, hkv, d, generator=g).to(dtype).to(DEV) for _ in range(2))
    q = torch.randn(sum(new), hq, d, generator=g).to(dtype).to(DEV)
    offs = [0] + np.cumsum(new).tolist()
    return (q, k, v, tables.to(DEV), torch.tensor(offs, dtype=torch.int32, device=DEV),
            torch.tensor(ctx, dtype=torch.int32, device=DEV), offs, ctx)


def _heads_float64(q, k, v, t, offs, ctx, heads):
    """(sequence, head, rows, scores [n, ctx] with the causal mask, V [ctx, D]) in float64."""
    bs, hkv, d = k.shape[1:]
    hq = q.shape[1]
    for s, x in enumerate(ctx):
        n = offs[s + 1] - offs[s]
        if n == 0:
            continue
        pages = t[s, :-(-x // bs)].long()
        causal = torch.arange(x, device=DEV)[None] > torch.arange(x - n, x, device=DEV)[:, None]
        for h in heads:
            kh = k[pages][:, :, h * hkv // hq].reshape(-1, d)[:x].double()
            vh = v[pages][:, :, h * hkv // hq].reshape(-1, d)[:x].double()
            sc = q[offs[s]:offs[s + 1], h].double() @ kh.t().contiguous() / d ** 0.5
            yield s, h, slice(offs[s], offs[s + 1]), sc.masked_fill_(causal, float("-inf")), vh


@pytest.mark.parametrize("form,dtype,new,cached,hq,hkv,d,bs", [
    ("wide", torch.bfloat16, [500], [0], 12, 2, 128, 16),           # a fresh prompt
    ("wide", torch.bfloat16, [64] * 6, [500] * 6, 12, 2, 128, 16),  # chunks over cached tokens
    ("wide", torch.float16, [100] * 16, [100] * 16, 14, 2, 64, 32),
    ("stream", torch.float16, [100], [1000], 12, 2, 128, 16),       # several blocks a range
    ("stream", torch.bfloat16, [16], [4000], 32, 8, 128, 16),
    ("stream", torch.float16, [90, 40], [3000, 2500], 14, 2, 64, 16),
])
def test_prefill_rounds_probabilities_relative_to_each_blocks_own_maximum(form, dtype, new, cached,
                                                                        hq, hkv, d, bs):
    """The error against 64 bits is no larger than with the probabilities of every 64-key block
    rounded to 16 bits relative to that block's own maximum and all else exact.  (One maximum
    per row, the first block's, is 2.5-10% worse.)  The bound's 0.5%: fp32 scores and sums move
    a probability across a rounding boundary now and then."""
    q, k, v, t, o, c, offs, ctx = _device_case(new, cached, hq, hkv, d, bs, dtype, sum(new) + d)
    assert _form(q, k, t, new) == form
    got = ops.prefill_paged(q, k, v, t, o, c, max(new)).double()
    err = emu = 0.0
    for _, h, rows, sc, vh in _heads_float64(q, k, v, t, offs, ctx, range(hq)):
        want = torch.softmax(sc, -1) @ vh
        m = torch.stack([b.max(-1).values for b in sc.split(64, -1)], -1)
        top = m.max(-1, keepdim=True).values
        num, den = torch.zeros_like(want), torch.zeros(len(want), 1, device=DEV).double()
        for j, b in enumerate(sc.split(64, -1)):
            mj = m[:, j:j + 1].clamp_min(-1e30)
            p = torch.exp(b - mj).to(dtype).double()
            w = torch.exp(mj - top)
            num += w * (p @ vh[64 * j:64 * (j + 1)])
            den += w * p.sum(-1, keepdim=True)
        err += (got[rows, h] - want).square().sum().item()
        emu += ((num / den).to(dtype).double() - want).square().sum().item()
    assert err ** 0.5 <= 1.005 * emu ** 0.5, (err ** 0.5, emu ** 0.5)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form,new,cached", [("wide", [600], [0]), ("stream", [70], [1500])])
def test_prefill_follows_falling_and_rising_scores(dtype, form, new, cached):
    """Block maxima that fall by 12 from block to block and then rise again: the reference of
    the probabilities follows them down no further than the sums allow, and back up."""
    q, k, v, t, o, c, offs, ctx = _device_case(new, cached, 12, 2, 128, 16, dtype, 5)
    assert _form(q, k, t, new) == form
    x, pages = ctx[0], t[0].long()
    step = -12.0 * (torch.arange(x, device=DEV) // 64).float()
    step = torch.maximum(step, step.flip(0))                       # falls, then rises
    k[..., 0] = 0
    flat = k[pages].flatten(0, 1)
    flat[:x, :, 0] = (step / 8.0)[:, None].to(dtype)
    k[pages] = flat.view(-1, *k.shape[1:])
    q[..., 0] = 8.0 * 128 ** 0.5                                   # score += step (key)
    got = ops.prefill_paged(q, k, v, t, o, c, max(new)).double()
    assert got.isfinite().all()
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)  # rounding of 16-bit values: of the
    for _, h, rows, sc, vh in _heads_float64(q, k, v, t, offs, ctx, (0, 5, 11)):  # output, and
        err = (got[rows, h] - torch.softmax(sc, -1) @ vh).abs().max()  # of p in o and in l
        assert err <= 3 * unit * vh.abs().max(), (h, err)


def _range_rule(new, cached, hq, hkv, nwg_max=256):
    """(T, workgroups) of the stream-K split as its rule has them: ranges of at least
    ceil(nb_max / 30) 64-key blocks, and where T blocks are fewer than three a workgroup, in
    128-row units of at least nine blocks and 480 rows x blocks on average, of the root of
    blocks x (0.2 + 1.3 rows / 128)."""
    g = hq // hkv
    blocks, units, rows, nb_max = 0, 0, 0, 0
    for n, c in zip(new, cached):
        rows += n * g
        for rb in range(-(-n * g // 128)):
            nb = (c + (min(128 * (rb + 1), n * g) - 1) // g) // 64 + 1
            blocks, units, nb_max = blocks + nb, units + 1, max(nb_max, nb)
    t, avg = blocks * hkv, blocks / max(units, 1)
    r = max(1, -(-nb_max // 30))
    if t < 3 * nwg_max and avg >= 9 and avg * rows >= 480 * units:
        r = max(r, math.ceil(math.sqrt(avg * (0.2 + 1.3 * rows / (128 * units)))))
    nwg = max(1, min(nwg_max, t // r))
    return t, nwg & ~7 if nwg >= 8 else nwg


@pytest.mark.parametrize("dtype,max_tol,mean_tol", [(torch.float16, 2e-3, 2e-4),
                                                    (torch.bfloat16, 1.6e-2, 1.6e-3)])
@pytest.mark.parametrize("new,cached,hq,hkv,d,bs", [
    ([100], [1000], 12, 2, 128, 16),                 # longer ranges
    ([30], [4000], 12, 2, 128, 16),
    ([200, 100], [300, 1500], 12, 2, 128, 32),
    ([16], [4001], 32, 8, 128, 16),
    ([8] * 8, [600] * 8, 14, 2, 64, 32),             # few rows a unit, short ranges
    ([5, 0, 9], [9000, 7, 3001], 71, 1, 64, 16),
    ([1, 2], [640, 4000], 14, 2, 64, 16),            # too few rows: as with any length
    ([1] * 5, [2841] * 5, 28, 4, 128, 16),
    ([37] * 40, [3000] * 40, 12, 2, 128, 16),        # more blocks than three a workgroup
])
def test_stream_k_ranges_follow_rows_and_blocks(dtype, max_tol, mean_tol, new, cached, hq, hkv, d, bs):
    """The split of chunks over cached tokens is the rule's, planned and unplanned give the
    same bits on one workspace call after call, and match float64."""
    q, k, v, t, o, c, offs, ctx = _device_case(new, cached, hq, hkv, d, bs, dtype, sum(cached))
    assert _form(q, k, t, new) == _form(q, k, t, new, planned=True) == "stream"
    plan = ops.prefill_paged_plan(o, c, sum(new), hq, hkv, t.shape[1], bs)
    header = plan.buffer[:16].view(torch.int32).tolist()
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    want_t, want_nwg = _range_rule(new, cached, hq, hkv, cus)
    assert header[:4] == [want_nwg, want_t, want_t // want_nwg, want_t % want_nwg]
    got = ops.prefill_paged(q, k, v, t, o, c, max(new))
    for _ in range(2):
        assert torch.equal(ops.prefill_paged(q, k, v, t, o, c, max(new), plan=plan), got)
        assert torch.equal(ops.prefill_paged(q, k, v, t, o, c, max(new)), got)
    for _, h, rows, sc, vh in _heads_float64(q, k, v, t, offs, ctx, sorted({0, hq // 2, hq - 1})):
        err = (got[rows, h].double() - torch.softmax(sc, -1) @ vh).abs()
        assert err.max() <= max_tol and err.mean() <= mean_tol, (h, err.max(), err.mean())


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form,new,cached,hq,hkv,d,bs,q_scale", [
    ("stream", [40, 130, 1], [3000, 200, 640], 12, 2, 128, 16, 8.0),
    ("stream", [33, 129], [2990, 1], 14, 2, 64, 32, 16.0),
    ("stream", [65, 1, 17], [2047, 63, 0], 16, 2, 128, 32, 1.0),
    ("stream", [77], [1501], 14, 2, 64, 16, 1.0),
    ("stream", [37] * 40, [3000] * 40, 12, 2, 128, 16, 8.0),
    ("wide", [40, 130, 1], [300, 20, 64], 6, 1, 128, 16, 16.0),
    ("wide", [900, 33], [0, 70], 14, 2, 64, 32, 16.0),
])
def test_prefill_large_scores_on_each_kernel(form, dtype, new, cached, hq, hkv, d, bs, q_scale):
    """Scores over hundreds (q scaled), head groups of 7, 64-dim heads, blocks of 32 and odd
    remainders, on the kernel named; a running maximum over part of a block's keys lets exp2
    and the 16-bit probabilities overflow.  The bound: rounding of the output and, in the
    numerator and the sum, of the probabilities, each half a unit of the 16-bit type; scores of
    300 in fp32 move a probability by less than a hundredth of that in bf16, a tenth in fp16."""
    q, k, v, t, o, c, offs, ctx = _device_case(new, cached, hq, hkv, d, bs, dtype, sum(new) + hq)
    q = (q.float() * q_scale).to(dtype)
    assert _form(q, k, t, new) == form
    got = ops.prefill_paged(q, k, v, t, o, c, max(new))
    plan = ops.prefill_paged_plan(o, c, sum(new), hq, hkv, t.shape[1], bs)
    assert got.isfinite().all()
    assert torch.equal(ops.prefill_paged(q, k, v, t, o, c, max(new), plan=plan), got)
    unit = 2.0 ** (-11 if dtype == torch.float16 else -8)
    for _, h, rows, sc, vh in _heads_float64(q, k, v, t, offs, ctx, sorted({0, hq // 2, hq - 1})):
        err = (got[rows, h].double() - torch.softmax(sc, -1) @ vh).abs()
        assert err.max() <= 3.2 * unit * vh.abs().max(), (h, err.max())


def test_pages_reserved_ahead_do_not_change_a_prefill():
    """attention_for_request on a prompt whose request holds pages for later tokens: the
    kernel, and so every bit, is that of a request holding the prompt's pages only."""
    n, hq, hkv, d, bs = 1000, 12, 2, 128, 16
    g = torch.Generator().manual_seed(91)
    keys, values = (torch.randn(n, hkv, d, generator=g).half().to(DEV) for _ in range(2))
    q = torch.randn(n, hq, d, generator=g).half().to(DEV)
    outs = []
    for reserved in (n, 8 * n):
        cache = PagedKVCache(CacheLayout(1, 8 * n // bs, bs, hkv, d), device=DEV)
        cache.reserve("r", reserved)
        cache.write(0, "r", 0, keys, values)
        # (a length may be any number that is whole)
        for length in (n, float(n), torch.tensor(n)):
            outs.append(attention.attention_for_request(q, cache, 0, "r", length,
                                                        torch.arange(n, device=DEV)))
    assert all(torch.equal(outs[0], x) for x in outs[1:])
    forms = [ops.prefill_form(1, n, n, hq, hkv, d, bs, w // bs, torch.float16) for w in (1008, 8 * n)]
    assert forms == ["wide", "stream"]


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("form,bs,hq,hkv,d", [("wide", 16, 12, 2, 128), ("tile", 8, 4, 4, 64)])
@pytest.mark.parametrize("seqs", [64, 65, 256, 257, 300])
def test_prefill_of_more_sequences_than_a_wave_holds(dtype, form, bs, hq, hkv, d, seqs):
    """Row blocks are found among the sequences 64 at a time, four such passes a round trip past
    64: sequences of no, one and a few tokens at the edges, against float64."""
    new = [(0, 1, 5, 16, 3, 40)[i % 6] for i in range(seqs)]
    new[-1] = 37
    cached = [(0, 7, 33)[i % 3] for i in range(seqs)]
    q, k, v, t, o, c, offs, ctx = _device_case(new, cached, hq, hkv, d, bs, dtype, seqs)
    assert _form(q, k, t, new) == form
    got = ops.prefill_paged(q, k, v, t, o, c, max(new)).double()
    tol = 2e-3 if dtype == torch.float16 else 1.6e-2
    for _, h, rows, sc, vh in _heads_float64(q, k, v, t, offs, ctx, (hq - 1,)):
        assert (got[rows, h] - torch.softmax(sc, -1) @ vh).abs().max() <= tol, rows
