"""Performance cases of the GPT-OSS-120B path: what one call, or one layer's or one step's calls, cost a program.

Every case is the work of one public entry point (or of the few that a program calls together), with the shapes, data
types and distributions of the repository's own configurations: hidden 2880, 128 experts of which 4 per token, MXFP4
experts (uniform E2M1 codes, E8M0 exponents 119..125), 64 query and 8 KV heads of 64, window 128, vocabulary 201,088.

Decode work runs as the repository's decode loops run it, from a hipGraph that was captured once over kept buffers;
prompt work runs as plain calls, since a prompt's length sets its shapes.  Where a program streams weights that no
cache holds (every layer has its own), a pass takes several layers, so that a pass's weights exceed the Infinity
Cache or nearly do.

Kinds (the listed cases, and the ranges that draw() covers):
  experts_decode    ResidentExperts.forward_decode, 1..8 tokens, t950 / PS4 / raw pools: the expert body of a decode step
  experts_prefill   ResidentExperts.forward_prefill, 9..4096 tokens (a prompt's tail, a short prompt, a full block),
                    t950 / PS4 / raw pools, Zipf(1.1) or uniform routing
  gemv              mxfp4_gemv / mxfp4_gemv_masked, 1..16 slots, PS4 / raw: the reference-named decode products
  gemm              mxfp4_gemm (M rows on each of E slots) or mxfp4_gemm_grouped_into (ragged pairs): the
                    reference-named prompt products, PS4 / raw
  attention_decode  decode_attention_batched, batch 1..8, contexts 64..8192: full layers (chunked) and sliding layers
                    (rolling cache) in turn
  attention_prefill prefill_attention, blocks of 1..4096 queries after 0..4096 earlier positions: a full layer and a
                    sliding one (rolling cache, then ring_write)
  core              FusedCore.run: the drop-in per-layer decode core
  model_decode      DecodeModel.run: one greedy step of a model of few layers with the full vocabulary
  model_prefill     DecodeModel.prefill: a prompt through a model of few layers
"""
from __future__ import annotations

import math
from dataclasses import replace

import torch

from neural_amd import fused_core as fc
from neural_amd import tiles
from neural_amd.attention import (SplitAttn, auto_split, decode_attention_batched, prefill_attention, ring_write)
from neural_amd.model import DecodeModel, random_weights, yarn_inv_freq
from neural_amd.moe.experts import ResidentExperts
from neural_amd.moe.layout import GPTOSS_LAYOUT, GPTOSS_LAYOUT_PS4, GPTOSS_LAYOUT_T950, mxfp4_pool_views
from neural_amd.q80.mxfp4_kernels import (GroupedGemmPlan, mxfp4_gemm, mxfp4_gemm_grouped_into, mxfp4_gemv,
                                          mxfp4_gemv_masked)

DEV = "cuda"
H, GU, NE, TOP_K = 2880, 5760, 128, 4
NQ, NKV, HD, WINDOW, VOCAB = 64, 8, 64, 128, 201088
CODE_BYTES = GPTOSS_LAYOUT.gate_pack_bytes + GPTOSS_LAYOUT.down_pack_bytes
EXPERT_BYTES = (GU + H) * (H // 2 + H // 32)             # codes and scales of one expert, 13,219,200
LAYOUTS = {"t950": GPTOSS_LAYOUT_T950, "ps4": GPTOSS_LAYOUT_PS4, "raw": GPTOSS_LAYOUT}
BF = torch.bfloat16


def listed():
    return [
        # One sequence's decode step: the expert body of 8 layers, one token each (the smallest batch).
        dict(name="experts_decode_b1", kind="experts_decode", layout="t950", batch=1, layers=8),
        # A few sequences decoding together, an odd batch.
        dict(name="experts_decode_b3", kind="experts_decode", layout="t950", batch=3, layers=4),
        # The largest decode batch.
        dict(name="experts_decode_b8", kind="experts_decode", layout="t950", batch=8, layers=2),
        # A short prompt (or the last block of a long one): more experts than tokens, an odd count.
        dict(name="experts_prefill_t23", kind="experts_prefill", layout="t950", tokens=23, zipf=False),
        # One MoE layer of a 2,048-token prompt with skewed expert popularity.
        dict(name="experts_prefill_t2048", kind="experts_prefill", layout="t950", tokens=2048, zipf=True),
        # The reference engine's decode products on a PS4 store: gate_up (shared x), then down (x per expert), with
        # the weights of non-resident experts zero.
        dict(name="gemv_masked_ps4_e4", kind="gemv", layout="ps4", slots=4, masked=True, layers=8),
        # The reference engine's ragged prompt products on a raw store: 500 tokens' pairs by expert.
        dict(name="gemm_grouped_raw_t500", kind="gemm", layout="raw", grouped=True, tokens=500, slots=0, rows=0),
        # Attention of one sequence's decode steps at a short context: latency and launches.
        dict(name="attention_decode_b1_c1000", kind="attention_decode", batch=1, context=1000, layers=8),
        # Attention of a whole 4,096-token prompt block.
        dict(name="attention_prefill_t4096", kind="attention_prefill", tokens=4096, before=0),
        # The drop-in decode core at a 4,096-token context: six layers, full and sliding.
        dict(name="core_c4096", kind="core", context=4096, layers=6),
        # One greedy token of a 4-layer model with the whole vocabulary at a 4,096-token context.
        dict(name="model_decode_c4096", kind="model_decode", context=4096, layers=4),
        # An odd-sized prompt through a 2-layer model, its last token's logits and the caches that decode goes on with.
        dict(name="model_prefill_t2501", kind="model_prefill", tokens=2501, layers=2),
    ]


def _log(rng, lo, hi):
    """An integer in [lo, hi], uniform in its logarithm."""
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    kind = rng.choice(["experts_decode", "experts_prefill", "gemv", "gemm", "attention_decode", "attention_prefill",
                       "core", "model_decode", "model_prefill"])
    layout = rng.choice(["t950", "t950", "t950", "ps4", "raw"])
    store = rng.choice(["ps4", "raw"])
    if kind == "experts_decode":
        batch = rng.randint(1, 8)
        return dict(kind=kind, layout=layout, batch=batch, layers=rng.randint(max(2, 8 // batch), 12))
    if kind == "experts_prefill":
        return dict(kind=kind, layout=layout, tokens=_log(rng, 9, 4096), zipf=rng.random() < 0.5)
    if kind == "gemv":
        return dict(kind=kind, layout=store, slots=rng.randint(1, 16), masked=rng.random() < 0.5,
                    layers=rng.randint(4, 8))
    if kind == "gemm":
        if rng.random() < 0.5:
            return dict(kind=kind, layout=store, grouped=True, tokens=_log(rng, 9, 2048), slots=0, rows=0)
        slots = _log(rng, 1, 32)
        return dict(kind=kind, layout=store, grouped=False, tokens=0, slots=slots, rows=_log(rng, 1, 4096 // slots))
    if kind == "attention_decode":
        return dict(kind=kind, batch=rng.randint(1, 8), context=_log(rng, 64, 8192), layers=2 * rng.randint(2, 6))
    if kind == "attention_prefill":
        return dict(kind=kind, tokens=_log(rng, 1, 4096), before=rng.choice([0, _log(rng, 1, 4096)]))
    if kind == "core":
        return dict(kind=kind, context=_log(rng, 64, 8192), layers=rng.randint(4, 8))
    if kind == "model_decode":
        return dict(kind=kind, context=_log(rng, 64, 8192), layers=rng.choice([2, 4]))
    return dict(kind=kind, tokens=_log(rng, 9, 2500), layers=2)


# ------------------------------------------------------------------------------------------------------- inputs
# In a whole model a layer's experts add about a tenth of the residual stream, as in a trained one (with exponents of
# 119..125 and random weights they would drown it, and a near tie in the routing would decide every later value).
MODEL_LOW = 111


def _gen(seed, stream):
    """A device generator for one stream of a case's inputs (streams are drawn independently of one another)."""
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * int(seed) + stream)
    return g


def _normal(g, *shape, std=1.0):
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(BF)


def _raw_chunk(seed, chunk, n, low=119):
    """Slots of one layer in the raw store layout: uniform codes, E8M0 exponents uniform in low..low + 6."""
    g = _gen(seed, 1000 + chunk)
    buf = torch.empty(n, GPTOSS_LAYOUT.slot_bytes, dtype=torch.uint8, device=DEV)
    codes = torch.empty(n, CODE_BYTES // 4, dtype=torch.int32, device=DEV)
    codes.random_(-2 ** 31, 2 ** 31, generator=g)
    buf[:, :CODE_BYTES] = codes.view(torch.uint8)
    buf[:, CODE_BYTES:] = torch.randint(low, low + 7, (n, GPTOSS_LAYOUT.slot_bytes - CODE_BYTES), generator=g, device=DEV,
                                        dtype=torch.uint8)
    return buf


def _pool(seed, layout, chunks, n=NE, low=119):
    """A resident pool of ``chunks`` x ``n`` slots in the given layout."""
    lay = LAYOUTS[layout]
    pool = torch.empty(chunks * n, lay.slot_bytes, dtype=torch.uint8, device=DEV)
    for c in range(chunks):
        raw = _raw_chunk(seed, c, n, low)
        dst = pool[c * n:(c + 1) * n]
        if layout == "t950":
            tiles.repack_to_t950(raw, dst)
        elif layout == "raw":
            dst.copy_(raw)
        else:                                           # PS4 rows: the base, then 4-bit deltas 0..6 (low = even)
            dst[:, :CODE_BYTES] = raw[:, :CODE_BYTES]
            d = (raw[:, CODE_BYTES:] - low).view(n, GU + H, H // 64, 2)
            rows = dst[:, CODE_BYTES:].view(n, GU + H, 1 + H // 64)
            rows[:, :, 0] = low
            rows[:, :, 1:] = d[..., 0] | (d[..., 1] << 4)
    return pool


def _biases(seed, n_layers):
    g = _gen(seed, 2)
    return _normal(g, n_layers * NE, GU, std=0.02), _normal(g, n_layers * NE, H, std=0.02)


def _experts(seed, layout, n_layers, low=119):
    bg, bd = _biases(seed, n_layers)
    return ResidentExperts(_pool(seed, layout, n_layers, low=low), replace(LAYOUTS[layout], n_layers=n_layers), bg, bd)


def _routing(seed, stream, tokens, zipf):
    """Top-4 ids [tokens, 4] and their softmax weights: from random router logits, or with Zipf(1.1) popularity."""
    g = _gen(seed, stream)
    logits = torch.randn(tokens, NE, generator=g, device=DEV)
    if zipf:                                            # draws without replacement ~ p by Gumbel noise on log p
        rank = torch.randperm(NE, generator=g, device=DEV) + 1
        u = torch.rand(tokens, NE, generator=g, device=DEV).clamp(1e-6, 1 - 1e-6)
        ids = (-1.1 * torch.log(rank.float()) - torch.log(-torch.log(u))).topk(TOP_K, -1).indices
        top = logits.gather(1, ids).sort(-1, descending=True).values
    else:
        top, ids = logits.topk(TOP_K, -1)
    return ids.contiguous(), torch.softmax(top, -1).to(BF).contiguous()


def _captured(fn):
    """fn() captured in a hipGraph after one eager call; returns (graph, what the captured call returned)."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        fn()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = fn()
    return g, out


def _pairs_by_expert(seed, tokens):
    """Rows per expert of a block's Zipf-routed pairs: [(expert, rows)], experts without rows left out."""
    ids, _ = _routing(seed, 3, tokens, True)
    n = torch.bincount(ids.view(-1), minlength=NE).tolist()
    return [(e, c) for e, c in enumerate(n) if c]


def _active(seed, layer, slots):
    """Active weights of one layer's slots: softmax weights, about one in four zero (an expert held elsewhere)."""
    g = _gen(seed, 40 + layer)
    w = torch.softmax(torch.randn(slots, generator=g, device=DEV), -1)
    w[torch.rand(slots, generator=g, device=DEV) < 0.25] = 0.0
    return w.to(BF)


def _attention_inputs(case, seed):
    """Per layer: q, K and V caches, sinks; and each sequence's position."""
    B, ctx = case["batch"], case["context"]
    pos = torch.tensor([ctx - 1 - (b * 37) % max(1, ctx // 2) for b in range(B)], dtype=torch.int64, device=DEV)
    layers = []
    for li in range(case["layers"]):
        g = _gen(seed, 60 + li)
        rows = ctx if li % 2 else WINDOW
        layers.append((_normal(g, B, NQ * HD), _normal(g, B, NKV, rows, HD), _normal(g, B, NKV, rows, HD),
                       _normal(g, NQ)))
    return pos, layers


def _prompt_attention_inputs(case, seed):
    g = _gen(seed, 80)
    T, p0 = case["tokens"], case["before"]
    full = (_normal(g, T, NQ, HD), _normal(g, 1, NKV, p0 + T, HD), _normal(g, 1, NKV, p0 + T, HD), _normal(g, NQ))
    slide = (_normal(g, T, NQ, HD), _normal(g, 1, NKV, WINDOW, HD), _normal(g, 1, NKV, WINDOW, HD), _normal(g, NQ),
             _normal(g, T, NKV, HD), _normal(g, T, NKV, HD))
    return full, slide


def _core_inputs(case, seed):
    w = random_weights(case["layers"], vocab=64, device=DEV, seed=seed)
    g = _gen(seed, 90)
    ctx = case["context"]
    mid0, g_out = _normal(g, 1, H), _normal(g, case["layers"], 1, H)
    caches = [(_normal(g, 1, NKV, r, HD), _normal(g, 1, NKV, r, HD))
              for r in (WINDOW if ly.sliding else ctx + 64 for ly in w.layers)]
    return w, mid0, g_out, caches


def _model_inputs(case, seed):
    """The dense weights, the tokens (a context and the next one, or a prompt) and, for a decode step, the caches."""
    w = random_weights(case["layers"], device=DEV, seed=seed)
    g = _gen(seed, 95)
    if case["kind"] == "model_prefill":
        return w, torch.randint(0, VOCAB, (case["tokens"],), generator=g, device=DEV).cpu(), None
    ctx = case["context"]
    tokens = torch.randint(0, VOCAB, (ctx + 1,), generator=g, device=DEV).cpu()
    return w, tokens, [(_normal(g, 1, NKV, r, HD), _normal(g, 1, NKV, r, HD))
                       for r in (WINDOW if ly.sliding else ctx + 64 for ly in w.layers)]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "experts_decode":
        n, B = case["layers"], case["batch"]
        ex = _experts(seed, case["layout"], n)
        x = [_normal(_gen(seed, 100 + li), B, H) for li in range(n)]
        routes = [_routing(seed, 200 + li, B, False) for li in range(n)]
        outs = torch.empty(n, B, H, dtype=BF, device=DEV)

        def step():
            for li in range(n):
                ex.forward_decode(li, x[li], *routes[li], out=outs[li])
            return outs

        return dict(keep=(ex, x, routes), graph=_captured(step))
    if kind == "experts_prefill":
        T = case["tokens"]
        return dict(ex=_experts(seed, case["layout"], 1), x=_normal(_gen(seed, 100), T, H),
                    route=_routing(seed, 3, T, case["zipf"]))
    if kind == "gemv":
        n, E = case["layers"], case["slots"]
        views = mxfp4_pool_views(_pool(seed, case["layout"], 1, n * E), LAYOUTS[case["layout"]])
        slots = [torch.arange(li * E, (li + 1) * E, device=DEV) for li in range(n)]
        x = [_normal(_gen(seed, 100 + li), 1, H) for li in range(n)]
        h = [_normal(_gen(seed, 200 + li), E, H) for li in range(n)]
        act = [_active(seed, li, E) for li in range(n)]

        def step():
            out = []
            for li in range(n):
                if case["masked"]:
                    out.append(mxfp4_gemv_masked(x[li], views[0], views[2], slots[li], act[li]))
                    out.append(mxfp4_gemv_masked(h[li], views[1], views[3], slots[li], act[li], per_expert_x=True))
                else:
                    out.append(mxfp4_gemv(x[li], views[0], views[2], slots[li]))
                    out.append(mxfp4_gemv(h[li], views[1], views[3], slots[li], per_expert_x=True))
            return out

        return dict(keep=(views, slots, x, h, act), graph=_captured(step))
    if kind == "gemm":
        if not case["grouped"]:
            E, M = case["slots"], case["rows"]
            views = mxfp4_pool_views(_pool(seed, case["layout"], 1, E), LAYOUTS[case["layout"]])
            return dict(views=views, slots=torch.arange(E, device=DEV), x=_normal(_gen(seed, 100), M, H),
                        h=_normal(_gen(seed, 101), M, H))
        views = mxfp4_pool_views(_pool(seed, case["layout"], 1), LAYOUTS[case["layout"]])
        groups = _pairs_by_expert(seed, case["tokens"])
        P = sum(c for _, c in groups)
        x, h = _normal(_gen(seed, 100), P, H), _normal(_gen(seed, 101), P, H)
        gu, y = torch.empty(P, GU, dtype=BF, device=DEV), torch.empty(P, H, dtype=BF, device=DEV)
        off, pg, pd = 0, [], []
        for e, c in groups:
            pg.append((x[off:off + c], e, gu[off:off + c]))
            pd.append((h[off:off + c], e, y[off:off + c]))
            off += c
        return dict(views=views, plans=(GroupedGemmPlan(pg), GroupedGemmPlan(pd)), out=(gu, y))
    if kind == "attention_decode":
        pos, layers = _attention_inputs(case, seed)
        split = SplitAttn(auto_split(case["context"]), case["context"], torch.device(DEV), batch=case["batch"])
        outs = torch.empty(case["layers"], case["batch"], NQ * HD, dtype=BF, device=DEV)

        def step():
            for li, (q, kc, vc, sinks) in enumerate(layers):
                if li % 2:
                    decode_attention_batched(q, kc, vc, sinks, pos, outs[li], HD ** -0.5, split=split)
                else:
                    decode_attention_batched(q, kc, vc, sinks, pos, outs[li], HD ** -0.5, sliding=WINDOW, ring=WINDOW)
            return outs

        return dict(keep=(pos, layers, split), graph=_captured(step))
    if kind == "attention_prefill":
        full, slide = _prompt_attention_inputs(case, seed)
        return dict(full=full, slide=slide, p0=case["before"], after=(slide[1].clone(), slide[2].clone()))
    if kind == "core":
        w, mid0, g_out, caches = _core_inputs(case, seed)
        ctx, n = case["context"], case["layers"]
        cg = fc.core_graphs(w, ctx + 64, DEV)
        core = fc.FusedCore(cg, DEV, ring=WINDOW, split_k=16)
        cg.pos.fill_(ctx)
        for lg, (k, v) in zip(cg.layers, caches):
            lg.k.copy_(k)
            lg.v.copy_(v)
        mid = torch.empty_like(mid0)
        z = lambda *s, dt=BF: torch.zeros(*s, dtype=dt, device=DEV)  # noqa: E731
        bx, bslots, bgids, bw = z(1, H), z(TOP_K, dt=torch.int64), z(TOP_K, dt=torch.int64), z(TOP_K)
        pack = z(H + 3 * TOP_K, dt=torch.float32)
        tab = torch.arange(n * NE, device=DEV)
        mids, hns = z(n, 1, H), z(n, 1, H)

        def step():
            mid.copy_(mid0)                             # the token's embedding
            for li in range(n):
                core.run(li, mid, g_out[li], None, tab, bx, bslots, bgids, bw, pack)
                mids[li].copy_(mid)                     # what the expert body and the next layer read
                hns[li].copy_(bx)
            return [mids, hns, core.logits] + [t for lg in cg.layers for t in (lg.k, lg.v)]

        return dict(keep=(w, cg, core, mid0, g_out, mid, bx, bslots, bgids, bw, pack, tab), graph=_captured(step))
    w, tokens, caches = _model_inputs(case, seed)
    ex = _experts(seed, "t950", case["layers"], MODEL_LOW)
    n = case["context"] if kind == "model_decode" else case["tokens"]
    m = DecodeModel(w, ex, smax=n + 64, keep_logits=True)
    if kind == "model_prefill":
        return dict(model=m, tokens=tokens)
    m.reset(tokens, pos=n)
    for dst, src in zip(m.kc + m.vc, [k for k, _ in caches] + [v for _, v in caches]):
        dst.copy_(src)
    m.capture()
    return dict(model=m, pos=m.pos.clone())


# --------------------------------------------------------------------------------------------------------- a pass
def run(state):
    if "graph" in state:
        graph, out = state["graph"]
        graph.replay()
        return out
    if "ex" in state:
        return state["ex"].forward_prefill(0, state["x"], *state["route"])
    if "plans" in state:
        v, (pg, pd) = state["views"], state["plans"]
        mxfp4_gemm_grouped_into(pg, v[0], v[2])
        mxfp4_gemm_grouped_into(pd, v[1], v[3])
        return list(state["out"])
    if "views" in state:
        v = state["views"]
        return [mxfp4_gemm(state["x"], v[0], v[2], state["slots"]), mxfp4_gemm(state["h"], v[1], v[3], state["slots"])]
    if "full" in state:
        p0 = state["p0"]
        q, kc, vc, sinks = state["full"]
        a = prefill_attention(q, kc, vc, sinks, p0, HD ** -0.5, 0, kc.shape[2])
        q, kc, vc, sinks, kn, vn = state["slide"]
        b = prefill_attention(q, kc, vc, sinks, p0, HD ** -0.5, WINDOW, 0, k_new=kn, v_new=vn, ring=WINDOW)
        ring_write(*state["after"], kn, vn, p0, WINDOW)  # a ring of its own: the state serves every pass
        return [a, b, *state["after"]]
    m = state["model"]
    if "tokens" in state:
        m.prefill(state["tokens"])
    else:
        m.pos.copy_(state["pos"])                       # the same position again: the state serves every pass
        m.run(1)
    return [m.logits] + m.kc + m.vc


# ---------------------------------------------------------------------------------------------------------- work
def _touched(tokens, zipf):
    """Expected distinct experts of a block."""
    if not zipf:
        return NE * (1 - (1 - TOP_K / NE) ** tokens)
    p = [r ** -1.1 for r in range(1, NE + 1)]
    return sum(1 - (1 - v / sum(p)) ** (TOP_K * tokens) for v in p)


def _experts_work(tokens, zipf):
    return (_touched(tokens, zipf) * EXPERT_BYTES + tokens * (4 * H + 40), 2 * TOP_K * tokens * 3 * H * H)


def _attention_work(queries, keys_read, pairs):
    """queries x 64 heads in and out, K/V rows read, (query, key) pairs attended."""
    return queries * NQ * HD * 4 + keys_read * NKV * HD * 4, 4 * NQ * HD * pairs


def _dense_work(rows):
    n = (NQ + 2 * NKV) * HD * H + H * NQ * HD + NE * H
    return 2 * n, 2 * n * rows


def work(case):
    kind = case["kind"]
    b = f = 0.0
    if kind == "experts_decode":
        b, f = (case["layers"] * v for v in _experts_work(case["batch"], False))
    elif kind == "experts_prefill":
        b, f = _experts_work(case["tokens"], case["zipf"])
    elif kind == "gemv":
        e = case["layers"] * case["slots"]
        on = 0.75 if case["masked"] else 1.0
        b = e * (on * (EXPERT_BYTES if case["layout"] == "raw" else GPTOSS_LAYOUT_PS4.slot_bytes) + 2 * (GU + H + H))
        f = 2 * on * e * (GU + H) * H
    elif kind == "gemm":
        rows = TOP_K * case["tokens"] if case["grouped"] else case["slots"] * case["rows"]
        n = _touched(case["tokens"], True) if case["grouped"] else case["slots"]
        x = 2 * rows if case["grouped"] else 2 * case["rows"]
        b, f = n * EXPERT_BYTES + 2 * x * H + 2 * rows * (GU + H), 2 * rows * (GU + H) * H
    elif kind == "attention_decode":
        B, ctx, n = case["batch"], case["context"], case["layers"] // 2
        keys = [ctx - (i * 37) % max(1, ctx // 2) for i in range(B)]
        for k in (sum(keys), sum(min(v, WINDOW) for v in keys)):
            v = _attention_work(B, k, k)
            b, f = b + n * v[0], f + n * v[1]
    elif kind == "attention_prefill":
        T, p0 = case["tokens"], case["before"]
        for keys, pairs in ((p0 + T, T * p0 + T * (T + 1) / 2),
                            (min(p0, WINDOW) + T, sum(min(p0 + i + 1, WINDOW) for i in range(T)))):
            v = _attention_work(T, keys, pairs)
            b, f = b + v[0], f + v[1]
        b += 2 * min(T, WINDOW) * NKV * HD * 2
    elif kind in ("core", "model_decode"):
        ctx = case["context"]
        for li in range(case["layers"]):
            keys = ctx + 1 if li % 2 else min(ctx + 1, WINDOW)
            for v in (_attention_work(1, keys, keys), _dense_work(1)) + \
                    ((_experts_work(1, False),) if kind == "model_decode" else ()):
                b, f = b + v[0], f + v[1]
        if kind == "model_decode":
            b, f = b + 2 * VOCAB * H, f + 2 * VOCAB * H
    else:
        T = case["tokens"]
        for li in range(case["layers"]):
            pairs = T * (T + 1) / 2 if li % 2 else sum(min(i + 1, WINDOW) for i in range(T))
            for v in (_attention_work(T, T, pairs), _dense_work(T), _experts_work(T, False)):
                b, f = b + v[0], f + v[1]
        b, f = b + 2 * VOCAB * H + 2 * T * H, f + 2 * VOCAB * H
    return {"bytes": b, "flops": f}


# About four times the error against the 64-bit results, which the bf16 rounding points between the products set.
_REL = {"experts_decode": 1.3e-2, "experts_prefill": 1.3e-2, "gemv": 7e-3, "gemm": 7e-3, "attention_decode": 1.6e-2,
        "attention_prefill": 9e-3, "core": 2e-2, "model_decode": 5e-2, "model_prefill": 5e-2}


def tolerance(case):
    return {"rel": _REL[case["kind"]]}


# --------------------------------------------------------------------------------------------------- 64-bit results
_E2M1 = [0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0]


def _dequant(raw, down):
    """fp64 weight matrix of one raw slot: [5760, 2880] gate_up rows or [2880, 2880] down rows."""
    r0, n = (GU, H) if down else (0, GU)
    codes = raw[r0 * (H // 2):(r0 + n) * (H // 2)].view(n, H // 2)
    exps = raw[CODE_BYTES + r0 * (H // 32):CODE_BYTES + (r0 + n) * (H // 32)].view(n, H // 32)
    table = torch.tensor(_E2M1 + [-v for v in _E2M1], dtype=torch.float64, device=DEV)
    w = torch.stack((table[(codes & 15).long()], table[(codes >> 4).long()]), -1).view(n, H // 32, 32)
    return (w * torch.exp2(exps.double() - 127)[..., None]).view(n, H)


def _exact_experts(raw, x, ids, wts, bias_gu, bias_dn):
    """The expert layer in fp64: clamped SwiGLU (alpha 1.702, limit 7) between the products, the top-4 weighted sum."""
    out = torch.zeros(x.shape[0], H, dtype=torch.float64, device=DEV)
    for e in ids.unique().tolist():
        tok, rank = (ids == e).nonzero(as_tuple=True)
        gu = x[tok].double() @ _dequant(raw[e], False).T + bias_gu[e].double()
        gate, up = gu[:, :H].clamp(max=7.0), gu[:, H:].clamp(-7.0, 7.0)
        h = (up + 1) * gate * torch.sigmoid(1.702 * gate)
        y = h @ _dequant(raw[e], True).T + bias_dn[e].double()
        out.index_add_(0, tok, y * wts[tok, rank].double()[:, None])
    return out


def _exact_attention(q, k, v, sinks, visible):
    """q [T, 64, 64], k and v [8, S, 64], visible [T, S]: softmax with each head's sink in the denominator, fp64."""
    out = torch.empty(q.shape, dtype=torch.float64, device=DEV)
    for h in range(NQ):
        s = (q[:, h].double() @ k[h // (NQ // NKV)].double().T) * HD ** -0.5
        s = torch.cat((s.masked_fill(~visible, -math.inf), sinks[h].double().expand(s.shape[0], 1)), 1)
        out[:, h] = torch.softmax(s, -1)[:, :-1] @ v[h // (NQ // NKV)].double()
    return out


def _rms(x, weight):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + 1e-5) * weight.double()


def _exact_core(ly, x, p0, cache):
    """One layer's dense core in fp64 for rows x [T, H] at positions p0 ..: RMSNorm, Q|K|V, YaRN RoPE, attention, o_proj
    and residual, post norm, router.  cache: (k, v) [1, 8, rows, 64] holding the positions before p0 (position j in row
    j % 128 on sliding layers).  Returns mid, hn, router logits and the cache with the rows stored."""
    T = x.shape[0]
    pos = torch.arange(p0, p0 + T, device=DEV)
    inv, scale = yarn_inv_freq()                        # the model's frequency table is an input, as in a checkpoint
    ang = pos.double()[:, None] * inv.double().to(DEV)
    cos, sin = torch.cos(ang)[:, None] * scale, torch.sin(ang)[:, None] * scale

    def rope(v):
        a, b = v[..., :HD // 2], v[..., HD // 2:]
        return torch.cat((a * cos - b * sin, b * cos + a * sin), -1)

    qkv = (_rms(x, ly.in_w) @ ly.Wqkv.double().T + ly.bqkv.double()).view(T, -1, HD)
    q, k, v = rope(qkv[:, :NQ]), rope(qkv[:, NQ:NQ + NKV]).transpose(0, 1), qkv[:, NQ + NKV:].transpose(0, 1)
    kc, vc = (c[0].double() for c in cache)
    old = torch.arange(max(0, p0 - WINDOW) if ly.sliding else 0, p0, device=DEV)
    rows = old % WINDOW if ly.sliding else old
    keys, at = torch.cat((old, pos))[None], pos[:, None]
    att = _exact_attention(q, torch.cat((kc[:, rows], k), 1), torch.cat((vc[:, rows], v), 1), ly.sinks,
                           (keys <= at) & (keys > at - WINDOW) if ly.sliding else keys <= at)
    mid = x + att.view(T, -1) @ ly.Wo.double().T + ly.bo.double()
    hn = _rms(mid, ly.post_w)
    last = torch.arange(max(0, T - WINDOW) if ly.sliding else 0, T, device=DEV)
    rows = pos[last] % WINDOW if ly.sliding else pos[last]
    kc[:, rows], vc[:, rows] = k[:, last], v[:, last]
    return mid, hn, hn @ ly.Wr.double().T + ly.br.double(), (kc[None], vc[None])


def _exact_model(case, seed):
    """The model in fp64.  A token whose fourth and fifth router logits nearly tie may take another expert here than
    in bf16, which moves its later values by a few per cent (see MODEL_LOW)."""
    w, tokens, caches = _model_inputs(case, seed)
    bg, bd = _biases(seed, case["layers"])
    p0 = case["context"] if caches else 0
    x, kv = w.embed[tokens[p0:].to(DEV)].double(), []
    for li, ly in enumerate(w.layers):
        if caches:
            cache = caches[li]
        else:
            rows = WINDOW if ly.sliding else case["tokens"] + 64
            cache = [torch.zeros(1, NKV, rows, HD, dtype=BF, device=DEV)] * 2
        mid, hn, logits, c = _exact_core(ly, x, p0, cache)
        top, ids = logits.topk(TOP_K, -1)
        lo = li * NE
        x = mid + _exact_experts(_raw_chunk(seed, li, NE, MODEL_LOW), hn, ids, torch.softmax(top, -1), bg[lo:lo + NE],
                                 bd[lo:lo + NE])
        kv.append(c)
    logits = torch.cat([part.double() @ _rms(x[-1], w.final_w) for part in w.lm_head.split(8192)])
    return [logits] + [k for k, _ in kv] + [v for _, v in kv]


def exact(case, seed):
    kind = case["kind"]
    if kind == "experts_decode":
        bg, bd = _biases(seed, case["layers"])
        out = []
        for li in range(case["layers"]):
            ids, wts = _routing(seed, 200 + li, case["batch"], False)
            lo = li * NE
            out.append(_exact_experts(_raw_chunk(seed, li, NE), _normal(_gen(seed, 100 + li), case["batch"], H), ids,
                                      wts, bg[lo:lo + NE], bd[lo:lo + NE]))
        return torch.stack(out)
    if kind == "experts_prefill":
        T = case["tokens"]
        return _exact_experts(_raw_chunk(seed, 0, NE), _normal(_gen(seed, 100), T, H),
                              *_routing(seed, 3, T, case["zipf"]), *_biases(seed, 1))
    if kind == "gemv":
        n, E = case["layers"], case["slots"]
        raw, out = _raw_chunk(seed, 0, n * E), []
        for li in range(n):
            x, h = _normal(_gen(seed, 100 + li), 1, H).double(), _normal(_gen(seed, 200 + li), E, H).double()
            on = (_active(seed, li, E) != 0).double() if case["masked"] else torch.ones(E, device=DEV).double()
            out.append(torch.stack([on[i] * (_dequant(raw[li * E + i], False) @ x[0]) for i in range(E)]))
            out.append(torch.stack([on[i] * (_dequant(raw[li * E + i], True) @ h[i]) for i in range(E)]))
        return out
    if kind == "gemm":
        if not case["grouped"]:
            E, M = case["slots"], case["rows"]
            raw = _raw_chunk(seed, 0, E)
            x, h = _normal(_gen(seed, 100), M, H).double(), _normal(_gen(seed, 101), M, H).double()
            return [torch.stack([v @ _dequant(raw[e], d).T for e in range(E)]) for v, d in ((x, False), (h, True))]
        raw, groups = _raw_chunk(seed, 0, NE), _pairs_by_expert(seed, case["tokens"])
        P = sum(c for _, c in groups)
        x, h = _normal(_gen(seed, 100), P, H), _normal(_gen(seed, 101), P, H)
        out = []
        for v, d in ((x, False), (h, True)):
            parts = v.split([c for _, c in groups])
            out.append(torch.cat([p.double() @ _dequant(raw[e], d).T for p, (e, _) in zip(parts, groups)]))
        return out
    if kind == "attention_decode":
        pos, layers = _attention_inputs(case, seed)
        out = []
        for li, (q, kc, vc, sinks) in enumerate(layers):
            rows = []
            for b, p in enumerate(pos.tolist()):        # a rolling cache holds the last WINDOW positions, in any order
                n = p + 1 if li % 2 else min(p + 1, WINDOW)
                rows.append(_exact_attention(q[b].view(1, NQ, HD), kc[b, :, :n], vc[b, :, :n], sinks,
                                             torch.ones(1, n, dtype=torch.bool, device=DEV)).view(-1))
            out.append(torch.stack(rows))
        return torch.stack(out)
    if kind == "attention_prefill":
        T, p0 = case["tokens"], case["before"]
        (q, kc, vc, sinks), (qs, ks, vs, ss, kn, vn) = _prompt_attention_inputs(case, seed)
        at = torch.arange(p0, p0 + T, device=DEV)[:, None]
        a = _exact_attention(q, kc[0], vc[0], sinks, torch.arange(p0 + T, device=DEV)[None] <= at)
        first = max(0, p0 - WINDOW)                     # positions first .. p0 - 1 come from the rolling cache
        old = torch.arange(first, p0, device=DEV)
        keys = torch.arange(first, p0 + T, device=DEV)[None]
        b = _exact_attention(qs, torch.cat((ks[0][:, old % WINDOW], kn.transpose(0, 1)), 1),
                             torch.cat((vs[0][:, old % WINDOW], vn.transpose(0, 1)), 1), ss,
                             (keys <= at) & (keys > at - WINDOW))
        kr, vr = ks.clone(), vs.clone()
        last = torch.arange(max(0, T - WINDOW), T, device=DEV)
        kr[0][:, (p0 + last) % WINDOW] = kn[last].transpose(0, 1)
        vr[0][:, (p0 + last) % WINDOW] = vn[last].transpose(0, 1)
        return [a, b, kr.double(), vr.double()]
    if kind == "core":
        w, mid, g_out, caches = _core_inputs(case, seed)
        x, mids, hns, kv = mid.double(), [], [], []
        for li, ly in enumerate(w.layers):
            x, hn, logits, c = _exact_core(ly, x + (g_out[li].double() if li else 0), case["context"], caches[li])
            mids.append(x)
            hns.append(hn)
            kv += c
        return [torch.stack(mids), torch.stack(hns), logits[0]] + kv
    return _exact_model(case, seed)
