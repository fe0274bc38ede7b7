"""Timing cases of the DASH attention path: what a program that uses this package calls,
through its public entry points, from the smallest decode step to a training step over a
27,300-token sequence.

Six kinds of pass, each with its own inputs, exact result and work:

  decode      one decode step of a layer (pipeline.decode_step), contiguous or paged cache
  prefill     routing and attention of a prompt or of packed documents (pipeline.prefill)
  layer       the prefill of one decoder layer as the inference overlay runs it: page
              candidates, router front end, scores, routing, attention, decode caches
  extend      chunked prefill over a paged cache with cached prefixes (serving)
  train       one training step of the attention module: DashAttention.forward and the
              gradients of its inputs and router parameters
  attn_train  routing and attention forward and backward on given block scores

Heads (10), head and index dim (128), hidden size (1,280), block sizes, windows and routed
blocks are those of the checkpoint's configuration (block 32, 4 local blocks, 12 routed of
16 scored) and of the benchmark workloads (block 64, windows of 512 and 1,024, 8 or 16
routed); pages hold 273 image tokens.
"""

import math
import random
from types import SimpleNamespace

import torch
import torch.nn.functional as F

from ananta_ocr_amd import dash_attention, modeling_deepseekv2, ops, pages, pipeline

D = 128
H = 10
HIDDEN = H * D
PAGE = 273                               # image tokens of a page
IMG, MARK, TEXT = 5, 9, 7                # token ids: image token, page marker, text
IDX_SCALE = 128.0 / math.sqrt(128.0)     # the checkpoint's dash_scaling_factor / sqrt(d)
FLOOR = 1e-4
SCALE = 1.0 / math.sqrt(D)
DEV = "cuda"


# ------------------------------------------------------------------------------ the cases

def listed():
    return [
        # The first tokens of a short single-page answer: one sequence, latency and launches.
        dict(name="decode_b1_s389", kind="decode", B=1, lo=389, hi=389, bs=32, lb=4, K=12,
             topm=16, paged=False, bf16_out=True, layout=0),
        # Batched decode of long documents (the benchmark's contiguous decode workload).
        dict(name="decode_b8_s27300", kind="decode", B=8, lo=27300, hi=27300, bs=64, lb=16,
             K=16, topm=16, paged=False, bf16_out=False, layout=0),
        # One layer of a serving step: 32 sequences of 10 to 100 pages in a paged cache.
        dict(name="decode_paged_b32", kind="decode", B=32, lo=2730, hi=27300, bs=64, lb=16,
             K=16, topm=16, paged=True, bf16_out=True, layout=5),
        # A ten-page prompt.
        dict(name="prefill_s2730", kind="prefill", S=2730, docs=0, bs=64, lb=8, K=8, topm=8,
             layout=0),
        # A hundred-page prompt, 5 % of whose key blocks stand out (the headline workload).
        dict(name="prefill_s27300", kind="prefill", S=27300, docs=0, bs=64, lb=16, K=16,
             topm=16, layout=0),
        # Sixteen documents of 1 to 40 pages packed into one call.
        dict(name="prefill_packed16", kind="prefill", S=10920, docs=16, bs=64, lb=8, K=8, topm=8,
             layout=4),
        # A decoder layer's prefill of a 30-page prompt with the checkpoint's configuration.
        dict(name="layer_s8301", kind="layer", S=8301, bs=32, lb=4, K=12, topm=16,
             stage0="head_cls", paged_prompt=True),
        # The same call for a checkpoint routed by the indexer scores (the module's default
        # stage 0), on a ten-page prompt without page markers.
        dict(name="layer_indexer_s2730", kind="layer", S=2730, bs=32, lb=4, K=12, topm=16,
             stage0="indexer", paged_prompt=False),
        # A serving engine's extend step: four requests, each with a cached prefix and a
        # chunk of new tokens.
        dict(name="extend_b4", kind="extend", B=4, lo=0, hi=13650, chunk_lo=256,
             chunk_hi=2048, bs=64, lb=8, K=16, topm=16, layout=3),
        # Training at the start of the k schedule (64 routed blocks), two ten-page rows.
        dict(name="train_b2_s2730", kind="train", B=2, S=2730, bs=32, lb=4, step=0,
             stage0="indexer"),
        # Training after the k schedule's end (12 routed blocks), a hundred-page row.
        dict(name="train_s27300", kind="train", B=1, S=27300, bs=32, lb=4, step=1000,
             stage0="indexer"),
        # The routed attention's own training step (the benchmark's training workload).
        dict(name="attn_train_s27300", kind="attn_train", B=1, S=27300, bs=64, lb=16, K=16),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode", "decode", "prefill", "prefill", "layer", "extend", "train",
                       "attn_train"])
    layout = rng.randrange(1 << 20)
    if kind == "decode":
        hi = _log(rng, 200, 27300)
        bs, lb, K, topm = rng.choice([(32, 4, 12, 16), (64, 8, 8, 8), (64, 16, 16, 16)])
        return dict(kind=kind, B=_log(rng, 1, 32), lo=max(1, hi // rng.choice([1, 3, 10])), hi=hi,
                    bs=bs, lb=lb, K=K, topm=topm, paged=rng.random() < 0.6,
                    bf16_out=rng.random() < 0.7, layout=layout)
    if kind == "prefill":
        bs, lb, K, topm = rng.choice([(32, 4, 12, 16), (64, 8, 8, 8), (64, 16, 16, 16)])
        docs = rng.choice([0, 0, rng.randrange(2, 17)])
        S = _log(rng, 100, 27300 if docs == 0 else 8000)
        return dict(kind=kind, S=S, docs=docs, bs=bs, lb=lb, K=K, topm=topm, layout=layout)
    if kind == "layer":
        stage0 = rng.choice(["head_cls", "head_cls", "indexer"])
        return dict(kind=kind, S=_log(rng, 300, 16000), bs=rng.choice([32, 32, 64]), lb=4, K=12,
                    topm=16, stage0=stage0, paged_prompt=rng.random() < 0.5)
    if kind == "extend":
        bs, lb = rng.choice([(32, 4), (64, 8)])
        hi = _log(rng, 64, 13650)
        c = _log(rng, 16, 2048)
        return dict(kind=kind, B=rng.randrange(1, 5), lo=0, hi=hi, chunk_lo=max(1, c // 4),
                    chunk_hi=c, bs=bs, lb=lb, K=rng.choice([12, 16]), topm=16, layout=layout)
    if kind == "train":
        return dict(kind=kind, B=rng.choice([1, 1, 2]), S=_log(rng, 300, 12000),
                    bs=rng.choice([32, 32, 64]), lb=4, step=rng.choice([0, 300, 600, 1000]),
                    stage0=rng.choice(["indexer", "indexer", "head_cls"]))
    bs, lb = rng.choice([(32, 4), (64, 8), (64, 16)])
    return dict(kind=kind, B=rng.choice([1, 2]), S=_log(rng, 300, 13000), bs=bs, lb=lb,
                K=rng.choice([8, 12, 16, 32]))


def _lengths(c):
    """Lengths of a decode batch, of packed documents, or (context, chunk) of an extend
    batch: part of the case, not of its seed."""
    r = random.Random(c["layout"])
    if c["kind"] == "decode":
        return [r.randint(c["lo"], c["hi"]) for _ in range(c["B"])]
    if c["kind"] == "extend":
        return [(r.randint(c["lo"], c["hi"]), r.randint(c["chunk_lo"], c["chunk_hi"]))
                for _ in range(c["B"])]
    if c["docs"] == 0:
        return [c["S"]]
    if c["S"] >= 2 * PAGE:                       # documents of whole pages, S the longest
        return [PAGE * r.randint(1, c["S"] // PAGE) for _ in range(c["docs"])]
    return [r.randint(1, c["S"]) for _ in range(c["docs"])]


def _routed_k(c):
    """Routed blocks of a training step: the schedule's 64 to 12 over 1,000 steps."""
    return max(12, min(64, int(round(64 * (12 / 64) ** min(1.0, c["step"] / 1000)))))


# ------------------------------------------------------------------------------ the inputs

def _gen(seed):
    return torch.Generator(DEV).manual_seed(seed)


def _randn(g, *shape, std=1.0):
    return torch.randn(shape, generator=g, device=DEV) * std


def _bf16(g, *shape, std=D ** -0.5):
    """Standard deviation 1/sqrt(128) as the benchmark's q, k and v."""
    x = torch.empty(shape, dtype=torch.bfloat16, device=DEV)
    return x.normal_(0.0, std, generator=g)


def _rope(S, g=None):
    inv = 1.0 / 5.0e5 ** (torch.arange(0, D, 2, device=DEV).double() / D)
    ang = torch.arange(S, device=DEV).double()[:, None] * inv[None]
    emb = torch.cat([ang, ang], -1)[None]
    return emb.cos().bfloat16(), emb.sin().bfloat16()


def _router(c, stage0, scaling, floor):
    sp = dict(sparse_block_size=c["bs"], sparse_local_block=c["lb"], dash_scaling_factor=scaling,
              dash_prior_floor=floor, dash_sigma=1.0, dash_topk_blocks=c.get("K", 12),
              sparse_index_dim=D, dash_stage0=stage0, dash_image_only=True)
    cfg = SimpleNamespace(num_attention_heads=H, num_key_value_heads=H, hidden_size=HIDDEN,
                          rms_norm_eps=1e-6, sparse_attention_config=sp)
    return dash_attention.DashAttention(cfg).to(DEV), cfg


def _set_router(router, g):
    with torch.no_grad():
        for p in (router.q_proj.weight, router.k_proj.weight):
            p.copy_(_randn(g, D, HIDDEN, std=HIDDEN ** -0.5))
        for p in (router.q_norm.weight, router.k_norm.weight):
            p.copy_(_randn(g, D, std=0.1))
        router.head_cls.copy_(_randn(g, D, std=0.5))
    return router.bfloat16()


def _heads(x):
    """[B, S, H * D] projections as the layer's [B, H, S, D] view."""
    return x.view(x.shape[0], x.shape[1], H, D).transpose(1, 2)


def _prompt(S, marked):
    """Token ids of a prompt: a start token, pages of image tokens (with a marker each, or
    without), then text."""
    ids = [1]
    page = ([MARK] if marked else []) + [IMG] * PAGE
    while len(ids) + len(page) + 8 <= S:
        ids += page
    ids += [TEXT] * (S - len(ids))
    return torch.tensor([ids[:S]], dtype=torch.int64)


def prepare(case, seed):
    c, g = case, _gen(seed)
    s = SimpleNamespace(c=c)
    kind = c["kind"]
    if kind == "decode":
        lens = _lengths(c)
        B, bs = c["B"], c["bs"]
        nblk = (max(lens) + bs - 1) // bs
        s.hc = _randn(g, D, std=0.5)
        s.q = _bf16(g, B, H, D)
        s.idx_q = s.q.float().mean(1)[:, None]
        s.lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
        if c["paged"]:
            npg = [(n + bs - 1) // bs for n in lens]
            perm = torch.randperm(sum(npg), generator=g, device=DEV).to(torch.int32)
            s.table = torch.zeros(B, nblk, dtype=torch.int32, device=DEV)
            o = 0
            for b, n in enumerate(npg):
                s.table[b, :n] = perm[o:o + n]
                o += n
            s.k, s.v = (_bf16(g, sum(npg), bs, H, D) for _ in range(2))
            s.idx_k = s.k.float().mean(2)
            s.kw = dict(seq_lens=s.lens, block_table=s.table, page_size=bs)
        else:
            S = max(lens)
            s.k, s.v = (_bf16(g, B, H, S, D) for _ in range(2))
            s.idx_k = s.k.float().mean(1)
            s.kw = {} if min(lens) == S else dict(seq_lens=s.lens)
        s.state = pipeline.init_decode_state(s.idx_k, s.hc, bs, nblk, **s.kw)
    elif kind == "prefill":
        lens = _lengths(c)
        S = sum(lens)
        s.q, s.k, s.v = (_bf16(g, 1, H, S, D) for _ in range(3))
        if c["docs"] == 0:
            nblk = (S + c["bs"] - 1) // c["bs"]
            u = F.normalize(_randn(g, D), dim=0)
            for b in torch.randperm(nblk, generator=g, device=DEV)[:nblk // 20].tolist():
                s.k[:, :, b * c["bs"]:(b + 1) * c["bs"]] += (2.0 * u).bfloat16()
        s.idx_q, s.idx_k = s.q.float().mean(1), s.k.float().mean(1)
        s.hc = _randn(g, D, std=0.5)
        s.cu, s.longest = None, None
        if c["docs"]:
            s.cu = torch.tensor([0] + lens, device=DEV).cumsum(0).to(torch.int32)
            s.longest = max(lens)
    elif kind == "layer":
        S = c["S"]
        s.router, cfg = _router(c, c["stage0"], 128.0 if c["stage0"] == "head_cls" else 2.0,
                                FLOOR)
        s.router = _set_router(s.router, g).eval()
        model = torch.nn.Module()
        model.router, model.config = s.router, cfg
        modeling_deepseekv2.configure_dash_inference(model, True, topm=c["topm"])
        s.layer = SimpleNamespace(layer_idx=0)
        s.hs = _bf16(g, 1, S, HIDDEN, std=1.0)
        s.q, s.k, s.v = (_heads(_bf16(g, 1, S, HIDDEN)) for _ in range(3))
        s.pe = _rope(S)
        s.pos = torch.arange(S, device=DEV)[None]
        s.ids = _prompt(S, c["paged_prompt"]).to(DEV)
    elif kind == "extend":
        B, bs = c["B"], c["bs"]
        ctx = [a for a, _ in _lengths(c)]
        new = [b for _, b in _lengths(c)]
        lens = [a + b for a, b in zip(ctx, new)]
        P = (max(lens) + bs - 1) // bs
        npg = [(n + bs - 1) // bs for n in lens]
        pool = sum(npg) + 3
        perm = torch.randperm(pool, generator=g, device=DEV).to(torch.int32)
        s.table = torch.zeros(B, P, dtype=torch.int32, device=DEV)
        o = 0
        for b, n in enumerate(npg):
            s.table[b, :n] = perm[o:o + n]
            o += n
        s.k, s.v = (_bf16(g, pool, bs, H, D) for _ in range(2))
        s.idx_k = s.k.float().mean(2)
        T = sum(new)
        s.q = _bf16(g, T, H, D)
        s.idx_q = s.q.float().mean(1)
        s.hc = _randn(g, D, std=0.5)
        s.lens = torch.tensor(lens, dtype=torch.int32, device=DEV)
        s.ctx = torch.tensor(ctx, dtype=torch.int32, device=DEV)
        s.cu = torch.tensor([0] + new, device=DEV).cumsum(0).to(torch.int32)
        s.longest = max(new)
        s.state = pipeline.KBarPageCache(pool, D, DEV)
        s.state.put_sequences(s.idx_k, s.hc, bs, s.table, s.ctx)
    elif kind == "train":
        B, S = c["B"], c["S"]
        # the schedule's clock is the trainer's optimizer step
        dash_attention.K_SCHEDULE.attach(SimpleNamespace(global_step=c["step"]))
        dash_attention.K_SCHEDULE.k = dash_attention.K_SCHEDULE.k_for(c["step"])
        # the constructor's defaults; for head_cls the checkpoint's scaling
        s.router, _ = _router(c, c["stage0"], 128.0 if c["stage0"] == "head_cls" else 2.0, 1e-2)
        s.router.stage0 = c["stage0"]
        s.router = _set_router(s.router, g).train()
        s.hs = _bf16(g, B, S, HIDDEN, std=1.0).requires_grad_()
        s.q, s.k, s.v = (_heads(_bf16(g, B, S, HIDDEN)).requires_grad_() for _ in range(3))
        s.pe = tuple(t.expand(B, -1, -1) for t in _rope(S))
        s.pos = torch.arange(S, device=DEV)[None].expand(B, -1)
        s.dout = _heads(_bf16(g, B, S, HIDDEN, std=1.0))
        s.params = [s.router.q_proj.weight, s.router.k_proj.weight, s.router.q_norm.weight,
                    s.router.k_norm.weight]
        if c["stage0"] == "head_cls":
            s.params.append(s.router.head_cls)
    else:
        B, S = c["B"], c["S"]
        s.q, s.k, s.v = (_bf16(g, B, H, S, D).requires_grad_() for _ in range(3))
        s.dout = _bf16(g, B, H, S, D, std=1.0)
        kb = ops.kbar(s.k.detach().float().mean(1), torch.zeros(D, device=DEV), c["bs"])
        s.z = ops.block_scores(s.q.detach().float().mean(1), kb, c["bs"], c["lb"])
        s.z = s.z.clone().requires_grad_()
    return s


# -------------------------------------------------------------------------------- one pass

def run(s):
    c = s.c
    kind = c["kind"]
    if kind == "decode":
        out = pipeline.decode_step(
            s.state, s.q, s.k, s.v, s.idx_q, s.idx_k, s.hc, c["bs"], c["lb"], IDX_SCALE, FLOOR,
            1.0, c["K"], c["topm"], out_dtype=torch.bfloat16 if c["bf16_out"] else torch.float32,
            **s.kw)
        return [out, s.state.kbar]
    if kind == "prefill":
        return pipeline.prefill(s.q, s.k, s.v, s.idx_q, s.idx_k, s.hc, c["bs"], c["lb"], IDX_SCALE,
                                FLOOR, 1.0, c["K"], c["topm"], cu_seqlens=s.cu,
                                max_seqlen=s.longest)
    if kind == "layer":
        S = c["S"]
        nblk = (S + c["bs"] - 1) // c["bs"]
        img, ipi, qpi, _ = pages.page_ids(s.ids, IMG, MARK, S, PAGE, True)
        if c["paged_prompt"]:
            cand = pages.block_cand(s.pos, nblk, c["bs"], img, ipi, qpi)
        else:
            cand = pages.block_cand(s.pos, nblk, c["bs"], img, None, None)
        past = SimpleNamespace()
        out = modeling_deepseekv2._infer_prefill_attend(
            s.layer, s.router, s.hs, s.q, s.k, s.v, s.pe, s.pos, cand, None, past)
        kept = {"out": out, "idx_k": past._dash_idx_k[0]}
        if c["stage0"] == "head_cls":
            kept["kbar"] = past._dash_decode[0].kbar[:, :nblk]
        return kept
    if kind == "extend":
        out = pipeline.extend_prefill(
            s.state, s.q, s.k, s.v, s.idx_q, s.idx_k, s.hc, c["bs"], c["lb"], IDX_SCALE, FLOOR,
            1.0, c["K"], c["topm"], s.table, s.lens, s.ctx, s.cu, max_query_len=s.longest)
        return [out, s.state.kbar]
    if kind == "train":
        out = s.router(s.hs, s.q, s.k, s.v, position_embeddings=s.pe, position_ids=s.pos)
        grads = torch.autograd.grad(out, [s.q, s.k, s.v, s.hs] + s.params, s.dout)
        return [out, *grads]
    idx, bias, valid = ops.train_route(s.z, None, IDX_SCALE, FLOOR, 1.0, c["K"])
    out = ops.attn_prefill_autograd(s.q, s.k, s.v, idx, bias, valid, c["bs"],
                                    c["bs"] * c["lb"], SCALE)
    return [out, *torch.autograd.grad(out, [s.q, s.k, s.v, s.z], s.dout)]


# ------------------------------------------------------------------- the work of one pass

def _pairs(S, first, bs, lb, K):
    """(query, key) pairs of one head: the window and K routed blocks below it, for the
    queries first .. S - 1."""
    lw, n = bs * lb, 0
    for lo in range(first, S, 64):                 # 64 queries at a time, at their middle
        hi = min(lo + 64, S)
        t = (lo + hi) // 2
        n += (hi - lo) * (min(t + 1, lw) + min(K * bs, max(0, t + 1 - lw)))
    return n


def work(case):
    c = case
    kind, bs, lb = c["kind"], c["bs"], c["lb"]
    row = H * D * 2                                # one token of q, k, v or out in bf16
    if kind == "decode":
        keys = sum(_pairs(n, n - 1, bs, lb, c["K"]) for n in _lengths(c))
        blocks = sum((n + bs - 1) // bs for n in _lengths(c))
        return {"bytes": 2 * row * keys + blocks * D * 4 + c["B"] * (bs * D * 4 + 2 * row),
                "flops": 4 * D * H * keys + 2 * D * blocks}
    if kind == "prefill":
        lens = _lengths(c)
        T = sum(lens)
        pairs = sum(_pairs(n, 0, bs, lb, c["K"]) for n in lens)
        causal = sum(n * (n / bs) / 2 for n in lens)
        return {"bytes": T * (4 * row + 2 * D * 4), "flops": 4 * D * H * pairs + 2 * D * causal}
    if kind == "layer":
        S = c["S"]
        scored = S * S / 2 if c["stage0"] == "indexer" else S * (S / bs) / 2
        return {"bytes": S * (HIDDEN * 2 + 4 * row + D * 4 + 2 * D * 2 + 8) + 2 * D * HIDDEN * 2,
                "flops": 4 * D * H * _pairs(S, 0, bs, lb, c["K"]) + 2 * D * scored
                + 4 * D * HIDDEN * S}
    if kind == "extend":
        pairs = sum(_pairs(a + b, a, bs, lb, c["K"]) for a, b in _lengths(c))
        new = sum(b for _, b in _lengths(c))
        total = sum(a + b for a, b in _lengths(c))
        blocks = sum((a + b) / bs for a, b in _lengths(c))
        causal = sum(b * (a + b / 2) / bs for a, b in _lengths(c))
        return {"bytes": 2 * row * total + new * (2 * row + 2 * D * 4) + blocks * D * 4,
                "flops": 4 * D * H * pairs + 2 * D * causal}
    S, B = c["S"], c["B"]
    K = _routed_k(c) if kind == "train" else c["K"]
    pairs = B * _pairs(S, 0, bs, lb, K)
    nblk = (S + bs - 1) // bs
    attn = {"bytes": B * S * 8 * row, "flops": 14 * D * H * pairs}
    if kind == "attn_train":
        return {"bytes": attn["bytes"] + B * S * nblk * 8, "flops": attn["flops"]}
    scored = B * S * S / 2 if c["stage0"] == "indexer" else B * S * nblk / 2
    return {"bytes": attn["bytes"] + B * S * HIDDEN * 4 + 2 * D * HIDDEN * 4,
            "flops": attn["flops"] + 2 * D * scored + 12 * D * HIDDEN * B * S}


def tolerance(case):
    """About four times the relative error against 64-bit arithmetic: bf16 outputs 1.7e-3,
    with bf16 softmax weights as the matrix cores take them up to 3.3e-3, behind the router
    front end and its bf16 roundings 5e-3, its gradients 6e-3; fp32 outputs 2e-7 (a sum in
    another order).  In 1e-4 to 1e-3 of the rows two scores all but tie and another block may
    be routed: such a row moves by up to its own size, hence `max`."""
    kind = case["kind"]
    if kind == "decode":
        return {"rel": 7e-3, "max": 0.3} if case["bf16_out"] else {"rel": 1e-5, "max": 1e-3}
    return {"rel": {"extend": 7e-3, "prefill": 1.3e-2, "attn_train": 1.6e-2, "layer": 2e-2,
                    "train": 2.4e-2}[kind], "max": 0.9}


# ------------------------------------------------------------- the same in 64-bit arithmetic

NEG = -1.0e9


def _entmax15(x):
    """1.5-entmax by the sorted threshold (Peters et al. 2019, algorithm 2)."""
    x = (x - x.amax(-1, keepdim=True)) / 2
    srt = torch.sort(x, dim=-1, descending=True).values
    n = torch.arange(1, x.shape[-1] + 1, device=x.device, dtype=x.dtype)
    mean = srt.cumsum(-1) / n
    var = (srt ** 2).cumsum(-1) / n - mean ** 2
    tau = mean - ((1 - n * var) / n).clamp(min=0).sqrt()
    size = (tau <= srt).sum(-1, keepdim=True).clamp(min=1)
    return (x - tau.gather(-1, size - 1)).clamp(min=0) ** 2


def _select(z, cand, idx_scale, floor, K, topm):
    """Per-block bias [.., nblk] of scores z (-inf where not routed).  topm None: training
    (entmax over the whole row, first K of the masked prior)."""
    nblk = z.shape[-1]
    remote = z > NEG / 2
    c = remote if cand is None else remote & cand
    c = torch.where(c.any(-1, keepdim=True), c, remote)
    x = torch.where(c, z * idx_scale, torch.full_like(z, -1.0e4))
    if topm is None:
        prior = _entmax15(x)
        p, i = torch.sort(prior.masked_fill(~c, -1.0), dim=-1, descending=True, stable=True)
        p, i = p[..., :min(K, nblk)], i[..., :min(K, nblk)]
        valid = p >= 0
    else:
        xv, i = torch.sort(x, dim=-1, descending=True, stable=True)
        m = min(topm, nblk)
        k = max(1, min(K, m))
        p, i = _entmax15(xv[..., :m])[..., :k], i[..., :k]
        valid = c.gather(-1, i)
    lp = torch.log(p.clamp_min(floor))
    mu = torch.where(valid, lp, torch.zeros_like(lp)).sum(-1, keepdim=True) / \
        valid.sum(-1, keepdim=True).clamp(min=1)
    bias = torch.where(valid, lp - mu, torch.full_like(lp, -math.inf))
    return torch.full_like(z, -math.inf).scatter(-1, i, bias)


def _attend(q, k, v, pos, block_bias, bs, lb):
    """q [H,n,D] at positions pos [n] over k, v [H,S,D]: window keys with bias 0, keys of
    the routed blocks below the window with the block's bias."""
    S, lw = k.shape[1], bs * lb
    j = torch.arange(S, device=k.device)
    far = (pos[:, None] - lw) >= j[None]
    near = (j[None] <= pos[:, None]) & ~far
    kb = block_bias.repeat_interleave(bs, -1)[:, :S]
    none = torch.full_like(kb, -math.inf)
    bias = torch.where(near, torch.zeros_like(kb), torch.where(far, kb, none))
    return torch.softmax(q @ k.transpose(1, 2) * SCALE + bias[None], -1) @ v


def _kbar(ik, hc, bs):
    """Block summaries [nblk, d] of index keys [S, d]: softmax over a block's keys of
    key . head_cls / sqrt(d)."""
    S, nblk = ik.shape[0], (ik.shape[0] + bs - 1) // bs
    logit = (ik * hc).sum(-1) / math.sqrt(D)
    logit = F.pad(logit, (0, nblk * bs - S), value=-math.inf).view(nblk, bs)
    kk = F.pad(ik, (0, 0, 0, nblk * bs - S)).view(nblk, bs, D)
    return (torch.softmax(logit, -1)[..., None] * kk).sum(1)


def _z_headcls(iq, kb, pos, bs, lb):
    c = torch.arange(kb.shape[0], device=kb.device)
    z = iq @ kb.t() / math.sqrt(D)
    return torch.where(c[None] <= pos[:, None] // bs - lb, z, torch.full_like(z, NEG))


def _z_indexer(iq, ik, pos, bs, lb):
    S, nblk = ik.shape[0], (ik.shape[0] + bs - 1) // bs
    s = iq @ ik.t()
    far = torch.arange(S, device=s.device)[None] <= pos[:, None] - bs * lb
    s = F.pad(torch.where(far, s, torch.full_like(s, NEG)), (0, nblk * bs - S), value=NEG)
    return s.view(-1, nblk, bs).amax(-1)


def _chunks(lo, hi, n=512):
    return [(a, min(a + n, hi)) for a in range(lo, hi, n)]


def _round(x):
    """x rounded to bf16 where the path rounds, with the gradient of no rounding."""
    return x + (x.bfloat16().double() - x).detach()


def _index_qk(hs, wq, wk, nq, nk, cos, sin):
    """Index queries and keys [S, d]: bf16 projections, normalized in high precision, then
    rotated in bf16."""
    out = []
    cos, sin = cos.double(), sin.double()
    for w, n in ((wq, nq), (wk, nk)):
        p = _round(hs @ w.t())
        y = _round(p * torch.rsqrt(p.pow(2).mean(-1, keepdim=True) + 1e-6) * (1 + n))
        a, b = y.chunk(2, -1)
        out.append(_round(_round(y * cos) + _round(torch.cat((-b, a), -1) * sin)))
    return out


def _page_cand(ids, marked, pos, nblk, bs):
    """Candidate blocks of a prompt's queries: the image blocks of the query's own page
    (with markers; after the last image: every block), or every image block."""
    S = ids.shape[0]
    img = ids == IMG
    if not marked:
        blk = F.pad(img, (0, nblk * bs - S)).view(nblk, bs).any(-1)
        cand = blk[None].expand(pos.shape[0], nblk)
    else:
        page = (ids == MARK).cumsum(0) - 1
        last = int(img.nonzero().max()) if bool(img.any()) else -1
        key = torch.where(img, page, torch.full_like(page, -1))
        key = F.pad(key, (0, nblk * bs - S), value=-1).view(nblk, bs)
        query = torch.where(torch.arange(S, device=ids.device) <= last, page,
                            torch.full_like(page, -1))[pos]
        cand = torch.zeros(pos.shape[0], nblk, dtype=torch.bool, device=ids.device)
        for n in range(bs):
            cand |= (key[:, n][None] == query[:, None]) & (query[:, None] >= 0)
    return cand | ~cand.any(-1, keepdim=True)


def _prefill64(q, k, v, z_of, cand_of, bs, lb, idx_scale, floor, K, topm, first=0):
    """[H, n, D] of the queries first .. first + n - 1 (q [H,n,D]) over k, v [H,S,D]."""
    out = torch.empty_like(q)
    for a, b in _chunks(first, first + q.shape[1]):
        pos = torch.arange(a, b, device=q.device)
        z = z_of(a - first, b - first, pos)
        bias = _select(z, cand_of(pos), idx_scale, floor, K, topm)
        out[:, a - first:b - first] = _attend(q[:, a - first:b - first], k[:, :b], v[:, :b], pos,
                                              bias, bs, lb)
    return out


def _train64(q, k, v, dout, z_of, bs, lb, idx_scale, floor, K):
    """Output of the training attention of one row, with the gradients of q, k, v and of
    what z_of needs accumulated by autograd.  q, k, v [H,S,D] leaves."""
    out = torch.empty_like(q)
    for a, b in _chunks(0, q.shape[1]):
        pos = torch.arange(a, b, device=q.device)
        bias = _select(z_of(a, b, pos), None, idx_scale, floor, K, None)
        o = _attend(q[:, a:b], k[:, :b], v[:, :b], pos, bias, bs, lb)
        o.backward(dout[:, a:b])
        out[:, a:b] = o.detach()
    return out


def _leaf(x):
    return x.detach().double().requires_grad_()


def exact(case, seed):
    c = case
    s = prepare(case, seed)
    kind, bs, lb = c["kind"], c["bs"], c["lb"]
    if kind == "decode":
        out, kept = [], torch.zeros_like(s.state.kbar, dtype=torch.float64)
        for b, n in enumerate(_lengths(c)):
            if c["paged"]:
                p = s.table[b, :(n + bs - 1) // bs].long()
                k, v = (x[p].flatten(0, 1)[:n].transpose(0, 1).double() for x in (s.k, s.v))
                ik = s.idx_k[p].flatten(0, 1)[:n].double()
            else:
                k, v, ik = s.k[b, :, :n].double(), s.v[b, :, :n].double(), s.idx_k[b, :n].double()
            pos = torch.tensor([n - 1], device=DEV)
            kb = _kbar(ik, s.hc.double(), bs)
            kept[b, :kb.shape[0]] = kb
            z = _z_headcls(s.idx_q[b].double(), kb, pos, bs, lb)
            bias = _select(z, None, IDX_SCALE, FLOOR, c["K"], c["topm"])
            out.append(_attend(s.q[b][:, None].double(), k, v, pos, bias, bs, lb)[:, 0])
        return [torch.stack(out), kept]
    if kind == "prefill":
        outs, o = [], 0
        for n in _lengths(c):
            q, k, v = (x[0, :, o:o + n].double() for x in (s.q, s.k, s.v))
            iq = s.idx_q[0, o:o + n].double()
            kb = _kbar(s.idx_k[0, o:o + n].double(), s.hc.double(), bs)
            outs.append(_prefill64(q, k, v, lambda a, b, p: _z_headcls(iq[a:b], kb, p, bs, lb),
                                   lambda p: None, bs, lb, IDX_SCALE, FLOOR, c["K"], c["topm"]))
            o += n
        return torch.cat(outs, 1)[None]
    if kind == "layer":
        S, r = c["S"], s.router
        nblk = (S + bs - 1) // bs
        w = [p.detach().double() for p in (r.q_proj.weight, r.k_proj.weight, r.q_norm.weight,
                                           r.k_norm.weight)]
        iq, ik = _index_qk(s.hs[0].double(), *w, s.pe[0][0], s.pe[1][0])
        scaling = 128.0 if c["stage0"] == "head_cls" else 2.0
        got = {"idx_k": ik[None]}
        if c["stage0"] == "head_cls":
            kb = _kbar(ik, r.head_cls.detach().double(), bs)
            got["kbar"] = kb[None]

            def z_of(a, b, p):
                return _z_headcls(iq[a:b], kb, p, bs, lb)
        else:
            def z_of(a, b, p):
                return _z_indexer(iq[a:b], ik, p, bs, lb)
        got["out"] = _prefill64(
            s.q[0].double(), s.k[0].double(), s.v[0].double(), z_of,
            lambda p: _page_cand(s.ids[0], c["paged_prompt"], p, nblk, bs), bs, lb,
            scaling / math.sqrt(D), FLOOR, c["K"], c["topm"])[None]
        return got
    if kind == "extend":
        outs, o, kept = [], 0, torch.zeros_like(s.state.kbar, dtype=torch.float64)
        for i, (ctx, new) in enumerate(_lengths(c)):
            n = ctx + new
            p = s.table[i, :(n + bs - 1) // bs].long()
            k, v = (x[p].flatten(0, 1)[:n].transpose(0, 1).double() for x in (s.k, s.v))
            kb = _kbar(s.idx_k[p].flatten(0, 1)[:n].double(), s.hc.double(), bs)
            kept[p] = kb
            iq = s.idx_q[o:o + new].double()
            q = s.q[o:o + new].transpose(0, 1).double()
            outs.append(_prefill64(q, k, v, lambda a, b, p: _z_headcls(iq[a:b], kb, p, bs, lb),
                                   lambda p: None, bs, lb, IDX_SCALE, FLOOR, c["K"], c["topm"],
                                   first=ctx))
            o += new
        return [torch.cat(outs, 1).transpose(0, 1), kept]
    out, dq, dk, dv, dz, dhs = [], [], [], [], [], []
    if kind == "attn_train":
        for b in range(c["B"]):
            q, k, v, z = (_leaf(x[b]) for x in (s.q, s.k, s.v, s.z))
            out.append(_train64(q, k, v, s.dout[b].double(), lambda a, e, p: z[a:e], bs, lb,
                                IDX_SCALE, FLOOR, c["K"]))
            for to, x in ((dq, q), (dk, k), (dv, v), (dz, z)):
                to.append(x.grad)
        return [torch.stack(x) for x in (out, dq, dk, dv, dz)]
    w = [_leaf(p) for p in s.params]
    scaling = 128.0 if c["stage0"] == "head_cls" else 2.0
    for b in range(c["B"]):
        q, k, v, hs = (_leaf(x[b]) for x in (s.q, s.k, s.v, s.hs))
        made = _index_qk(hs, *w[:4], s.pe[0][b], s.pe[1][b])
        if c["stage0"] == "head_cls":
            made[1] = _kbar(made[1], w[4], bs)
        iq, key = (x.detach().requires_grad_() for x in made)
        z = _z_headcls if c["stage0"] == "head_cls" else _z_indexer
        out.append(_train64(q, k, v, s.dout[b].double(),
                            lambda a, e, p: z(iq[a:e], key, p, bs, lb), bs, lb,
                            scaling / math.sqrt(D), 1e-2, _routed_k(c)))
        torch.autograd.backward(made, [iq.grad, key.grad])
        for to, x in ((dq, q), (dk, k), (dv, v), (dhs, hs)):
            to.append(x.grad)
    return [torch.stack(x) for x in (out, dq, dk, dv, dhs)] + [x.grad for x in w]
