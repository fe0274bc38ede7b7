"""The block-grouped extend attention (ops.attn_extend) against the row-by-row decode kernels
(ops.attn_rows) and 64-bit arithmetic.

Both hold scores, weights and sums in 32 bits.  A sum of n products of magnitude at most w in
another order differs by at most n 2^-24 w; with the weights normalised and n <= 2,500 keys
that is 1.5e-4 of the largest |v|, and in the usual square-root growth 3e-6; 2e-5 is stated.
"""

import math

import pytest
import torch

from ananta_ocr_amd import ops, pipeline
from test_gpu_extend import test_extend_prefill_matches_per_request_oracle as _oracle_case

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _make(ctxs, news, H, bs, K, seed, lw, pad=0):
    g = torch.Generator().manual_seed(seed)
    lens = [a + b for a, b in zip(ctxs, news)]
    P = max((n + bs - 1) // bs for n in lens) + pad
    pool = sum((n + bs - 1) // bs for n in lens) + 2
    perm = torch.randperm(pool, generator=g)
    table = torch.full((len(lens), P), 10 ** 8, dtype=torch.int32)   # unused entries: no page
    k = (torch.randn(pool, bs, H, 128, generator=g) * 0.7).bfloat16()
    v = torch.randn(pool, bs, H, 128, generator=g).bfloat16()
    o = 0
    for b, n in enumerate(lens):
        c = (n + bs - 1) // bs
        table[b, :c] = perm[o:o + c].to(torch.int32)
        if n % bs:                                   # rows past the end are never read
            v[perm[o + c - 1], n % bs:] = float("nan")
            k[perm[o + c - 1], n % bs:] = float("nan")
        o += c
    T = sum(news)
    q = (torch.randn(T, H, 128, generator=g) * 0.7).bfloat16()
    # block ids in and out of range, repeated, within the window, and not valid
    idx = torch.randint(-1, P + 2, (T, K), generator=g, dtype=torch.int32)
    bias = torch.randn(T, K, generator=g)
    valid = torch.rand(T, K, generator=g) < 0.8
    cu = torch.tensor([0] + news).cumsum(0).to(torch.int32)
    return q, k, v, idx, bias, valid, lens, table, cu


def _exact(q, k, v, idx, bias, valid, lens, table, cu, ctxs, bs, lw, scale, rows):
    out = torch.zeros(len(rows), q.shape[1], 128, dtype=torch.float64)
    for i, r in enumerate(rows):
        b = int((cu[1:] <= r).sum())
        qp = min(ctxs[b] + r - int(cu[b]), lens[b] - 1)
        n = (lens[b] + bs - 1) // bs
        pg = table[b, :n].long()
        kk = k[pg].flatten(0, 1)[:lens[b]].double()
        vv = v[pg].flatten(0, 1)[:lens[b]].double()
        ls = qp - lw + 1
        add = torch.full((lens[b],), -math.inf, dtype=torch.float64)
        add[max(ls, 0):qp + 1] = 0.0
        seen = set()
        for s in range(idx.shape[1]):
            c = int(idx[r, s])
            if not valid[r, s] or c < 0 or c >= n or c * bs >= ls or c in seen:
                continue
            seen.add(c)
            add[c * bs:min((c + 1) * bs, ls, lens[b])] = float(bias[r, s])
        w = torch.softmax(torch.einsum("hd,nhd->hn", q[r].double(), kk) * scale + add, -1)
        out[i] = torch.einsum("hn,nhd->hd", w, vv)
    return out


@pytest.mark.parametrize("ctxs,news,H,bs,lw,K", [
    ([0], [128], 2, 64, 128, 8),              # whole tiles from the first token
    ([63, 0, 700], [1, 129, 127], 3, 64, 256, 16),
    ([1, 31, 32], [31, 33, 96], 2, 32, 128, 12),
    ([2000], [65], 2, 32, 96, 64),            # four groups of slots
    ([500, 90], [64, 300], 1, 64, 512, 5),    # slots not in fours; rows without routed keys
    ([1234], [700], 4, 64, 512, 1),           # chunks of more than 256 pairs
    ([17, 3000], [40, 30], 10, 64, 1000, 17),  # window not a multiple of the item
])
def test_extend_attention_matches_rows_and_exact(ctxs, news, H, bs, lw, K):
    data = _make(ctxs, news, H, bs, K, sum(news) + K, lw, pad=1)
    q, k, v, idx, bias, valid, lens, table, cu = data
    scale = 1.0 / math.sqrt(128)
    T = q.shape[0]
    d = [x.to(DEV) for x in (q, k, v, idx, bias, valid)]
    ctx = torch.tensor(ctxs, dtype=torch.int32, device=DEV)
    ln = torch.tensor(lens, dtype=torch.int32, device=DEV)
    seq = torch.arange(len(news)).repeat_interleave(torch.tensor(news)).to(DEV)
    pos = ctx[seq] + torch.arange(T, device=DEV) - cu.to(DEV)[seq]
    got = ops.attn_extend(*d, ln, ctx, cu.to(DEV), max(news), table.to(DEV), bs, lw, scale)
    # the row path reads table entries of used pages only, too
    old = ops.attn_rows(*d, pos, seq, bs, lw, scale, seq_lens=ln, block_table=table.to(DEV),
                        page_size=bs)
    assert (got - old).abs().max().item() <= 2e-5 * old.abs().max().item()
    rows = sorted(set(torch.linspace(0, T - 1, 40).long().tolist()))
    ref = _exact(*data, ctxs, bs, lw, scale, rows)
    err = (got[rows].cpu().double() - ref).norm() / ref.norm()
    old_err = (old[rows].cpu().double() - ref).norm() / ref.norm()
    # no further from 64 bits than the row-by-row kernels (0.78 to 0.94 of their error here)
    assert err <= 1.05 * old_err, (err, old_err)
    half = ops.attn_extend(*d, ln, ctx, cu.to(DEV), max(news), table.to(DEV), bs, lw, scale,
                           out_dtype=torch.bfloat16)
    assert torch.equal(half, got.bfloat16())


@pytest.mark.parametrize("bs", [32, 64])
def test_values_that_are_not_finite_stay_with_their_rows(bs):
    """A V element that is not finite reaches the rows whose window holds its key and the rows
    routed to its block, in its head and dim, and no others, which keep their bits."""
    ctxs, news, H, lw, K = [300, 40], [200, 130], 2, 96, 4
    q, k, v, idx, bias, valid, lens, table, cu = _make(ctxs, news, H, bs, K, 5, lw)
    scale = 0.1
    d = [torch.tensor(lens, device=DEV), torch.tensor(ctxs, device=DEV), cu.to(DEV), max(news),
         table.to(DEV), bs, lw, scale]

    def run(v):
        return ops.attn_extend(*[x.to(DEV) for x in (q, k, v, idx, bias, valid)], *d).cpu()
    clean = run(v)
    assert clean.isfinite().all()
    # request, key, head, dim: an old key, a key of the chunk (later than half of its rows, on
    # a 64-key item's edge and within one), the last key
    bad = [(0, 250, 0, 3, math.nan), (0, 383, 1, 77, math.inf), (0, 384, 0, 127, -math.inf),
           (0, 405, 1, 0, math.inf), (1, 20, 1, 64, math.nan), (1, 169, 0, 9, math.nan)]
    w = v.clone()
    hit = torch.zeros(clean.shape, dtype=torch.bool)
    for b, key, h, dim, x in bad:
        w[table[b, key // bs], key % bs, h, dim] = x
        for r in range(int(cu[b]), int(cu[b + 1])):
            qp = ctxs[b] + r - int(cu[b])
            routed = any(valid[r, s] and idx[r, s] == key // bs and key // bs * bs < qp - lw + 1
                         for s in range(K))
            hit[r, h, dim] |= qp - lw < key <= qp or routed
    got = run(w)
    assert torch.equal(~got.isfinite(), hit)
    assert torch.equal(got[~hit], clean[~hit])


def test_extend_attention_rows_do_not_depend_on_each_other():
    """Rows in another batch (other tiles, chunks and requests beside them), and q, k and v
    with other strides: the same bits."""
    ctxs, news, H, bs, lw, K = [300, 900], [200, 333], 2, 64, 256, 8
    q, k, v, idx, bias, valid, lens, table, cu = _make(ctxs, news, H, bs, K, 3, lw)
    scale = 0.1
    both = ops.attn_extend(*[x.to(DEV) for x in (q, k, v, idx, bias, valid)],
                           torch.tensor(lens, device=DEV), torch.tensor(ctxs, device=DEV),
                           cu.to(DEV), max(news), table.to(DEV), bs, lw, scale)
    cut = 100                                  # request 1 from its 100th new row on
    r = slice(news[0] + cut, sum(news))
    qs = torch.stack([q[r], q[r]], 1).to(DEV)[:, 1]                 # strided rows
    ks, vs = (torch.cat([x, x], 2).to(DEV)[:, :, H:] for x in (k, v))
    one = ops.attn_extend(qs, ks, vs, *[x[r].to(DEV) for x in (idx, bias, valid)],
                          torch.tensor(lens[1:], device=DEV),
                          torch.tensor([ctxs[1] + cut], device=DEV),
                          torch.tensor([0, news[1] - cut], device=DEV), news[1] - cut,
                          table[1:].to(DEV), bs, lw, scale)
    assert torch.equal(one, both[r])


def test_extend_prefill_blocks_beyond_the_grouped_path():
    """128-key blocks: summaries, scores and attention by the general path."""
    _oracle_case([900, 1300, 40], [300, 0, 13], 2, 128, 2, 4, 4)


def test_extend_scores_equal_the_general_path():
    """Summaries in the pool, block scores, positions and block counts against kbar and
    block_scores over per-request summaries, with an empty chunk among the requests and index
    rows in a wider buffer."""
    g = torch.Generator().manual_seed(1)
    bs, lb, ctxs, news = 32, 2, [70, 5, 0, 64], [100, 0, 33, 1]
    lens = [a + b for a, b in zip(ctxs, news)]
    B, T, P = len(lens), sum(news), 8
    table = torch.randperm(B * P + 3, generator=g)[:B * P].view(B, P).to(torch.int32).to(DEV)
    ik = torch.randn(B * P + 3, bs, 256, generator=g).to(DEV)[:, :, 128:]
    iq = torch.randn(T, 384, generator=g).to(DEV)[:, 128:256]
    hc = torch.randn(129, generator=g).to(DEV)[1:]
    i32 = dict(dtype=torch.int32, device=DEV)
    ctx, ln = torch.tensor(ctxs, **i32), torch.tensor(lens, **i32)
    cu = torch.tensor([0] + news, **i32).cumsum(0).to(torch.int32)
    assert ops.extend_scores_ok(iq, ik, torch.zeros(B * P + 3, 128, device=DEV), bs)
    general = pipeline.KBarPageCache(B * P + 3, 128, DEV)
    general.refresh_from(ik, hc.clone(), bs, table, ln, ctx // bs)   # 16-byte aligned, too
    state = pipeline.KBarPageCache(B * P + 3, 128, DEV)
    z, q_pos, row_nblk = ops.extend_scores(iq, ik, hc, cu, ctx, ln, table, state.kbar, bs, lb,
                                           max(news))
    assert torch.equal(state.kbar, general.kbar)
    seq = torch.arange(B).repeat_interleave(torch.tensor(news)).to(DEV)
    pos = ctx[seq] + torch.arange(T, device=DEV) - cu[seq]
    assert torch.equal(q_pos, pos.to(torch.int32))
    assert torch.equal(row_nblk, (ln[seq] + bs - 1) // bs)
    kb = general.kbar[table.long().reshape(-1)].view(B, P, -1)
    ref = ops.block_scores(iq[None], kb, bs, lb, q_pos=q_pos, cu_seqlens=cu, max_seqlen=max(news),
                           key_lens=ln, S=P * bs)
    assert torch.equal(z, ref)


@pytest.mark.parametrize("lens", [[1], [64, 1, 65], [300, 0, 0, 31], [0, 200, 257]])
def test_packed_row_blocks(lens):
    cu = torch.tensor([0] + lens).cumsum(0).to(DEV)
    n = torch.tensor(lens)
    ref = torch.repeat_interleave((n + 63) // 64, n).to(torch.int32)
    assert torch.equal(ops.packed_row_blocks(cu, sum(lens), 64).cpu(), ref)
