"""The matrix-core block-max scores (dash_block_max_fused) and their gradient
(dash_block_max_backward) on the GPU against 64-bit tensor ops: tile and block edges, ragged
lengths, packed positions, segment starts, equal keys (which share a gradient), scores at
the clamp and operands that are not finite.

Score tolerance: an fp32 dot product of 128 terms in any order is within 128 * 2^-24 of the
sum of the terms' magnitudes."""

import math
from types import SimpleNamespace

import pytest
import torch

from ananta_ocr_amd import ops
from ananta_ocr_amd.dash_attention import DashAttention
from oracle import dash_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"
DOT = 128 * 2.0 ** -24


def _router(bs, lb):
    sp = dict(sparse_block_size=bs, sparse_local_block=lb, sparse_index_dim=128)
    return DashAttention(SimpleNamespace(num_attention_heads=2, hidden_size=256,
                                         rms_norm_eps=1e-6, sparse_attention_config=sp)).to(DEV)


def _magnitude(q, k, bs, nblk):
    """[B, C, nblk] largest sum of |q_i k_i| of a block."""
    m = q.abs() @ k.abs().transpose(1, 2)
    return torch.nn.functional.pad(m, (0, nblk * bs - k.shape[1])).view(*m.shape[:2], nblk, bs).amax(-1)


def _bounds(q, k, pos, bs, nblk, lw):
    """[B, C, nblk] least and largest block score of fp32 dot products in any order."""
    s, e = q @ k.transpose(1, 2), DOT * (q.abs() @ k.abs().transpose(1, 2))
    hidden = torch.arange(k.shape[1], device=q.device) > pos[..., None] - lw
    out = []
    for x in (s - e, s + e):
        x = x.clamp(-1e4, 1e4).masked_fill(hidden, -1e9)
        x = torch.nn.functional.pad(x, (0, nblk * bs - k.shape[1]), value=-1e9)
        out.append(x.view(*x.shape[:2], nblk, bs).amax(-1))
    return out


@pytest.mark.parametrize("B,S,bs,lb", [(1, 1, 32, 1), (2, 31, 32, 1), (1, 333, 32, 4),
                                       (2, 700, 64, 2), (1, 385, 96, 1), (1, 641, 128, 1),
                                       (1, 4200, 32, 4), (1, 5000, 64, 1)])
def test_training_scores_and_gradients(B, S, bs, lb):
    g = torch.Generator().manual_seed(S + bs)
    r = _router(bs, lb)
    nblk = (S + bs - 1) // bs
    iq, ik = (torch.randn(B, S, 128, generator=g) for _ in range(2))
    if S > 300:
        ik[:, 40:44] = ik[:, 40:41]                 # equal keys within one block
        ik[:, 70] = 0.0
        iq[:, S - 1] *= 2.0e4                       # scores beyond the clamp
        # beyond the bf16 parts' range (2^60 = 1.15e18); their products' sums stay in range
        iq[0, S - 2], ik[0, 100] = 2.0e18, 2.0e18 * ik[0, 100]
    pos = torch.arange(S).expand(B, S).clone()
    if B > 1:
        pos[1] = torch.cat([torch.arange(S // 2), torch.arange(S - S // 2)])
    iq, ik, pos = iq.to(DEV), ik.to(DEV), pos.to(DEV)
    a, b = iq.clone().requires_grad_(), ik.clone().requires_grad_()
    assert ops.block_max_train_ok(a, b, bs)
    z = r._block_scores_train(a, b, pos, nblk)
    c, d = iq.double().requires_grad_(), ik.double().requires_grad_()
    ref = r._block_scores_train(c, d, pos, nblk)    # 64-bit inputs: the tensor ops
    # a masked block is exactly that; else the score lies between the largest of the visible
    # keys' clamped lower bounds and that of their upper bounds
    assert torch.equal(z == -1e9, ref == -1e9)
    least, most = _bounds(iq.double(), ik.double(), pos, bs, nblk, lb * bs)
    assert torch.all((z.double() >= least) & (z.double() <= most))
    # a gradient on a few entries of each row, the masked ones included
    dz = torch.randn(z.shape, generator=g).to(DEV)
    dz = torch.where(torch.rand(z.shape, generator=g).to(DEV) < 0.3, dz, torch.zeros_like(dz))
    z.backward(dz)
    ref.backward(dz.double())
    for x, y in ((a, c), (b, d)):
        # sums of up to 0.3 S terms in fp32, in another order
        bound = 1e-5 * y.grad.abs().amax(-1, keepdim=True) + 1e-5
        assert torch.all((x.grad.double() - y.grad).abs() <= bound)
    z2 = r._block_scores_train(a, b, pos, nblk)     # the same gradient bits on every run
    again = torch.autograd.grad(z2, (a, b), dz)
    assert torch.equal(again[0], a.grad) and torch.equal(again[1], b.grad)


@pytest.mark.parametrize("mode", [0, 1])
@pytest.mark.parametrize("B,C,Sk,bs,lw", [(2, 64, 64, 32, 32), (1, 300, 1111, 64, 100),
                                          (2, 129, 500, 96, 1), (1, 200, 2500, 128, 128)])
def test_scores_match_oracle(B, C, Sk, bs, lw, mode, monkeypatch):
    monkeypatch.setattr(ops, "BLOCK_MAX_FUSED_ROWS", 1)
    g = torch.Generator().manual_seed(C + bs + mode)
    q, k = torch.randn(B, C, 128, generator=g), torch.randn(B, Sk, 128, generator=g)
    pos = torch.randint(0, Sk, (B, C), generator=g)
    nblk = (Sk + bs - 1) // bs + 1                  # one block past the keys
    seg = (pos // 3) if mode == 1 else torch.zeros_like(pos)
    out = ops.block_max_score(q.to(DEV), k.to(DEV), pos.to(DEV), seg.to(DEV), bs, nblk, lw,
                              mode=mode).cpu()
    if mode == 1:
        ref = O.block_max_score(q.double().float(), k, pos, seg, bs, nblk, lw)
    else:
        ref = O.block_scores_indexer(q, k, pos, nblk, bs, lw)
    seen = ref > -5e8
    assert torch.equal(out[~seen], ref[~seen])
    tol = 2 * DOT * _magnitude(q, k, bs, nblk)      # both sides are fp32
    assert torch.all((out - ref).abs()[seen] <= tol[seen])


@pytest.mark.parametrize("mode", [0, 1])
def test_scores_of_values_that_are_not_finite(mode, monkeypatch):
    """The matrix-core kernel gives what the row-by-row kernel gives."""
    g = torch.Generator().manual_seed(3)
    q, k = torch.randn(1, 96, 128, generator=g), torch.randn(1, 400, 128, generator=g)
    q[0, 5, 3], q[0, 6, 4], k[0, 33, 7], k[0, 95, 0] = math.inf, math.nan, -math.inf, math.nan
    k[0, 200:216] = 3.0e38
    pos = torch.full((1, 96), 399)
    args = (q.to(DEV), k.to(DEV), pos.to(DEV), None, 32, 13, 32)
    old = ops.block_max_score(*args, mode=mode)
    monkeypatch.setattr(ops, "BLOCK_MAX_FUSED_ROWS", 1)
    out = ops.block_max_score(*args, mode=mode)
    assert torch.equal(out.isnan(), old.isnan()) and torch.equal(out.isinf(), old.isinf())
    fin = old.isfinite()
    torch.testing.assert_close(out[fin], old[fin], atol=1e-4, rtol=1e-5)
    assert torch.equal(out[~fin & ~old.isnan()], old[~fin & ~old.isnan()])


@pytest.mark.parametrize("values", ["normal", "tiny", "large", "spread", "special"])
@pytest.mark.parametrize("B,C,Sk,bs,lw,mode", [(1, 1, 389, 32, 128, 0), (2, 129, 500, 96, 1, 1),
                                               (1, 300, 1111, 64, 100, 1), (1, 900, 900, 32, 1, 0),
                                               (1, 257, 2500, 128, 128, 0)])
def test_scores_are_the_row_by_row_bits(B, C, Sk, bs, lw, mode, values, monkeypatch):
    """A row's inference scores are the same bits in a call of any number of rows: whole
    prompts, chunks and decode steps route rows that all but tie alike."""
    g = torch.Generator().manual_seed(C + bs)
    q, k = torch.randn(B, C, 128, generator=g), torch.randn(B, Sk, 128, generator=g)
    if values == "tiny":                            # sums below the smallest normal value
        q, k = q * 1e-20, k * 1e-19
    elif values == "large":                         # sums that overflow
        q, k = q * 1e18, k * 1e20
    elif values == "spread":                        # the order of the sum shows in every bit
        q = q * (12 * torch.randn(q.shape, generator=g)).exp()
        k = k * (12 * torch.randn(k.shape, generator=g)).exp()
    elif values == "special":
        q[0, 0, 3], k[0, 33, 7], k[0, 95, 0] = math.inf, -math.inf, math.nan
        k[0, 200:216], k[0, 300], k[0, 301] = 3.0e38, 0.0, 1e-42
        q[0, C // 2] = 0.0
    pos = torch.arange(Sk - C, Sk).expand(B, C)
    seg = (pos // 3).to(DEV) if mode == 1 else None
    nblk = (Sk + bs - 1) // bs + 1
    args = (q.to(DEV), k.to(DEV), pos.to(DEV), seg, bs, nblk, lw)
    out = ops.block_max_score(*args, mode=mode)
    monkeypatch.setattr(ops, "BLOCK_MAX_FUSED_ROWS", C + 1)
    old = ops.block_max_score(*args, mode=mode)
    assert torch.equal(out.view(torch.int32), old.view(torch.int32))


def test_rows_off_a_16_byte_boundary():
    """Index queries and keys that are views at an odd place of a flat buffer."""
    g = torch.Generator().manual_seed(9)
    flat = torch.randn(2 * 300 * 128 + 1, generator=g).to(DEV)
    q, k = (flat[1 + i * 300 * 128:][:300 * 128].view(1, 300, 128) for i in range(2))
    pos = torch.arange(300, device=DEV)[None]
    args = (pos, None, 32, 10, 32)
    assert torch.equal(ops.block_max_score(q, k, *args, mode=0),
                       ops.block_max_score(q.clone(), k.clone(), *args, mode=0))
    out = []
    for x in ((q, k), (q.clone(), k.clone())):
        a, b = (t.detach().requires_grad_() for t in x)
        z = ops.block_max_train(a, b, pos, 32, 32, 10, None)
        out.append((z, *torch.autograd.grad(z.square().sum() * 1e-9, (a, b))))
    for x, y in zip(*out):
        assert torch.equal(x, y)


def test_gradient_of_the_gradient():
    """create_graph goes through the tensor ops."""
    r = _router(32, 1)
    a, b = (torch.randn(1, 100, 128, device=DEV, requires_grad=True) for _ in range(2))
    pos = torch.arange(100, device=DEV)[None]
    z = r._block_scores_train(a, b, pos, 4)
    w = torch.randn_like(z)
    (da,) = torch.autograd.grad(z, a, w, create_graph=True)
    (db,) = torch.autograd.grad(da.square().sum(), b)
    z2 = r._block_scores_ops(a, b, pos, 4)
    (da2,) = torch.autograd.grad(z2, a, w, create_graph=True)
    (db2,) = torch.autograd.grad(da2.square().sum(), b)
    torch.testing.assert_close(da, da2, atol=1e-5, rtol=1e-5)
    torch.testing.assert_close(db, db2, atol=1e-4, rtol=1e-4)
