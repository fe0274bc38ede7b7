"""The key-major backward kernel on stages cut into parts: most queries route to the same few
blocks, so that one stage has many times the steps of the others.  Against torch autograd in
fp32 on the CPU with the tolerances of test_gpu_backward.py."""

import math

import pytest
import torch

from ananta_ocr_amd import ops
from test_gpu_backward import _case, _close_grad, _ref

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,H,S,bs,lw,K", [
    (1, 1, 3000, 32, 128, 4),       # two heavy blocks in one stage
    (2, 2, 2111, 64, 100, 3),       # a part ends inside the window's steps or on their edge
    (1, 1, 1900, 96, 96, 2),        # stages that span two blocks
    (1, 1, 1800, 128, 64, 2),       # two stages per block
    (1, 2, 1601, 64, 1024, 2),      # a window of many steps: parts of at least twice as many
])
def test_backward_heavy_blocks(B, H, S, bs, lw, K):
    q, k, v, topi, bias, valid, dout = _case(S, B, H, S, bs, lw, K, dup=False)
    torch.manual_seed(S)
    topi[..., 0] = 0
    topi[..., 1] = torch.where(torch.rand(B, S) < 0.9, 1, topi[..., 1])
    scale = 1 / math.sqrt(128)
    qr, kr, vr = (t.float().requires_grad_() for t in (q, k, v))
    br = bias.clone().requires_grad_()
    out_r = _ref(qr, kr, vr, topi, br, valid, bs, lw, scale)
    out_r.backward(dout.float())
    args = [t.to(DEV) for t in (q, k, v)]
    r = [t.to(DEV) for t in (topi, bias, valid)]
    out, lse = ops.attn_prefill(*args, *r, bs, lw, scale, return_lse=True)
    dq, dk, dv, db = ops.attn_prefill_backward(*args, out, lse, dout.to(DEV), *r, bs, lw, scale)
    _close_grad(dq, qr.grad, "dq")
    _close_grad(dk, kr.grad, "dk")
    _close_grad(dv, vr.grad, "dv")
    _close_grad(db, br.grad, "dbias")


def _heavy(topi, nblk_of, seed):
    """Most rows route to their document's first two blocks."""
    g = torch.Generator().manual_seed(seed)
    topi[..., 0] = 0
    topi[..., 1] = torch.where(torch.rand(topi.shape[:-1], generator=g) < 0.9,
                               torch.ones(()).long(), topi[..., 1] % nblk_of)
    return topi


def test_backward_heavy_blocks_of_unequal_documents():
    """Cut stages of several documents of very different lengths, whose parts share one pool:
    every document's gradients against a run of its own."""
    lens = [1, 2600, 40, 0, 300, 1900, 64]
    cu = torch.tensor([0] + lens).cumsum(0)
    bs, lw, K = 64, 100, 3
    q, k, v, topi, bias, valid, dout = _case(21, 1, 2, int(cu[-1]), bs, lw, K, dup=False)
    for d0, d1 in zip(cu.tolist(), cu.tolist()[1:]):
        if d1 > d0:
            nb = (d1 - d0 + bs - 1) // bs
            topi[:, d0:d1] = _heavy(topi[:, d0:d1] % nb, nb, d0) % nb
    scale = 1 / math.sqrt(128)
    args = [t.to(DEV) for t in (q, k, v)]
    r = [t[0].to(DEV) for t in (topi, bias, valid)]
    cu_t = cu.to(torch.int32).to(DEV)
    out, lse = ops.attn_prefill(*args, *r, bs, lw, scale, cu_seqlens=cu_t, return_lse=True)
    dq, dk, dv, db = ops.attn_prefill_backward(*args, out, lse, dout.to(DEV), *r, bs, lw, scale,
                                               cu_seqlens=cu_t)
    for d0, d1 in zip(cu.tolist(), cu.tolist()[1:]):
        if d1 == d0:
            continue
        sl = slice(d0, d1)
        qr, kr, vr = (t[:, :, sl].float().requires_grad_() for t in (q, k, v))
        br = bias[:, sl].clone().requires_grad_()
        _ref(qr, kr, vr, topi[:, sl], br, valid[:, sl], bs, lw, scale).backward(dout[:, :, sl].float())
        _close_grad(dq[:, :, sl], qr.grad, f"dq doc {d0}")
        _close_grad(dk[:, :, sl], kr.grad, f"dk doc {d0}")
        _close_grad(dv[:, :, sl], vr.grad, f"dv doc {d0}")
        _close_grad(db[sl][None], br.grad, f"dbias doc {d0}")


def test_backward_heavy_blocks_with_segment_starts():
    """Cut stages whose keys some rows see from their segment start on."""
    S, bs, lw, K = 2400, 64, 128, 4
    q, k, v, topi, bias, valid, dout = _case(22, 1, 2, S, bs, lw, K, dup=False)
    topi = _heavy(topi, (S + bs - 1) // bs, 22)
    kmin = torch.zeros(1, S, dtype=torch.int32)
    kmin[:, 30:], kmin[:, 900:], kmin[:, 2000:] = 30, 77, 1990
    scale = 1 / math.sqrt(128)
    qr, kr, vr = (t.float().requires_grad_() for t in (q, k, v))
    br = bias.clone().requires_grad_()
    out_r = _ref(qr, kr, vr, topi, br, valid, bs, lw, scale, kmin=kmin)
    out_r.backward(dout.float())
    args = [t.to(DEV) for t in (q, k, v)]
    r = [t.to(DEV) for t in (topi, bias, valid)]
    km = kmin.to(DEV)
    out, lse = ops.attn_prefill(*args, *r, bs, lw, scale, kmin=km, return_lse=True)
    dq, dk, dv, db = ops.attn_prefill_backward(*args, out, lse, dout.to(DEV), *r, bs, lw, scale,
                                               kmin=km)
    _close_grad(out, out_r.detach(), "out")
    _close_grad(dq, qr.grad, "dq")
    _close_grad(dk, kr.grad, "dk")
    _close_grad(dv, vr.grad, "dv")
    _close_grad(db, br.grad, "dbias")
