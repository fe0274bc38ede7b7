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
