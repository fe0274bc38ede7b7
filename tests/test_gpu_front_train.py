"""The training router front end in the library (ops.router_front_train) against the same by
tensor ops and against 64-bit arithmetic without rounding.

The tensor ops round the projection, the norm's output, the rotary products and every gradient
between them to bf16 (2^-9 each); the library rounds the same forward values and, of the
gradients, only that of the projection and the results.  So its error against 64 bits may not
exceed the tensor ops' (plus a tenth, for the order of sums), and the outputs agree to the
projection's rounding, which flips by one bf16 step (2^-8) where the sums' order decides it.
"""

import pytest
import torch

from ananta_ocr_amd import dash_attention as DA
from ananta_ocr_amd import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _exact(hs, wq, wk, nq, nk, cos, sin):
    """Index queries and keys in 64 bits (finite inputs, no value at a clamp)."""
    out = []
    for w, n in ((wq, nq), (wk, nk)):
        p = hs @ w.t()
        y = p * torch.rsqrt(p.pow(2).mean(-1, keepdim=True) + 1e-6) * (1 + n)
        if cos is not None:
            a, b = y.chunk(2, -1)
            y = y * cos[..., :128].double() + torch.cat((-b, a), -1) * sin[..., :128].double()
        out.append(y)
    return out


def _inputs(B, S, hid, rope, seed):
    g = torch.Generator().manual_seed(seed)
    hs = torch.randn(B, S, hid, generator=g).bfloat16()
    w = [(torch.randn(128, hid, generator=g) * hid ** -0.5).bfloat16() for _ in range(2)]
    n = [(torch.randn(128, generator=g) * 0.1).bfloat16() for _ in range(2)]
    cos = sin = None
    if rope is not None:
        ang = torch.rand(1, S, 64, generator=g) * 6.3
        cos, sin = (torch.cat([f(ang)] * 2, -1).to(rope) for f in (torch.cos, torch.sin))
        cos, sin = (t.to(DEV).expand(B, -1, -1) for t in (cos, sin))
    gr = [torch.randn(B, S, 128, generator=g).to(DEV) for _ in range(2)]
    return [t.to(DEV) for t in (hs, *w, *n)], cos, sin, gr


def _run(f, leaves, cos, sin, gr, double=False):
    x = [(t.detach().double() if double else t.detach().clone()).requires_grad_() for t in leaves]
    out = f(x)
    return list(out) + list(torch.autograd.grad(out, x, [g.to(out[0].dtype) for g in gr]))


@pytest.mark.parametrize("B,S,hid,rope", [
    (1, 1, 128, torch.bfloat16),            # one row, one column tile
    (2, 63, 256, torch.float32),
    (1, 64, 384, None),
    (3, 129, 1280, torch.bfloat16),         # a row tile with one row
    (1, 2753, 1280, torch.bfloat16),        # several row ranges, the last one short
])
def test_front_train_matches_tensor_ops(B, S, hid, rope):
    leaves, cos, sin, gr = _inputs(B, S, hid, rope, S + hid)
    assert ops.router_front_train_ok(*leaves, cos, sin)
    got = _run(lambda x: ops.router_front_train(*x, 1e-6, cos, sin, DA._front_train_ops), leaves, cos,
               sin, gr)
    old = _run(lambda x: DA._front_train_ops(*x, cos, sin, 1e-6), leaves, cos, sin, gr)
    ref = _run(lambda x: _exact(*x, cos, sin), leaves, cos, sin, gr, double=True)
    for name, a, b, r in zip(("iq", "ik", "hs", "wq", "wk", "nq", "nk"), got, old, ref):
        assert a.dtype == b.dtype and a.shape == b.shape
        err, before = ((t.double() - r).norm() / r.norm() for t in (a, b))
        assert err <= 1.1 * before + 1e-4, (name, err.item(), before.item())


def test_front_train_guards_and_layouts():
    """Non-finite hidden states (zero gradient there), non-finite and huge output gradients
    (sanitized), rows of a wider buffer, and a graph of the gradient."""
    leaves, cos, sin, gr = _inputs(2, 70, 256, torch.bfloat16, 1)
    hs = leaves[0]
    hs[0, 3, 5], hs[1, 69, 255], hs[0, 64, 0] = float("nan"), float("inf"), -float("inf")
    gr[0][0, 5, 6], gr[1][1, 2, 3], gr[0][1, 7, 7] = float("nan"), float("inf"), 1e6
    wide = torch.zeros(2, 70, 512, dtype=torch.bfloat16, device=DEV)
    wide[..., 256:] = hs
    got = _run(lambda x: ops.router_front_train(*x, 1e-6, cos, sin, DA._front_train_ops),
               leaves, cos, sin, gr)
    old = _run(lambda x: DA._front_train_ops(*x, cos, sin, 1e-6), leaves, cos, sin, gr)
    assert (got[2][~torch.isfinite(hs)] == 0).all()
    for a, b in zip(got, old):
        assert torch.isfinite(a).all()
        assert (a.double() - b.double()).norm() <= 3e-2 * b.double().norm()
    x = [wide[..., 256:].requires_grad_()] + [t.requires_grad_() for t in leaves[1:]]
    out = ops.router_front_train(*x, 1e-6, cos, sin, DA._front_train_ops)
    again = torch.autograd.grad(out, x, gr)
    for a, b in zip(again, got[2:]):
        assert torch.equal(a, b)
    out = ops.router_front_train(*x, 1e-6, cos, sin, DA._front_train_ops)
    first = torch.autograd.grad(out, x[3], gr, create_graph=True)[0]
    assert torch.autograd.grad(first.float().sum(), x[1])[0].isfinite().all()


@pytest.mark.parametrize("which", range(5))
def test_front_train_parameters_in_a_flat_buffer(which):
    """Hidden states, a projection or a norm weight at an odd place of a flat buffer, in bf16
    and (norm weights) fp32: the same bits as from its own buffer, forward and backward."""
    leaves, cos, sin, gr = _inputs(2, 70, 256, torch.bfloat16, 2)
    for dtype in [torch.bfloat16] + [torch.float32] * (which > 2):
        x = [t.to(dtype) if i == which else t for i, t in enumerate(leaves)]
        got = []
        for odd in (False, True):
            y = [t.detach().clone() for t in x]
            if odd:
                flat = torch.zeros(x[which].numel() + 1, dtype=dtype, device=DEV)
                y[which] = flat[1:].view(x[which].shape).copy_(x[which])
            y = [t.requires_grad_() for t in y]
            assert ops.router_front_train_ok(*y, cos, sin)
            out = ops.router_front_train(*y, 1e-6, cos, sin, DA._front_train_ops)
            got.append(list(out) + list(torch.autograd.grad(out, y, gr)))
        for a, b in zip(*got):
            assert torch.equal(a, b)


def test_front_train_leaves_wrapped_modules_alone():
    """A projection with a hook, or replaced, runs as a module."""
    r = DA.DashAttention(__import__("types").SimpleNamespace(
        num_attention_heads=2, hidden_size=256, rms_norm_eps=1e-6,
        sparse_attention_config=dict(sparse_block_size=32, sparse_local_block=2,
                                     sparse_index_dim=128))).to(DEV).bfloat16()
    hs = torch.randn(1, 40, 256, device=DEV).bfloat16()
    seen = []
    plain = r._index_qk_train(hs, None)
    h = r.q_proj.register_forward_hook(lambda m, i, o: seen.append(1) or 2 * o)
    r._index_qk_train(hs, None)
    assert seen
    h.remove()
    assert torch.equal(r._index_qk_train(hs, None)[0], plain[0])
