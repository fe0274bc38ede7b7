"""Inputs of the training front end and indexer scores that the library refuses or takes in
another way, checked on the CPU before any launch."""

from types import SimpleNamespace

import pytest
import torch

from ananta_ocr_amd import dash_attention as DA
from ananta_ocr_amd import ops


class OnGpu(torch.Tensor):
    """A CPU tensor that says it is on the GPU: what follows the device checks then fails
    here instead of reading a host pointer."""

    @property
    def is_cuda(self):
        return True


def _gpu(*shape):
    return torch.zeros(*shape).as_subclass(OnGpu)


def _no_launch(monkeypatch):
    def load():
        raise AssertionError("the library was reached")
    monkeypatch.setattr(ops._lib, "load", load)


def test_positions_in_host_memory_are_refused(monkeypatch):
    _no_launch(monkeypatch)
    iq, ik = _gpu(1, 64, 128), _gpu(1, 64, 128)
    pos = torch.arange(64)[None]
    assert ops.block_max_train_ok(iq, ik, 32)
    with pytest.raises(ValueError, match="GPU tensors"):
        ops.block_max_train(iq, ik, pos, 32, 32, 2, None)
    with pytest.raises(ValueError, match="GPU tensors"):
        ops.block_max_train(iq, torch.zeros(1, 64, 128), pos.as_subclass(OnGpu), 32, 32, 2, None)
    with pytest.raises(ValueError, match="GPU tensors"):
        ops.block_max_score(iq, ik, pos.as_subclass(OnGpu), pos, 32, 2, 32)


@pytest.mark.parametrize("rows,cols", [(1, 64), (2, 64), (1, 100), (2, 65)])
def test_positions_beyond_the_sequence_are_left_out(rows, cols, monkeypatch):
    """The tensor ops slice position_ids to the queries, so longer ones are taken."""
    got = []
    monkeypatch.setattr(ops._BlockMaxFn, "apply", lambda *a: got.append(a))
    iq = _gpu(2, 64, 128)
    pos = torch.arange(rows * cols).view(rows, cols)
    ops.block_max_train(iq, iq, pos.as_subclass(OnGpu), 32, 32, 2, None)
    (call,) = got
    assert torch.equal(call[2].as_subclass(torch.Tensor), pos[:, :64].expand(2, 64).int())
    assert call[2].is_contiguous()


@pytest.mark.parametrize("leaf", [0, 1])
def test_gradient_of_the_gradient_of_one_operand(leaf, monkeypatch):
    """create_graph where only the queries or only the keys require a gradient, as with one
    projection frozen."""
    monkeypatch.setattr(ops, "_block_max_fused", lambda q, k, *a, **kw: (q @ k.mT, None))
    x = [torch.randn(1, 8, 128) for _ in range(2)]
    x[leaf].requires_grad_()
    z = ops._BlockMaxFn.apply(*x, None, 32, 32, 8, lambda iq, ik, pos, nblk: (iq @ ik.mT).square())
    (g,) = torch.autograd.grad(z, x[leaf], torch.ones_like(z), create_graph=True)
    (gg,) = torch.autograd.grad(g.square().sum(), x[leaf])
    y = [t.detach().clone() for t in x]
    y[leaf].requires_grad_()
    (h,) = torch.autograd.grad((y[0] @ y[1].mT).square().sum(), y[leaf], create_graph=True)
    (hh,) = torch.autograd.grad(h.square().sum(), y[leaf])
    assert torch.equal(g, h) and torch.equal(gg, hh)


@pytest.mark.parametrize("need", [(0, 1, 0, 1, 0), (0, 0, 1, 0, 0), (1, 0, 0, 0, 0)])
def test_front_gradient_of_the_gradient_with_one_side_frozen(need):
    """create_graph where only the query or only the key side (or only the hidden states)
    requires a gradient."""
    g = torch.Generator().manual_seed(1)
    x = [torch.randn(1, 8, 128, generator=g), *(torch.randn(128, 128, generator=g) / 11 for _ in "qk"),
         *(torch.randn(128, generator=g) * 0.1 for _ in "qk")]
    for t, n in zip(x, need):
        t.requires_grad_(bool(n))
    grads = [torch.randn(1, 8, 128, generator=g) for _ in range(2)]
    ctx = SimpleNamespace(saved_tensors=(*x, None, None, None), cfg=(1e-6, DA._front_train_ops),
                          needs_input_grad=tuple(map(bool, need)) + (False,) * 4)
    got = ops._RouterFrontFn.backward(ctx, *grads)
    leaves = [t for t, n in zip(x, need) if n]
    out = DA._front_train_ops(*x, None, None, 1e-6)
    loss = sum((o * d).sum() for o, d in zip(out, grads))
    ref = torch.autograd.grad(loss, leaves, create_graph=True)
    assert [t is not None for t in got[:5]] == [bool(n) for n in need]
    for a, b in zip([t for t in got if t is not None], ref):
        torch.testing.assert_close(a, b)
        (c,) = torch.autograd.grad(a.square().sum(), leaves[0], retain_graph=True)
        assert c.isfinite().all() and c.abs().max() > 0


@pytest.mark.parametrize("offset", [0, 1, 2, 4])
def test_float_rows_at_any_offset_of_a_buffer(offset):
    """Rows for 16-byte loads: a contiguous view that starts off a 16-byte boundary is copied."""
    flat = torch.arange(2 * 5 * 128 + 8.0)
    assert flat.data_ptr() % 16 == 0
    x = flat[offset:offset + 1280].view(2, 5, 128)
    y = ops._f4_rows(x)
    assert torch.equal(x, y) and y.data_ptr() % 16 == 0 and y.is_contiguous()
    assert (y.data_ptr() == x.data_ptr()) == (offset % 4 == 0)
