"""Which attention method an inference prefill calls, and with what, for the package's routers
and for routers with methods of their own (on the CPU, with the kernels replaced)."""

from types import SimpleNamespace

import pytest
import torch

from ananta_ocr_amd import modeling_deepseekv2 as M
from ananta_ocr_amd.dash_attention import DashAttention


class OnGpu(torch.Tensor):
    """A CPU tensor that says it is on the GPU."""

    @property
    def is_cuda(self):
        return True


class Router(DashAttention):
    def __init__(self):
        torch.nn.Module.__init__(self)
        self.block_size, self.stage0, self.use_triton = 32, "indexer", True
        self._infer_params = dict(idx_scale=1.0, floor=1e-4, sigma=1.0, K=2, topm=2)

    def router_qk(self, hs, pe):
        return hs, hs

    def block_scores(self, iq, ik, q_pos=None, nblk=None, kbar=None):
        return torch.zeros(1, iq.shape[1], nblk)


def _prefill(router, monkeypatch, dtype=torch.bfloat16, first=0, mask=None):
    monkeypatch.setattr(M.ops, "route", lambda z, *a: (
        torch.ones(*z.shape[:2], 2, dtype=torch.int32), torch.zeros(*z.shape[:2], 2),
        torch.ones(*z.shape[:2], 2, dtype=torch.uint8)))
    q = torch.zeros(1, 2, 64, 128, dtype=dtype).as_subclass(OnGpu)
    pos = torch.arange(first, first + 64)[None]
    return M._infer_prefill_attend(SimpleNamespace(layer_idx=0), router, torch.zeros(1, 64, 128),
                                   q, q, q, None, pos, None, mask, None)


@pytest.mark.parametrize("first", [0, 5])
@pytest.mark.parametrize("masked", [False, True])
def test_own_methods_get_64_bit_ids(first, masked, monkeypatch):
    seen = []

    class Own(Router):
        def _forward_triton(self, q, k, v, topi, bias, valid, S, nblk, pos):
            seen.append(("triton", topi.dtype, int(pos[0, 0])))

        def _forward_dense(self, q, k, v, topi, bias, valid, S, nblk, mask):
            seen.append(("dense", topi.dtype, mask is not None))
            return torch.zeros(64, nblk).gather(1, topi[0])          # needs 64-bit ids

    mask = torch.zeros(1, 1, 64, 64) if masked else None
    _prefill(Own(), monkeypatch, first=first, mask=mask)
    want = [] if masked else [("triton", torch.int64, first)]
    assert seen == want + [("dense", torch.int64, masked)]


def test_own_dense_alone_and_as_an_attribute(monkeypatch):
    seen = []

    def dense(q, k, v, topi, *a):
        seen.append(topi.dtype)
        return q

    class Own(Router):
        def _forward_dense(self, *a):
            return dense(*a)

    _prefill(Own(), monkeypatch)
    r = Router()
    r._forward_dense = dense
    _prefill(r, monkeypatch)
    assert seen == [torch.int64] * 2


@pytest.mark.parametrize("dtype,first,calls", [
    (torch.bfloat16, 0, ["attn"]), (torch.bfloat16, 5, ["attn"]),
    (torch.float32, 0, ["entry"]), (torch.float32, 5, ["entry", "attn"])])
def test_the_packages_routers(dtype, first, calls, monkeypatch):
    """bf16 goes to the attention at once, whatever the positions; other types through the
    entry point, whose positions must count from 0."""
    from ananta_ocr_amd import sparse_gather
    seen = []

    def entry(q, k, v, idx, bias, pos, *a):
        seen.append("entry")
        return q if int(pos[0, 0]) == 0 else None

    def attn(q, k, v, idx, *a, **kw):
        seen.append("attn")
        return q
    monkeypatch.setattr(sparse_gather, "triton_gather_attention_e2e", entry)
    monkeypatch.setattr(M.ops, "attn_prefill", attn)
    r = Router()
    r.local_window, r._scale = 64, 0.1
    _prefill(r, monkeypatch, dtype=dtype, first=first)
    assert seen == calls
