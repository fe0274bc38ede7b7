"""Inference routing of rows whose entries tie: few candidate or remote blocks among many (the
others all at the floor), and ties above it, against the oracle, exactly."""

import pytest
import torch

from ananta_ocr_amd import ops
from oracle import dash_oracle as O

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("nblk,topm", [(70, 16), (300, 16), (300, 5), (427, 1), (900, 16)])
def test_route_rows_of_few_candidates(nblk, topm):
    g = torch.Generator().manual_seed(nblk + topm)
    rows = 96
    z = torch.randn(rows, nblk, generator=g)
    z[::3] = (z[::3] * 2).round() / 2                    # ties among the candidates, too
    z[1::6] = 0.25                                       # every entry equal
    cand = torch.zeros(rows, nblk, dtype=torch.bool)
    for r in range(rows):                                # 0 .. 95 candidates (0: every block)
        cand[r, torch.randperm(nblk, generator=g)[:r]] = True
    z[5::4, nblk // 3:] = -1.0e9                         # few remote blocks
    got = ops.route(z.to(DEV), cand.to(DEV), 2.0, 1e-4, 1.0, 12, topm)
    ref = O.infer_route_select(z, cand, 2.0, 1e-4, 1.0, 12, topm)
    assert torch.equal(got[0].cpu().long(), ref[0].long())
    assert torch.equal(got[2].cpu(), ref[2])
    assert torch.allclose(got[1].cpu(), ref[1], rtol=1e-5, atol=1e-5)
