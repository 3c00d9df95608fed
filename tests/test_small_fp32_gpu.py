"""fp32 projections of few positions (16-position blocks in the triangle multiplication, one
block per weight chunk in the grid attention) on a real MI355X: the bits of the kernels that
larger problems run."""

from __future__ import annotations

import pytest
import torch

from tests._helpers import mod

pytestmark = pytest.mark.gpu

ops = mod("ops")
attention = mod("attention")


@pytest.fixture(scope="module")
def dev():
    if not torch.cuda.is_available():
        pytest.skip("needs a GPU")
    return torch.device("cuda:0")


# one token; 33: a ragged tile past a 32-position one; 64: whole tiles, half the padded frame
@pytest.mark.parametrize("N,B", [(1, 300), (33, 5), (64, 5)])
@pytest.mark.parametrize("kind", ["out", "in", "rows", "cols"])
def test_small_projection_equals_large(dev, kind, N, B):
    """A single item runs the small forms, a batch of B the large ones; a position's sums do
    not depend on the split, so item 0 has equal bits."""
    torch.manual_seed(N)
    if kind in ("out", "in"):
        m = (ops.TriangleMulOutgoing if kind == "out" else ops.TriangleMulIncoming)(128)
    else:
        m = attention.GridSelfAttention(128, 4, transpose=kind == "cols")
    for p in m.parameters():
        if p.dim() == 2:
            torch.nn.init.normal_(p, std=p.shape[1] ** -0.5)
    m = m.to(dev).eval()
    z = torch.randn(B, N, N, 128, device=dev)
    mask = (torch.rand(B, N, N, device=dev) > 0.2).float()
    print(f"[small fp32] {kind} N={N} B={B}", flush=True)
    with torch.no_grad():
        one = m(z[:1].contiguous(), mask[:1].contiguous())
        many = m(z, mask)
    assert torch.isfinite(one).all()
    assert torch.equal(one[0], many[0])
