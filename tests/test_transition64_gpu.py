"""GPU: the fused transition at 64 channels with bf16 GEMMs (the template stack's factor 2 and
the MSA stack's factor 4; reference ``primitives.py:193-251``): row counts around the 32-row
wave tiles, both streams, in place, into another residual, and an unaligned input (which takes
the row GEMMs). Against the oracle in fp64 by the bf16 rule."""

from __future__ import annotations

import pytest
import torch

from oracle import pairformer_ref as R
from tests._helpers import assert_bf16_rule, mod, to

pytestmark = pytest.mark.gpu
primitives = mod("primitives")
kernels = mod("kernels")
BF = torch.bfloat16
C = 64


def _params(factor, seed):
    g = torch.Generator().manual_seed(seed)
    rn = lambda *s: torch.randn(*s, generator=g)  # noqa: E731
    return {"norm.weight": 1 + 0.1 * rn(C), "norm.bias": 0.1 * rn(C), "linear1.weight": rn(2 * factor * C, C) / 8,
            "linear2.weight": rn(C, factor * C) / (8 * factor**0.5)}  # fmt: skip


def _module(dev, factor, seed):
    p = _params(factor, seed)
    m = primitives.TransitionBlock(C, factor).eval()
    m.load_state_dict(p)
    return m.to(dev), p


@pytest.mark.parametrize("stream", [BF, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("factor", [2, 4])
@pytest.mark.parametrize("M", [1, 16, 31, 33, 255, 257, 20000])
def test_transition64(dev, M, factor, stream):
    print(f"[transition64] M={M} factor={factor} {stream}", flush=True)
    m, p = _module(dev, factor, M + factor)
    x = torch.randn(M, C, generator=torch.Generator().manual_seed(M)).to(dev, stream)
    res = torch.randn(M, C, generator=torch.Generator().manual_seed(M + 1)).to(dev, stream)
    with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=stream == torch.float32):
        got = m(x)
        inplace, _ = m.forward_residual_(x.clone())
        other, _ = m.run(x, out=res.clone(), accumulate=True)
        eager = R.transition(x.to(BF), to(p, dev, BF))
    ref = R.transition(x.double(), to(p, dev, torch.float64))
    assert got.dtype == stream
    print("   ", assert_bf16_rule(got.cpu(), eager.float().cpu(), ref.cpu(), f"transition64 M={M}"), flush=True)
    for out, base in ((inplace, x), (other, res)):
        want = base.double() + got.double()  # one rounding, against the separately rounded update
        tol = (2.0**-7 if stream == BF else 2.0**-22) * want.abs().max().item()
        assert (out.double() - want).abs().max().item() <= tol


def test_transition64_unaligned(dev):
    print("[transition64] input 2 bytes off a 16-byte boundary", flush=True)
    m, _ = _module(dev, 2, 9)
    x = torch.randn(300, C, generator=torch.Generator().manual_seed(1)).to(dev, BF)
    off = torch.empty(x.numel() + 1, dtype=BF, device=dev)[1:].view(x.shape).copy_(x)
    with torch.no_grad():
        a, b = m(x).float(), m(off).float()
    # the same roundings of LN, hidden units and output, sums in another order
    assert (a - b).norm() <= 4e-3 * a.norm()
