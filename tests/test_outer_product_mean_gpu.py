"""GPU: the fused outer-product mean (bf16 operands at 64 MSA channels, 32 hidden, 128 or 256
pair channels; reference ``ops.py:683-785``): tiles of 8 x 8 residues and 64 sequences cut by N
and S, both streams, a batch of two, and the in-place residual. Against the oracle in fp64 by
the bf16 rule (relL2(HIP - exact) <= 2 relL2(eager bf16 - exact)); batch items bit for bit
independent."""

from __future__ import annotations

import pytest
import torch

from oracle import pairformer_ref as R
from tests._helpers import assert_bf16_rule, mod, sub, to

pytestmark = pytest.mark.gpu
W = mod("weights")
ops = mod("ops")
BF = torch.bfloat16


@pytest.mark.parametrize("stream", [BF, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("S,N,B,cz", [(1, 1, 1, 128), (63, 7, 1, 128), (64, 8, 2, 128), (65, 9, 1, 128),
                                      (200, 33, 1, 128), (129, 70, 1, 256), (40, 17, 2, 256)])  # fmt: skip
def test_opm_fused(dev, S, N, B, cz, stream):
    print(f"[opm fused] S={S} N={N} B={B} cz={cz} {stream}", flush=True)
    p = sub(W.make_evoformer_block_weights(7 + N, perturb_affine=True, c_pair=cz), "outer_product.")
    m = ops.OuterProductMean(64, cz).eval()
    m.load_state_dict(p)
    m = m.to(dev).to(stream)
    g = torch.Generator().manual_seed(S + N)
    msa = torch.randn(B, S, N, 64, generator=g).to(dev, stream)
    mask = (torch.rand(B, S, N, generator=g) > 0.2).float().to(dev)
    mask[:, 0] = 1.0  # every pair has a sequence: out_b / 1e-3 would be the whole norm
    pair = torch.randn(B, N, N, cz, generator=g).to(dev, stream)
    with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=stream == torch.float32):
        got = m(msa, mask)
        last = m(msa[-1:], mask[-1:])
        res = m.forward_residual_(pair.clone(), msa, mask)
        eager = R.outer_product_mean(msa.to(BF), mask.to(BF), to(p, dev, BF))
    ref = R.outer_product_mean(msa.double(), mask.double(), to(p, dev, torch.float64))
    assert got.dtype == stream and torch.equal(last, got[-1:])
    print("   ", assert_bf16_rule(got.cpu(), eager.float().cpu(), ref.cpu(), f"opm S={S} N={N}"), flush=True)
    # one rounding of pair + update, against the separately rounded update
    want = pair.double() + got.double()
    tol = (2.0**-7 if stream == BF else 2.0**-22) * want.abs().max().item()
    assert (res.double() - want).abs().max().item() <= tol
