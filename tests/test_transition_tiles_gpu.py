"""GPU: the pair transition's kernels by size (128 channels, factor 4; ``primitives.py:193-251``
with the fused single_to_pair of ``evoformer.py:322-328``): four-wave and eight-wave tiles in
bf16, 16- and 32-row tiles in fp32, on both sides of each line, ragged rows, two batch items, in place. fp32 against float64 at 1e-5, bf16 by the bf16 rule; the
pair logits against LN + projection of the stored rows."""

from __future__ import annotations

import pytest
import torch

from oracle import pairformer_ref as R
from tests._helpers import assert_bf16_rule, assert_fp32_close, mod, sub, to

pytestmark = pytest.mark.gpu
W = mod("weights")
evoformer = mod("evoformer")
BF = torch.bfloat16
# on 256 CUs the lines lie at 4096 rows (fp32) and 32768 (bf16)


@pytest.mark.parametrize("regime", ["fp32", "bf16", "amp"])
@pytest.mark.parametrize("B,N", [(1, 1), (1, 5), (2, 33), (1, 64), (1, 65), (1, 90), (1, 91), (1, 181), (1, 182)])
def test_pair_transition_sizes(dev, B, N, regime):
    print(f"[pair transition] B={B} N={N} {regime}", flush=True)
    sd = W.make_block_weights(N, perturb_affine=True)
    blk = evoformer.PairFormerBlock(128, 384).eval()
    blk.load_state_dict(sd)
    stream = BF if regime == "bf16" else torch.float32
    cdt = torch.float32 if regime == "fp32" else BF
    blk = blk.to(dev).to(stream)
    p = sub(sd, "pair_transition.")
    z = torch.randn(B, N, N, 128, generator=torch.Generator().manual_seed(N)).to(dev, stream)
    with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=regime == "amp"):
        upd = blk.pair_transition(z)
        res, logits = blk.pair_transition.forward_residual_(z.clone(), s2p=blk._s2p_operands(cdt))
        eager = R.transition(z.to(cdt), to(p, dev, cdt)) if regime == "bf16" else R.transition(z, to(p, dev))
    ref = R.transition(z.double(), to(p, dev, torch.float64))
    # single_to_pair reads the stored rows; its operands are rounded to the GEMM dtype
    d = to(sd, dev, torch.float64)
    lref = R.layer_norm(res.double(), d["single_to_pair_norm.weight"], d["single_to_pair_norm.bias"])
    lref = (lref @ d["single_to_pair.weight"].T).movedim(-1, -3)
    if regime == "fp32":
        assert_fp32_close(upd.cpu(), ref.cpu(), what=f"transition N={N}")
        assert_fp32_close(logits.cpu(), lref.cpu(), what=f"logits N={N}")
    else:
        assert_bf16_rule(upd.float().cpu(), eager.float().cpu(), ref.cpu(), f"transition N={N}")
        # two bf16-rounded operands, 128 products: 2^-8 sqrt(2) of the norm at most
        assert (logits.double() - lref).norm() <= 2.0**-7.5 * lref.norm()
    want = z.double() + upd.double()
    tol = (2.0**-7 if stream == BF else 2.0**-22) * want.abs().max().item()
    assert (res.double() - want).abs().max().item() <= tol
