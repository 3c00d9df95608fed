"""GPU: the fused pair-weighted MSA averaging (bf16 operands, 64 MSA channels in 8 heads; 64,
128 or 256 pair channels; reference ``attention.py:272-341``): tiles of 64 queries / keys and 8
sequences cut by N and S, columns no sequence holds, both streams, a batch of two, the in-place
residual, and an unaligned MSA (which takes the batched GEMMs). Against the oracle in fp64 by
the bf16 rule; batch items bit for bit independent."""

from __future__ import annotations

import pytest
import torch

from oracle import pairformer_ref as R
from tests._helpers import assert_bf16_rule, mod, sub, to

pytestmark = pytest.mark.gpu
W = mod("weights")
attention = mod("attention")
BF = torch.bfloat16


def _module(dev, cz, seed):
    p = sub(W.make_evoformer_block_weights(seed, perturb_affine=True, c_pair=cz), "row_attn.")
    m = attention.MSAAttention(64, cz).eval()
    m.load_state_dict(p)
    return m.to(dev), p


def _inputs(dev, B, S, N, cz, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    msa = torch.randn(B, S, N, 64, generator=g).to(dev, dtype)
    pair = torch.randn(B, N, N, cz, generator=g).to(dev, dtype)
    mask = (torch.rand(B, S, N, generator=g) > 0.2).float()
    mask[:, :, N // 2 :: 5] = 0.0  # columns no sequence holds
    mask[:, 0, 0] = 1.0
    return msa, mask.to(dev), pair


@pytest.mark.parametrize("stream", [BF, torch.float32], ids=["bf16", "fp32"])
@pytest.mark.parametrize("S,N,B,cz", [(1, 1, 1, 128), (7, 15, 1, 128), (8, 64, 2, 128), (9, 65, 1, 64),
                                      (130, 33, 1, 128), (20, 150, 1, 256)])  # fmt: skip
def test_msa_attention_fused(dev, S, N, B, cz, stream):
    print(f"[pav fused] S={S} N={N} B={B} cz={cz} {stream}", flush=True)
    m, p = _module(dev, cz, 11 + N)
    msa, mask, pair = _inputs(dev, B, S, N, cz, stream, S + N)
    with torch.no_grad(), torch.autocast("cuda", dtype=BF, enabled=stream == torch.float32):
        got = m(msa, mask, pair)
        last = m(msa[-1:], mask[-1:], pair[-1:])
        res = m.forward_residual_(msa.clone(), mask, pair)
        eager = R.msa_attention(msa.to(BF), mask, pair.to(BF), to(p, dev, BF))
    ref = R.msa_attention(msa.double(), mask.double(), pair.double(), to(p, dev, torch.float64))
    assert got.dtype == stream and torch.equal(last, got[-1:])
    print("   ", assert_bf16_rule(got.cpu(), eager.float().cpu(), ref.cpu(), f"pav S={S} N={N}"), flush=True)
    want = msa.double() + got.double()  # one rounding of msa + update, against the separately rounded update
    tol = (2.0**-7 if stream == BF else 2.0**-22) * want.abs().max().item()
    assert (res.double() - want).abs().max().item() <= tol


def test_msa_attention_unaligned(dev):
    print("[pav] MSA 2 bytes off a 16-byte boundary", flush=True)
    m, _ = _module(dev, 128, 5)
    msa, mask, pair = _inputs(dev, 1, 12, 40, 128, BF, 6)
    off = torch.empty(msa.numel() + 1, dtype=BF, device=dev)[1:].view(msa.shape).copy_(msa)
    with torch.no_grad():
        a, b = m(msa, mask, pair).float(), m(off, mask, pair).float()
    # two bf16 evaluations with the same roundings of every intermediate, sums in another order
    assert (a - b).norm() <= 4e-3 * a.norm()
