"""fp16 decode at D = 128 on grids whose plain forward keeps Q's own bits: the
packed tile keeps them too.  The LSE of rows with large scores shows it: a
product Q * scale rounded to fp16 first moves a score of 36 by some 0.007."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

# (B, Sq, Sk, H, Hk, causal): one key range, and several (few packed tiles)
CASES = [(32, 1, 300, 32, 8, True), (32, 2, 333, 32, 4, True), (16, 1, 260, 64, 8, False),
         (64, 1, 700, 16, 1, True)]


@pytest.mark.parametrize("B,Sq,Sk,H,Hk,causal", CASES)
def test_packed_scores_keep_their_bits(B, Sq, Sk, H, Hk, causal):
    from flash_attn_volta import flash_attn_forward_gqa
    print(f"[case] packed scale {(B, Sq, Sk, H, Hk, causal)}", flush=True)
    D, grp = 128, H // Hk
    gen = torch.Generator().manual_seed(31)
    q, k, v = ((6 * torch.randn(shape, generator=gen)).half()
               for shape in ((B, Sq, H, D), (B, Sk, Hk, D), (B, Sk, Hk, D)))
    _, lse = flash_attn_forward_gqa(q.cuda(), k.cuda(), v.cuda(), causal=causal,
                                    return_softmax_lse=True)
    qh = q.double().view(B, Sq, Hk, grp, D).permute(0, 2, 3, 1, 4).reshape(B, Hk, grp * Sq, D)
    s = (qh @ k.double().permute(0, 2, 3, 1).contiguous() / D ** 0.5).view(B, Hk, grp, Sq, Sk)
    if causal:
        hidden = torch.arange(Sk)[None] > torch.arange(Sq)[:, None] + (Sk - Sq)
        s = s.masked_fill(hidden, float("-inf"))
    ref = torch.logsumexp(s, dim=-1).view(B, H, Sq)
    # a sum of 128 products in fp32: at most 128 * 2^-24 of sum |q k| / sqrt(D),
    # here about 128 * 36 * 0.64 / 11.3 = 260, is 2e-3
    assert (lse.cpu().double() - ref).abs().max().item() < 2e-3
