"""The forward's layouts on both sides of the launcher's lines (grid sizes of
128-row workgroups at, just under and just over each), against float32 torch
attention on the same inputs: head dims 64 and 128, causal and not, ragged
lengths, fp16 and bf16.

Bound: probabilities and the output are each rounded to the element type once
(2^-11 and 2^-8 relative), and |O| <= max|V|, so |O - ref| <= 4 units of that
rounding of max|V|."""
from __future__ import annotations

import math

import pytest
import torch

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16

# (B, Sq, Sk, H, Hk, D, causal, dtype)
CASES = [
    (1, 8192, 8192, 8, 2, 128, True, BF16),       # eight waves, 256 rows
    (1, 8191, 8191, 8, 8, 128, True, F16),
    (1, 8100, 8100, 9, 9, 128, True, F16),        # 64 blocks of 128 rows, ragged
    (2, 2048, 2048, 16, 16, 128, False, F16),     # one full round of 256-row workgroups
    (2, 2048, 2100, 16, 4, 128, False, BF16),
    (1, 2048, 2048, 17, 17, 128, False, F16),
    (1, 2048, 2048, 33, 33, 128, True, F16),      # over two workgroups per CU
    (5, 1500, 1500, 9, 9, 128, True, BF16),
    (1, 4096, 4096, 17, 17, 64, False, F16),      # key split past one round
    (2, 1024, 1024, 32, 32, 64, False, F16),      # eight waves, one round
    (3, 333, 1100, 64, 64, 64, False, BF16),
    (1, 2100, 2100, 40, 8, 64, True, F16),
]


def _reference(q, k, v, causal):
    """float32, one head at a time."""
    B, Sq, H, D = q.shape
    Sk, grp = k.shape[1], H // k.shape[2]
    out = torch.empty(q.shape, dtype=torch.float32, device=q.device)
    mask = torch.ones(Sq, Sk, dtype=torch.bool, device=q.device).tril(Sk - Sq) if causal else None
    for b in range(B):
        for h in range(H):
            s = q[b, :, h].float() @ k[b, :, h // grp].float().T / math.sqrt(D)
            if causal:
                s.masked_fill_(~mask, -math.inf)
            out[b, :, h] = torch.softmax(s, dim=-1) @ v[b, :, h // grp].float()
    return out


@pytest.mark.parametrize("case", CASES, ids=["x".join(str(int(x)) for x in c[:7]) for c in CASES])
def test_forward_layouts(case):
    from flash_attn_volta import flash_attn_forward_gqa
    B, Sq, Sk, H, Hk, D, causal, dtype = case
    print(f"[case] forward layout {case}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(9)
    q, k, v = (torch.randn(B, S, h, D, generator=gen, device="cuda").to(dtype)
               for S, h in ((Sq, H), (Sk, Hk), (Sk, Hk)))
    out = flash_attn_forward_gqa(q, k, v, causal=causal)
    err = (out.float() - _reference(q, k, v, causal)).abs().max().item()
    unit = 2.0 ** -11 if dtype == F16 else 2.0 ** -8
    assert err <= 4 * unit * v.float().abs().max().item(), err
