"""The fused backward launch without a causal mask: bit for bit the three
separate launches (the same block code), with the workspace that allows no
sweep segments, and against the float64 oracle with the wrapper's workspace.

Sizes on both sides of the launcher's lines: single 64-row blocks, each
layout of the dK/dV and dQ blocks at D = 32 / 64, D = 128 grids that fit the
compute units at once and grids with a mostly empty last round, ragged and
unequal lengths, grouped heads, and neighbours that keep the two kernels.
"""
from __future__ import annotations

import pytest
import torch

from helpers import TOL, default_scale, max_abs
from oracle import attention as orc
from test_bwd_gpu import _bwd_capi, _bwd_three_launches

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16

SQUARE = [
    (3, 64, 5, 64), (1, 65, 2, 64), (1, 1, 1, 32),     # single blocks, the smallest
    (2, 600, 6, 64),                                   # both blocks split
    (4, 500, 12, 64),                                  # dK/dV split, dQ not (under 8 tiles)
    (10, 130, 40, 64),                                 # neither
    (130, 100, 8, 64),                                 # one- and two-tile sweeps: two kernels
    (2, 1000, 25, 32),
    (1, 1500, 8, 128),                                 # one round, key-split dQ blocks
    (2, 1000, 10, 128),                                # one round, whole dQ blocks
    (8, 301, 12, 128),                                 # a mostly empty last round
    (1, 2048, 16, 128),                                # a full round: two kernels
    (16, 197, 12, 128),                                # sweeps under 5 tiles: two kernels
    (1, 3200, 11, 128),                                # 50-tile sweeps, 275 blocks of 512
    (1, 3200, 14, 128),                                # 350 of 512: two kernels
    (1, 3200, 24, 128),                                # 600 of 768
    (1, 3200, 26, 128),                                # 650 of 768: two kernels
]


@pytest.mark.parametrize("B,S,H,D", SQUARE)
def test_fused_full_matches_three_launches(B, S, H, D):
    from flash_attn_volta import _capi, flash_attn_forward
    print(f"[case] fused full B={B} S={S} H={H} D={D}", flush=True)
    lib = _capi.load()
    q, k, v, do = (t.cuda() for t in orc.make_inputs(B, S, H, D, seed=27))
    o, lse = flash_attn_forward(q, k, v, return_softmax_lse=True)
    one = _bwd_capi(do, q, k, v, o, lse, False, lib.fa_bwd_workspace_bytes(B, S, H, D), 0xFF)
    three, blocks = _bwd_three_launches(do, q, k, v, o, lse, False, default_scale(D, None))
    for name, a, b, c in zip(("dq", "dk", "dv"), one, three, blocks):
        assert torch.isfinite(a.float()).all(), name
        assert torch.equal(a, b), f"{name} differs (max-abs {max_abs(a, b.float()):.3e})"
        assert torch.equal(a, c), f"fa_bwd_blocks {name} differs"


# (B, Sq, Sk, H, Hk, D, dtype)
CASES = [
    (2, 65, 700, 6, 6, 64, F16), (2, 700, 65, 6, 6, 64, F16), (1, 1, 300, 4, 4, 64, F16),
    (2, 600, 600, 6, 2, 64, BF16), (4, 500, 333, 12, 12, 64, F16), (1, 1024, 1024, 4, 4, 64, F16),
    (2, 150, 400, 8, 4, 32, BF16), (1, 1500, 700, 4, 4, 128, F16), (2, 333, 1000, 10, 10, 128, BF16),
    (8, 301, 301, 12, 12, 128, F16), (1, 500, 500, 14, 2, 128, BF16),
    (2, 200, 3000, 12, 4, 128, BF16),                  # grouped heads, three quarters of a round
    (2, 200, 3100, 12, 4, 128, F16),                   # more of it: two kernels
    (1, 130, 4600, 64, 8, 128, F16),                   # grouped heads, 288 blocks of 512
]


@pytest.mark.parametrize("case", CASES, ids=["x".join(str(x) for x in c[:6]) for c in CASES])
def test_fused_full_matches_oracle(case):
    from flash_attn_volta import _capi, flash_attn_backward_gqa, flash_attn_forward_gqa
    B, Sq, Sk, H, Hk, D, dtype = case
    print(f"[case] fused full vs oracle {case}", flush=True)
    q, k, v, do = orc.make_inputs_gqa(B, Sq, Sk, H, Hk, D, seed=28, dtype=dtype)
    sc = default_scale(D, None)
    o_ref, _ = orc.attention_fwd_gqa(q, k, v, False, sc)
    ref = orc.attention_bwd_gqa(do, q, k, v, False, sc, o=o_ref)[:3]
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    o, lse = flash_attn_forward_gqa(qd, kd, vd, return_softmax_lse=True)
    got = flash_attn_backward_gqa(dod, qd, kd, vd, o, lse)
    again = flash_attn_backward_gqa(dod, qd, kd, vd, o, lse)
    least = _bwd_capi(dod, qd, kd, vd, o, lse, False,
                      _capi.load().fa_bwd_workspace_bytes(B, Sq, H, D), 0xFF)
    tol = TOL if dtype == F16 else 4e-2
    for name, a, b, c, r in zip(("dq", "dk", "dv"), got, again, least, ref):
        assert max_abs(a, r) < tol, name
        assert torch.equal(a, b), name
        assert max_abs(c, r) < tol, name
