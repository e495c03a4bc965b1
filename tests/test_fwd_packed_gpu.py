"""The packed forward on the GPU: the rows of a tile are the (position, head)
pairs of one key/value head's group, in one key range written directly
(fa_fwd_gqa, decode with grouped heads on grids that fill the GPU) or in
several merged ranges (fa_fwd_ws, chunks of queries whose plain grid leaves
compute units idle).

Against the float64 oracle on seeded inputs, at the edges of what the rules
take: one-key caches, queries that see no key (Sk < Sq, causal: O = 0 and
LSE = +inf), groups that do not divide a tile, tiles of several positions,
ragged last tiles, transposed layouts.  Tolerance 1e-2 (fp16) and 4e-2
(bf16) on O and LSE, as for every other forward.
"""
from __future__ import annotations

import numpy as np
import pytest
import torch

from helpers import TOL, default_scale, max_abs
from oracle import attention as orc

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16

# (B, Sq, Sk, H, Hk, D, causal, dtype, transposed)
DIRECT = [
    (32, 1, 201, 32, 8, 128, True, BF16, False),    # one tile per CU, ragged cache
    (128, 1, 1, 14, 2, 64, True, F16, False),       # one key; 7 heads to a group
    (64, 8, 5, 32, 4, 64, True, F16, False),        # 64 rows; 3 positions see no key
    (86, 3, 130, 6, 3, 32, False, F16, True),       # 6-row tiles, all keys, transposed
    (256, 1, 65, 8, 1, 128, True, BF16, True),
]
CHUNKS = [
    (1, 130, 2100, 8, 2, 128, True, BF16, False),   # ragged last tile and range
    (1, 17, 3001, 28, 4, 128, True, F16, False),    # 7 heads: positions straddle tiles
    (2, 100, 5003, 14, 2, 64, True, F16, True),
    (1, 65, 4000, 4, 4, 32, False, F16, False),     # equal heads
    (1, 256, 8448, 8, 8, 64, True, BF16, False),
    (1, 70, 12100, 8, 2, 128, False, BF16, False),  # keys past an XCD's L2
]


def _ids(c):
    return "x".join(str(int(x)) for x in c[:7]) + ("b" if c[7] == BF16 else "h") + "t" * c[8]


def _check(case):
    from flash_attn_volta import flash_attn_forward_gqa
    B, Sq, Sk, H, Hk, D, causal, dtype, transposed = case
    print(f"[packed] case {_ids(case)}", flush=True)
    q, k, v, _ = orc.make_inputs_gqa(B, Sq, Sk, H, Hk, D, seed=41, dtype=dtype)
    qd, kd, vd = (t.cuda() for t in (q, k, v))
    if transposed:
        qd, kd, vd = (t.transpose(1, 2).contiguous().transpose(1, 2) for t in (qd, kd, vd))
    o, lse = flash_attn_forward_gqa(qd, kd, vd, causal=causal, return_softmax_lse=True)
    torch.cuda.synchronize()
    ro, rlse = orc.attention_fwd_gqa(q, k, v, causal, default_scale(D, None))
    tol = TOL if dtype == F16 else 4e-2
    lse = lse.double().cpu().numpy()
    assert np.array_equal(np.isinf(lse), np.isinf(rlse))
    seen = np.isfinite(rlse)
    assert max_abs(o, ro) <= tol and np.abs(lse[seen] - rlse[seen]).max() <= tol


@pytest.mark.parametrize("case", DIRECT, ids=[_ids(c) for c in DIRECT])
def test_packed_tile_written_directly(case):
    from flash_attn_volta import _capi
    B, Sq, Sk, H, Hk, D, causal = case[:7]
    assert _capi.load().fa_fwd_workspace_bytes(B, Sq, Sk, H, Hk, D, int(causal)) == 0
    _check(case)


@pytest.mark.parametrize("case", CHUNKS, ids=[_ids(c) for c in CHUNKS])
def test_chunks_in_merged_key_ranges(case):
    from flash_attn_volta import _capi
    B, Sq, Sk, H, Hk, D, causal = case[:7]
    assert _capi.load().fa_fwd_workspace_bytes(B, Sq, Sk, H, Hk, D, int(causal)) > 0
    assert _capi.load().fa_fwd_splitkv_workspace_bytes(B, Sq, Sk, H, Hk, D) == 0 or H // Hk * Sq <= 64
    _check(case)
