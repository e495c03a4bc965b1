"""dK/dV blocks swept in segments (fa_bwd_gqa with the workspace of
fa_bwd_best_workspace_bytes) on the GPU: against the float64 oracle, against
the unsplit schedule (rounding only), and bit for bit against itself on a
dirty workspace.

Sizes at the edges of the rule and of the split of the flattened (query head,
query tile) list: segments that start inside a head, blocks with fewer tiles
than segments (empty segments), ragged lengths, offsets, both directions of
Sq != Sk, every head dim, causal and not.  Tolerance 1e-2 (fp16) and 4e-2
(bf16) as for every other backward.
"""
from __future__ import annotations

import pytest
import torch

from helpers import TOL, default_scale, max_abs
from oracle import attention as orc
from test_bwd_gpu import _bwd_capi, _bwd_three_launches

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16

# (B, Sq, Sk, H, Hk, D, causal, dtype)
CASES = [
    (1, 700, 700, 14, 2, 128, True, BF16),      # 7 heads to a group, ragged
    (1, 512, 512, 8, 1, 128, True, F16),        # the last blocks: segments without tiles
    (1, 1300, 1300, 4, 4, 128, True, F16),      # equal heads
    (2, 900, 1500, 8, 2, 128, True, F16),       # keys before the first query
    (1, 1500, 700, 8, 2, 128, True, F16),       # queries that see no key
    (1, 777, 777, 14, 2, 64, True, F16),
    (2, 500, 650, 8, 2, 32, True, BF16),
    (1, 1030, 333, 4, 2, 128, False, F16),
    (1, 2100, 500, 4, 1, 64, False, BF16),
    (3, 64, 65, 32, 1, 32, False, F16),         # one tile a head, one key in the last block
]


@pytest.mark.parametrize("case", CASES, ids=["x".join(str(int(x)) for x in c[:7]) for c in CASES])
def test_segments_match_oracle_and_unsplit(case):
    from flash_attn_volta import _capi, flash_attn_forward_gqa
    B, Sq, Sk, H, Hk, D, causal, dtype = case
    print(f"[case] segments {case}", flush=True)
    lib = _capi.load()
    best = lib.fa_bwd_best_workspace_bytes(B, Sq, Sk, H, Hk, D, int(causal))
    minimum = lib.fa_bwd_workspace_bytes(B, Sq, H, D)
    one = 2 * B * Hk * Sk * D * 4
    assert best >= minimum + 2 * one and (best - minimum) % one == 0, "segments must apply"
    q, k, v, do = orc.make_inputs_gqa(B, Sq, Sk, H, Hk, D, seed=17, dtype=dtype)
    sc = default_scale(D, None)
    o_ref, _ = orc.attention_fwd_gqa(q, k, v, causal, sc)
    ref = orc.attention_bwd_gqa(do, q, k, v, causal, sc, o=o_ref)[:3]
    qd, kd, vd, dod = (t.cuda() for t in (q, k, v, do))
    o, lse = flash_attn_forward_gqa(qd, kd, vd, causal=causal, return_softmax_lse=True)
    unsplit = _bwd_capi(dod, qd, kd, vd, o, lse, causal, minimum, 0)
    seg = _bwd_capi(dod, qd, kd, vd, o, lse, causal, best, 0xFF)
    again = _bwd_capi(dod, qd, kd, vd, o, lse, causal, best, 0x00)
    torch.cuda.synchronize()
    tol = TOL if dtype == F16 else 4e-2
    for name, a, r, u, b in zip(("dq", "dk", "dv"), seg, ref, unsplit, again):
        assert max_abs(a, r) < tol, name
        assert max_abs(a, u.float()) < tol / 4, name
        assert torch.equal(a, b), name


def test_noalloc_keeps_its_schedule():
    """fa_bwd_gqa_noalloc gives fa_bwd_gqa's bits at the size
    fa_bwd_gqa_workspace_bytes names also where segments would fit its
    buffer."""
    from flash_attn_volta import _capi, flash_attn_forward_gqa
    from test_zz_no_alloc import _call
    B, S, H, Hk, D = 1, 700, 14, 2, 128
    print("[case] noalloc without segments", flush=True)
    lib = _capi.load()
    size = lib.fa_bwd_gqa_workspace_bytes(B, S, S, H, Hk, D, 1)
    assert size < lib.fa_bwd_best_workspace_bytes(B, S, S, H, Hk, D, 1) < _capi.NOALLOC_SCRATCH_BYTES
    q, k, v, do = (t.cuda() for t in orc.make_inputs_gqa(B, S, S, H, Hk, D, seed=18, dtype=F16))
    o, lse = flash_attn_forward_gqa(q, k, v, causal=True, return_softmax_lse=True)
    ref = _call(lib, "fa_bwd_gqa", do, q, k, v, o, lse, True,
                torch.full((size,), 0xA5, dtype=torch.uint8, device="cuda"))
    got = _call(lib, "fa_bwd_gqa_noalloc", do, q, k, v, o, lse, True)
    for a, b in zip(got, ref):
        assert torch.equal(a, b)


def test_dq_layout_beside_segments():
    """Segments that leave the fused launch leave its dQ layout too: dQ is then
    bit for bit fa_bwd_dq's on the same heads ungrouped, whose grid takes the
    same layout rule (208 blocks of 128 rows: key-split)."""
    from flash_attn_volta import _capi, flash_attn_forward_gqa
    B, S, H, Hk, D = 1, 1600, 16, 4, 128
    print("[case] dQ layout beside segments", flush=True)
    lib = _capi.load()
    best = lib.fa_bwd_best_workspace_bytes(B, S, S, H, Hk, D, 0)
    assert best > lib.fa_bwd_gqa_workspace_bytes(B, S, S, H, Hk, D, 0), "segments must apply"
    q, k, v, do = (t.cuda() for t in orc.make_inputs_gqa(B, S, S, H, Hk, D, seed=19, dtype=F16))
    o, lse = flash_attn_forward_gqa(q, k, v, return_softmax_lse=True)
    dq = _bwd_capi(do, q, k, v, o, lse, False, best, 0xFF)[0]
    ke, ve = (t.repeat_interleave(H // Hk, dim=2).contiguous() for t in (k, v))
    (ref, _, _), _ = _bwd_three_launches(do, q, ke, ve, o, lse, False, default_scale(D, None))
    assert torch.equal(dq, ref)
