"""head_dim 16 on its 16 columns (FA_HALF_COLS): against the float64 oracle
and, bit for bit, against the zero-padded general path, whose kernels do the
same sums.

Sizes at tile edges and the smallest ones; one head (rows 32 bytes apart, so a
row past the end lies inside a 64-byte row's extent), transposed and sliced
layouts, decode and chunk key splits, sweep segments, the balanced forward.
"""
from __future__ import annotations

import pytest
import torch

from helpers import TOL, max_abs
from oracle import attention as orc

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16

# (B, Sq, Sk, H, Hk, causal, dtype, layout)
CASES = [
    (1, 1, 1, 1, 1, True, F16, "bshd"),
    (2, 65, 65, 1, 1, True, F16, "bshd"),
    (1, 200, 63, 1, 1, False, BF16, "bshd"),
    (3, 129, 129, 4, 4, True, F16, "bhsd"),
    (2, 128, 300, 6, 3, False, BF16, "sliced"),
    (1, 300, 200, 4, 1, True, F16, "bshd"),        # queries that see no key
    (1, 1, 1000, 8, 2, True, BF16, "bshd"),        # decode, key ranges
    (1, 40, 2500, 8, 2, True, F16, "bhsd"),        # chunk, key ranges
    (1, 2100, 2100, 2, 2, True, F16, "bshd"),      # balanced forward
    (1, 800, 800, 14, 2, True, F16, "bshd"),       # sweep segments
    (40, 197, 197, 8, 8, False, F16, "bhsd"),      # several rounds
]


def _layout(t, name):
    if name == "bhsd":
        return t.transpose(1, 2).contiguous().transpose(1, 2)
    if name == "sliced":      # columns 16.. of wider rows, another row after each
        wide = torch.full((*t.shape[:3], 40), float("nan"), dtype=t.dtype, device=t.device)
        wide[..., 16:32] = t
        return wide[..., 16:32]
    # followed by NaNs: nothing past the last row may be read into a sum
    flat = torch.full((t.numel() + 4096,), float("nan"), dtype=t.dtype, device=t.device)
    flat[:t.numel()] = t.reshape(-1)
    return flat[:t.numel()].view(t.shape)


@pytest.mark.parametrize("case", CASES, ids=["x".join(str(x) for x in c[:6]) + c[7] for c in CASES])
def test_half_columns(case):
    from flash_attn_volta import backward as Bw, forward as F
    from flash_attn_volta import flash_attn_backward_gqa, flash_attn_forward_gqa, flash_attn_gqa
    B, Sq, Sk, H, Hk, causal, dtype, layout = case
    print(f"[case] D = 16 {case}", flush=True)
    cpu = orc.make_inputs_gqa(B, Sq, Sk, H, Hk, 16, seed=61, dtype=dtype)
    q, k, v, do = (_layout(t.cuda(), layout) for t in cpu)
    assert F.fwd_plan(q, k, v, causal, None, True, True) is not F._GENERIC
    o, lse = flash_attn_forward_gqa(q, k, v, causal=causal, return_softmax_lse=True)
    grads = flash_attn_backward_gqa(do, q, k, v, o, lse, causal=causal)
    # the general path pads to 32 columns
    po, plse = F._forward(q, k, v, causal, 0.25, True, True)
    pgrads = Bw._backward(do, q, k, v, po, plse, causal, 0.25, True)
    for a, b in zip((o, lse, *grads), (po, plse, *pgrads)):
        assert a.shape == b.shape and a.is_contiguous() and torch.equal(a, b)
    leaves = [t.detach().clone().requires_grad_() for t in (q, k, v)]
    out = flash_attn_gqa(*leaves, causal=causal)
    for a, b in zip((out, *torch.autograd.grad(out, leaves, do)), (o, *grads)):
        assert torch.equal(a, b)
    ro, _ = orc.attention_fwd_gqa(*cpu[:3], causal, 0.25)
    ref = orc.attention_bwd_gqa(cpu[3], *cpu[:3], causal, 0.25, o=ro)[:3]
    tol = TOL if dtype == F16 else 4e-2
    for a, r in zip((o, *grads), (ro, *ref)):
        assert max_abs(a, r) < tol


def test_reference_signature_and_bounds():
    """The fp16 entry points, and the sizes that keep the padded path or are
    refused."""
    import ctypes

    from flash_attn_volta import _capi, flash_attn, flash_attn_forward
    from flash_attn_volta.forward import planned_dim
    q, k, v, _ = (t.cuda() for t in orc.make_inputs(2, 77, 3, 16, seed=5))
    o = flash_attn_forward(q, k, v, causal=True)
    assert torch.equal(o, flash_attn(q, k, v, causal=True))
    assert max_abs(o, orc.attention_fwd(q.cpu(), k.cpu(), v.cpu(), True)[0]) < TOL
    far = torch.empty_strided((1, 3, 1, 16), (1 << 31, 1 << 30, 16, 1), dtype=F16, device="meta")
    assert not planned_dim(far) and planned_dim(q, k, v)
    lib, P = _capi.load(), 0x10000
    st = (ctypes.c_int64 * 4)(32 * 4 * 64, 32 * 4, 32, 1)
    args = (P, P, P, P, None, 1, 64, 64, 4, 4)
    for D in (64, 128, 16):
        assert lib.fa_fwd_gqa(*args, D, st, st, st, st, 0.1, 1, _capi.FA_HALF_COLS,
                              None) == _capi.FA_ERR_HEAD_DIM
