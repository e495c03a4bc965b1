"""apply_rotary_qk's C++ node against its general path (the Python Function):
outputs and gradients bit for bit, over the layouts and options the node
takes and those it leaves to the general path; and tables of unequal
strides, which the kernels cannot read, against equal ones."""
from __future__ import annotations

import pytest
import torch

from flash_attn_volta import rope as R

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16

# (B, S, H, Hk, D, q layout, tables, normed q, normed k, dtype)
CASES = [
    (1, 129, 8, 2, 128, "plain", "3d", True, True, BF16),
    (2, 65, 14, 2, 64, "sliced", "per batch", True, False, F16),
    (3, 1, 4, 4, 32, "bhsd", "2d", False, True, BF16),
    (1, 300, 3, 1, 16, "plain", "wide", False, False, F16),
    (2, 40, 4, 2, 128, "misaligned", "3d", True, True, F16),     # general path
    (2, 40, 4, 2, 128, "plain", "float32", True, True, BF16),    # general path
    (2, 40, 4, 2, 64, "plain", "unequal", True, False, BF16),    # general path
]


def _make(case):
    B, S, H, Hk, D, layout, tables, nq, nk, dtype = case
    gen = torch.Generator(device="cuda").manual_seed(3)

    def rn(*shape):
        return torch.randn(shape, generator=gen, device="cuda").to(dtype)
    if layout == "sliced":      # one projection's output, q and k beside each other
        both = rn(B, S, H + Hk, D)
        q, k = both[:, :, :H], both[:, :, H:]
    elif layout == "bhsd":
        q, k = rn(B, H, S, D).transpose(1, 2), rn(B, Hk, S, D).transpose(1, 2)
    elif layout == "misaligned":
        q, k = rn(B * S * H * D + 4)[4:].view(B, S, H, D), rn(B, S, Hk, D)
    else:
        q, k = rn(B, S, H, D), rn(B, S, Hk, D)
    ang = torch.rand(B if tables == "per batch" else 1, S, D, generator=gen, device="cuda") * 6.3
    cos, sin = ang.cos().to(dtype), ang.sin().to(dtype)
    if tables == "2d":
        cos, sin = cos[0], sin[0]
    elif tables == "wide":      # equal strides, not contiguous
        both = torch.cat((cos, sin), dim=-1)
        cos, sin = both[..., :D], both[..., D:]
    elif tables == "float32":
        cos, sin = ang.cos(), ang.sin()
    elif tables == "unequal":
        sin = torch.cat((sin, sin), dim=-1)[..., :D]
        assert sin.stride() != cos.stride()
    wq, wk = rn(D) if nq else None, rn(D) if nk else None
    return q, k, cos, sin, wq, wk, rn(B, S, H, D), rn(B, Hk, S, D).transpose(1, 2)


def _step(apply, q, k, cos, sin, wq, wk, gq, gk):
    leaves = [t.detach().requires_grad_() if t is not None else None for t in (q, k, wq, wk)]
    qo, ko = apply(leaves[0], leaves[1], cos, sin, leaves[2], leaves[3], 1e-6)
    grads = torch.autograd.grad((qo, ko), [t for t in leaves if t is not None], (gq, gk))
    return [qo, ko, *grads]


@pytest.mark.parametrize("case", CASES, ids=["x".join(str(x) for x in c[:7]) for c in CASES])
def test_node_matches_general_path(case):
    print(f"[case] rope node {case}", flush=True)
    args = _make(case)
    taken = R._cpp.rope(*args[:6], 1e-6) is not None
    assert taken == (case[5] != "misaligned" and case[6] not in ("float32", "unequal"))
    got = _step(R.apply_rotary_qk, *args)
    want = _step(R._RopeQkFn.apply, *args)
    assert len(got) == len(want)
    for a, b in zip(got, want):
        assert a.dtype == b.dtype and a.is_contiguous() and torch.equal(a, b)
    if case[6] == "unequal":
        q, k, cos, sin, *rest = args
        same = _step(R.apply_rotary_qk, q, k, cos, sin.contiguous(), *rest)
        for a, b in zip(got, same):
            assert torch.equal(a, b)
    with torch.no_grad():
        a, b = R.apply_rotary_qk(*args[:6], 1e-6), R.rope_qk_forward(*args[:6], 1e-6)
    assert all(torch.equal(x, y) for x, y in zip(a, b))
