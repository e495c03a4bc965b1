"""head_dim 16 at the sizes where its 16-column rows end: a head (and a tile of
128 rows) of 2^31 bytes and more, in a tensor's own layout or in the
contiguous one of the output or a gradient, runs on padded copies."""
from __future__ import annotations

import pytest
import torch

from flash_attn_volta.forward import planned_dim

F16 = torch.float16


def _meta(shape, stride):
    return torch.empty_strided(shape, stride, dtype=F16, device="meta")


@pytest.mark.parametrize("S,H,stride,planned", [
    (1000, 4, 64, True),
    ((1 << 20) + 1, 64, 16, False),        # transposed: small rows, but a contiguous out of 2^31
    (1 << 20, 64, 16, True),
    ((1 << 20) + 1, 64, 64 * 16, False),
    (129, 2, 1 << 23, False),
    (129, 2, (1 << 23) - 8, True),
    (2, 2, 1 << 23, True),                 # a tile of 128 rows ends at 127 strides
    (2, 2, 1 << 24, False),
    (1, 2, 1 << 40, True),                 # one row: its stride is never used
])
def test_planned_sizes(S, H, stride, planned):
    assert planned_dim(_meta((1, S, H, 16), (1 << 42, stride, S * 16, 1))) == planned


@pytest.mark.gpu
def test_wide_contiguous_output():
    """q transposed, rows of 32 bytes: its contiguous output spans 2 GiB a head."""
    from flash_attn_volta import flash_attn_forward_gqa
    print("[case] D = 16, an output of 2 GiB", flush=True)
    S, H = (1 << 20) + 1, 64
    gen = torch.Generator(device="cuda").manual_seed(2)
    q = torch.randn((1, H, S, 16), generator=gen, device="cuda", dtype=F16).transpose(1, 2)
    k, v = (torch.randn((1, 40, 2, 16), generator=gen, device="cuda", dtype=F16) for _ in range(2))
    out = flash_attn_forward_gqa(q, k, v)
    for i in (0, S // 2, S - 200):
        part = flash_attn_forward_gqa(q[:, i:i + 200], k, v)
        assert (out[:, i:i + 200].float() - part.float()).abs().max().item() < 1e-2


@pytest.mark.gpu
@pytest.mark.parametrize("S,stride", [(129, 1 << 23), (3, 1 << 24)])
def test_upstream_gradient_of_long_strides(S, stride):
    from flash_attn_volta import flash_attn, flash_attn_gqa
    print(f"[case] D = 16, dO of stride {stride}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v, do = (torch.randn((1, S, 2, 16), generator=gen, device="cuda", dtype=F16)
                   for _ in range(4))
    far = torch.empty((S - 1) * stride + 32, device="cuda", dtype=F16).as_strided(
        (1, S, 2, 16), (0, stride, 16, 1)).copy_(do)
    for fn in (flash_attn, flash_attn_gqa):
        leaves = [t.detach().requires_grad_() for t in (q, k, v)]
        out = fn(*leaves, causal=True)
        got = torch.autograd.grad(out, leaves, far, retain_graph=True)
        for a, b in zip(got, torch.autograd.grad(out, leaves, do)):
            assert torch.equal(a, b)
