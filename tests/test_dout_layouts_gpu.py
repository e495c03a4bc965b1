"""The autograd node's upstream gradient in the layouts a program hands it:
read in place where the kernels can, copied where they cannot; either way the
gradients are those of the contiguous copy, bit for bit."""
from __future__ import annotations

import pytest
import torch

from oracle import attention as orc

pytestmark = pytest.mark.gpu

B, S, H, D = 2, 200, 4, 64


def _layout(name, do):
    """A tensor equal to `do` (or, broadcast layouts, to its own contiguous
    copy) in the named layout."""
    if name == "contiguous":
        return do
    if name == "bhsd":
        return do.transpose(1, 2).contiguous().transpose(1, 2)
    if name == "sbhd":
        return do.transpose(0, 1).contiguous().transpose(0, 1)
    if name == "last dim strided":
        return do.transpose(2, 3).contiguous().transpose(2, 3)
    if name == "wide rows":
        wide = torch.zeros(B, S, H, 2 * D, dtype=do.dtype, device=do.device)
        wide[..., D:] = do
        return wide[..., D:]
    if name == "odd stride":
        wide = torch.zeros(B, S, H, D + 4, dtype=do.dtype, device=do.device)
        wide[..., :D] = do
        return wide[..., :D]
    if name == "misaligned":
        flat = torch.zeros(do.numel() + 4, dtype=do.dtype, device=do.device)
        flat[4:] = do.reshape(-1)
        return flat[4:].view(do.shape)
    if name == "one batch broadcast":
        return do[:1].expand(B, S, H, D)
    if name == "scalar broadcast":
        return do[:1, :1, :1, :1].expand(B, S, H, D)
    return do.float()   # another dtype


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("name", ["bhsd", "sbhd", "last dim strided", "wide rows", "odd stride",
                                  "misaligned", "one batch broadcast", "scalar broadcast",
                                  "float32"])
def test_upstream_gradient_layout(name, causal):
    from flash_attn_volta import flash_attn, flash_attn_gqa
    print(f"[case] dO {name} causal={causal}", flush=True)
    q, k, v, do = (t.cuda() for t in orc.make_inputs(B, S, H, D, seed=21))
    given = _layout(name, do)
    if name == "float32":
        plain = do
    else:
        plain = given.contiguous().clone()
        assert given.stride() != plain.stride() or given.data_ptr() % 16
    for fn in (flash_attn, flash_attn_gqa):
        got, want = [], []
        for upstream, grads in ((given, got), (plain, want)):
            leaves = [t.clone().requires_grad_() for t in (q, k, v)]
            # (a float32 upstream gradient reaches the node through a cast
            # of its output)
            out = fn(*leaves, causal=causal)
            grads += torch.autograd.grad(out.to(upstream.dtype), leaves, upstream)
        for a, b in zip(got, want):
            assert torch.equal(a, b)
