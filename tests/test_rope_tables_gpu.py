"""Rotary tables whose strides differ (a contiguous cos beside a sliced sin):
the kernels read both by one stride pair, so the wrapper makes them equal."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("which", ["cos", "sin"])
def test_tables_of_unequal_strides(which):
    from flash_attn_volta import rope_qk_backward, rope_qk_forward
    B, S, H, D = 2, 40, 3, 64
    print(f"[case] strided {which}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, k, gq, gk = (torch.randn(B, S, H, D, generator=gen, device="cuda").half() for _ in range(4))
    ang = torch.rand(1, S, D, generator=gen, device="cuda") * 6.3
    tabs = {"cos": ang.cos().half(), "sin": ang.sin().half()}
    plain = [t.clone() for t in tabs.values()]
    tabs[which] = torch.cat((tabs[which], tabs[which]), dim=-1)[..., :D]
    got = rope_qk_forward(q, k, *tabs.values()) + rope_qk_backward(gq, gk, q, k, *tabs.values())[:2]
    want = rope_qk_forward(q, k, *plain) + rope_qk_backward(gq, gk, q, k, *plain)[:2]
    assert all(torch.equal(a, b) for a, b in zip(got, want))
