"""Hooks on saved tensors (torch.autograd.graph): a backward reads whatever
tensors the hooks hand back in those tensors' own layouts, so the gradients are
those of a step without hooks, bit for bit; a tensor of another shape or dtype
is refused."""
from __future__ import annotations

import pytest
import torch
from torch.autograd.graph import save_on_cpu, saved_tensors_hooks

from flash_attn_volta import autograd as A
from flash_attn_volta import rope as R

pytestmark = pytest.mark.gpu

F16, BF16 = torch.float16, torch.bfloat16


def _reversed_dims(t):
    """The same values with the dims stored in the opposite order."""
    n = t.dim()
    return t.permute(*reversed(range(n))).contiguous().permute(*reversed(range(n)))


def _misaligned(t):
    flat = torch.empty(t.numel() + 3, dtype=t.dtype, device=t.device)
    flat[3:] = t.reshape(-1)
    return flat[3:].view(t.shape)


HOOKS = {
    "none": lambda: saved_tensors_hooks(lambda t: t, lambda t: t),
    "save_on_cpu": lambda: save_on_cpu(pin_memory=True),
    "reversed": lambda: saved_tensors_hooks(lambda t: t, _reversed_dims),
    "misaligned": lambda: saved_tensors_hooks(lambda t: t, _misaligned),
}


def _randn(gen, *shape, dtype):
    return torch.randn(shape, generator=gen, device="cuda").to(dtype)


def _qkv(B, Sq, Sk, H, Hk, D, layout, dtype):
    gen = torch.Generator(device="cuda").manual_seed(17)

    def mk(S, h):
        if layout == "bhsd":
            return _randn(gen, B, h, S, D, dtype=dtype).transpose(1, 2)
        if layout == "sliced":     # one part of a wider projection's rows
            return _randn(gen, B, S, 3 * h, D, dtype=dtype)[:, :, h:2 * h]
        return _randn(gen, B, S, h, D, dtype=dtype)
    return mk(Sq, H), mk(Sk, Hk), mk(Sk, Hk), _randn(gen, B, Sq, H, D, dtype=dtype)


def _attn_step(fn, args, causal, hooks):
    q, k, v, do = args
    leaves = [t.detach().requires_grad_() for t in (q, k, v)]
    with hooks():
        out = fn(*leaves, causal, None)
    return [out, *torch.autograd.grad(out, leaves, do)]


@pytest.mark.parametrize("hook", ["save_on_cpu", "reversed", "misaligned"])
@pytest.mark.parametrize("case", [
    (2, 130, 130, 4, 4, 16, "bhsd", False, F16),
    (2, 130, 130, 4, 4, 16, "sliced", True, F16),
    (1, 64, 200, 4, 2, 16, "bhsd", True, BF16),
    (2, 130, 130, 3, 3, 32, "sliced", False, F16),
    (2, 130, 130, 4, 4, 64, "bhsd", True, F16),
    (2, 77, 200, 8, 2, 64, "sliced", True, BF16),
    (1, 200, 200, 4, 4, 128, "bhsd", False, F16),
    (1, 200, 200, 4, 2, 128, "sliced", True, BF16),
], ids=lambda c: "x".join(str(x) for x in c))
def test_attention_gradients(case, hook):
    print(f"[case] hooks {hook} {case}", flush=True)
    *sizes, layout, causal, dtype = case
    B, Sq, Sk, H, Hk, D = sizes
    args = _qkv(*sizes, layout, dtype)
    # the public function (C++ node) and the Python Function behind it
    fns = [(A.flash_attn_gqa, A._FlashAttnGqaFn.apply)]
    if H == Hk and Sq == Sk and dtype == F16:
        fns.append((A.flash_attn, A._FlashAttnFn.apply))
    for node, python in fns:
        want = _attn_step(node, args, causal, HOOKS["none"])
        for fn in (node, python):
            got = _attn_step(fn, args, causal, HOOKS[hook])
            for a, b in zip(got, want):
                assert torch.equal(a, b)


def _rope_step(args, hooks):
    q, k, cos, sin, wq, wk, gq, gk = args
    leaves = [t.detach().requires_grad_() if t is not None else None for t in (q, k, wq, wk)]
    with hooks():
        out = R.apply_rotary_qk(leaves[0], leaves[1], cos, sin, leaves[2], leaves[3], 1e-6)
    return [*out, *torch.autograd.grad(out, [t for t in leaves if t is not None], (gq, gk))]


@pytest.mark.parametrize("hook", ["save_on_cpu", "reversed", "misaligned"])
@pytest.mark.parametrize("norm_q,norm_k", [(True, True), (True, False), (False, False)])
@pytest.mark.parametrize("B,D,layout", [(2, 128, "bhsd"), (1, 64, "sliced"), (2, 16, "bhsd")])
def test_rotary_gradients(B, D, layout, norm_q, norm_k, hook):
    print(f"[case] rope hooks {hook} B={B} D={D} {layout} norms {norm_q} {norm_k}", flush=True)
    S, H, Hk, dtype = 70, 6, 2, BF16
    q, k, _, gq = _qkv(B, S, S, H, Hk, D, layout, dtype)
    gen = torch.Generator(device="cuda").manual_seed(4)
    ang = torch.rand((B, S, D), generator=gen, device="cuda") * 6.3
    both = torch.cat((ang.cos(), ang.sin()), dim=-1).to(dtype)   # tables side by side
    wq, wk = (_randn(gen, D, dtype=dtype) if n else None for n in (norm_q, norm_k))
    args = (q, k, both[..., :D], both[..., D:], wq, wk, gq, _randn(gen, B, S, Hk, D, dtype=dtype))
    assert R._cpp.rope(*args[:6], 1e-6) is not None
    want = _rope_step(args, HOOKS["none"])
    for a, b in zip(_rope_step(args, HOOKS[hook]), want):
        assert torch.equal(a, b)


@pytest.mark.parametrize("unpack", [lambda t: t.float() if t.dtype == F16 else t.double(),
                                    lambda t: t[:, :1]], ids=["dtype", "shape"])
def test_other_tensors_are_refused(unpack):
    q, k, v, do = _qkv(1, 40, 40, 2, 2, 64, "plain", F16)
    leaves = [t.requires_grad_() for t in (q, k, v)]
    for fn in (A.flash_attn, A._FlashAttnFn.apply):
        with saved_tensors_hooks(lambda t: t, unpack):
            out = fn(*leaves, True, None)
        with pytest.raises((RuntimeError, AssertionError)):
            torch.autograd.grad(out, leaves, do)
    ang = torch.rand((1, 40, 64), device="cuda")
    w = torch.ones(64, dtype=F16, device="cuda")
    with saved_tensors_hooks(lambda t: t, lambda t: unpack(t) if t.dim() > 1 else t):
        out = R.apply_rotary_qk(leaves[0], leaves[1], ang.cos().to(F16), ang.sin().to(F16), w, w)
    with pytest.raises(RuntimeError):
        torch.autograd.grad(out, leaves[:2], (do, do))
