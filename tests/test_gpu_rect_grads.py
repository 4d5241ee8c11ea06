"""GPU: rectangular_causal_attention against the packed operator it stands on,
called on row slices of the same tensors: outputs and gradients are the same
bit for bit, for packed and strided K/V, with and without a prefix or a mask."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _leaves(sq, skv, hq, hkv, d, dtype, device, strided):
    gen = torch.Generator().manual_seed(sq + skv)
    wide = torch.randn(skv, 1, 2 * hkv, d, generator=gen).to(device, dtype)
    k, v = (wide[:, :, :hkv], wide[:, :, hkv:]) if strided else (wide[:, :, :hkv].contiguous(), wide[:, :, hkv:].contiguous())
    q = torch.randn(sq, 1, hq, d, generator=gen).to(device, dtype)
    return [t.detach().requires_grad_(True) for t in (q, k, v)]


@pytest.mark.parametrize("strided", [False, True], ids=["packed", "strided"])
@pytest.mark.parametrize("masked", [False, True], ids=["causal", "mask"])
@pytest.mark.parametrize("sq, skv, d, dtype", [(70, 211, 128, torch.bfloat16), (65, 65, 64, torch.bfloat16),
                                               (33, 40, 8, torch.bfloat16), (40, 100, 72, torch.float32)])
def test_rect_equals_sliced_prefix_attention(sq, skv, d, dtype, masked, strided, cuda_device):
    from bridge_amd import TPRPrefixAttention, TPRPrefixMeta, rectangular_causal_attention
    leaves = _leaves(sq, skv, 4, 2, d, dtype, cuda_device, strided)
    mask = None
    if masked:
        mask = torch.rand(sq, skv, generator=torch.Generator().manual_seed(1)).to(cuda_device) < 0.3
    print(f"[rect {sq}x{skv} d{d} masked={masked} strided={strided}]", flush=True)
    out = rectangular_causal_attention(*leaves, attention_mask=mask)
    dout = torch.randn(out.shape, generator=torch.Generator().manual_seed(2)).to(cuda_device, dtype)
    grads = torch.autograd.grad(out, leaves, dout)
    q, k, v = (t.squeeze(1) for t in leaves)
    p = skv - sq
    ref, _ = TPRPrefixAttention.apply(q, k[p:], v[p:], k[:p], v[:p], TPRPrefixMeta.shared_prefix(p, [sq]), None, None,
                                      False, None, mask)
    want = torch.autograd.grad(ref, leaves, dout.reshape(ref.shape))
    assert torch.equal(out, ref.reshape(out.shape))
    for name, a, b in zip(("dq", "dk", "dv"), grads, want):
        assert a.shape == b.shape and torch.equal(a, b), name
