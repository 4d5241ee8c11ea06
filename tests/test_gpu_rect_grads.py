"""GPU: rectangular_causal_attention against the packed operator it stands on,
called on row slices of the same tensors: outputs and gradients are the same
bit for bit, for packed and strided K/V, with and without a prefix or a mask;
and the check that sends the right-down causal mask to the unmasked kernels."""

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


@pytest.mark.parametrize("sq, skv", [(1, 1), (1, 50), (37, 37), (64, 128), (33, 4099), (300, 517)])
def test_causal_mask_check_sees_every_element(sq, skv, cuda_device):
    from bridge_amd.rectangular_attention import _is_right_down_causal
    cols, rows = torch.arange(skv), torch.arange(sq)
    mask = cols[None, :] > (skv - sq + rows[:, None])
    at = mask.to(cuda_device)
    assert _is_right_down_causal(at)
    assert _is_right_down_causal(mask.t().contiguous().to(cuda_device).t())                 # columns strided
    wide = torch.ones(sq, skv + 5, dtype=torch.bool, device=cuda_device)
    wide[:, 3:skv + 3] = at
    assert _is_right_down_causal(wide[:, 3:skv + 3])                                         # rows strided, odd start
    gen = torch.Generator().manual_seed(sq * skv)
    spots = {(0, 0), (sq - 1, skv - 1), (0, skv - 1), (sq - 1, 0)}
    spots |= {(int(torch.randint(sq, (1,), generator=gen)), int(torch.randint(skv, (1,), generator=gen))) for _ in range(20)}
    for r, c in sorted(spots):
        other = at.clone()
        other[r, c] = ~other[r, c]
        assert not _is_right_down_causal(other), (r, c)
