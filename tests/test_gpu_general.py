"""GPU: the general kernels (fp32; bf16 head sizes off the tuned families; key
masks) at the edges of their tiles -- 31, 32 and 33 rows, one row, split and
unsplit row blocks, padded head sizes -- against the fp64 oracle.

Bounds. fp32: every result is a sum of at most N fp32 products, so its relative
error is of the order 2^-24 sqrt(N) (rounding errors of either sign); N is
under 2^13 here, which gives 5.4e-6, doubled for the two chained products.
bf16: nothing but the results is rounded to bf16 (relative error at most 2^-9 =
1.95e-3 each); 2.1e-3 leaves 7% for the fp32 sums. Probabilities or dS held in
bf16 would show here: each alone adds an error of that size."""

from __future__ import annotations

import math

import pytest
import torch

from _helpers import make_inputs, oracle, random_key_mask, rel_l2, tree_of

pytestmark = pytest.mark.gpu

FP32_REL = 1.1e-5
BF16_REL = 2.1e-3

PF_SPLIT = 35  # header word of the plan: waves per row block

# (suffix lengths, prefix, query heads, KV heads)
SHAPES = {
    "one_row": ([1], 1, 2, 1),
    "tile_edges": ([31, 32, 33, 64, 65], 33, 4, 2),
    "no_prefix": ([40, 95], 0, 3, 1),
    "long_prefix_few_rows": ([5], 700, 4, 1),
    "unsplit": ([300, 230], 97, 64, 16),   # 64 heads x (10 + 8) row blocks: one wave each
}
KINDS = [(torch.float32, 64), (torch.float32, 128), (torch.float32, 40), (torch.float32, 256),
         (torch.bfloat16, 96), (torch.bfloat16, 32), (torch.bfloat16, 120), (torch.bfloat16, 200)]
# every padded head size has kernels of its own, split and unsplit, causal and masked


@pytest.mark.parametrize("masked", [False, True], ids=["causal", "masked"])
@pytest.mark.parametrize("dtype, d", KINDS, ids=[f"{str(t).split('.')[1]}_d{d}" for t, d in KINDS])
@pytest.mark.parametrize("shape", list(SHAPES))
def test_general_kernels_match_oracle(shape, dtype, d, masked, cuda_device):
    from bridge_amd import TPRPrefixMeta, tpr_prefix_attention
    lens, prefix, hq, hkv = SHAPES[shape]
    meta = TPRPrefixMeta.shared_prefix(prefix, lens)
    scale = 1.0 / math.sqrt(d)
    plan = meta.plan(hq, hkv, d, dtype, cuda_device, masked=masked)
    assert plan.path == "simt"
    assert (int(plan.host[PF_SPLIT]) == 1) == (shape == "unsplit")
    mask = random_key_mask(tree_of(meta), torch.Generator().manual_seed(d)) if masked else None
    q, k, v, pk, pv, dout = make_inputs(meta, hq, hkv, d, dtype, seed=d + len(shape), device=cuda_device)
    print(f"[general {shape} {dtype} d{d} masked={masked}]", flush=True)
    leaves = [t.clone().requires_grad_(True) for t in (q, k, v, pk, pv)]
    out, lse = tpr_prefix_attention(*leaves, meta, scale, attention_mask=None if mask is None else mask.to(cuda_device))
    out.backward(dout)
    torch.cuda.synchronize()
    ro, rl, rg = oracle(meta, q, k, v, pk, pv, dout, scale, mask=mask)
    bound = FP32_REL if dtype == torch.float32 else BF16_REL
    assert rel_l2(lse, rl) <= FP32_REL
    for name, x, r in zip(("out", "dq", "dk", "dv", "dpk", "dpv"), (out, *(t.grad for t in leaves)), (ro, *rg)):
        if r.numel() == 0 or (shape == "one_row" and name in ("dq", "dk", "dpk")):
            continue  # one row: dS = p (dp - delta) cancels, so its relative error has no such bound
        assert rel_l2(x, r) <= bound, name
