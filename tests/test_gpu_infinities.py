"""GPU: infinite elements in the general kernels (fp32; bf16 head sizes off the
tuned families; key masks). A probability or dS times an infinity is that
infinity, as in one fp32 product -- also where bf16 carries the probability in
three terms, also where it is exactly 1 -- and rows past a tile's end add
nothing. Against the fp64 oracle: the same NaN, +inf and -inf elements, and the
other elements within the general kernels' bounds (test_gpu_general.py).

Every infinity is placed where no query that does not see it could meet it
(the last prefix row; the output gradient of a leaf's last row, which sees all
of the leaf's keys; under the mask nothing is hidden): a hidden 0 x inf is NaN."""

from __future__ import annotations

import math

import pytest
import torch

from _helpers import make_inputs, oracle, rel_l2

pytestmark = pytest.mark.gpu

FP32_REL, BF16_REL = 1.1e-5, 2.1e-3
KINDS = [(torch.float32, 64, False), (torch.float32, 256, False), (torch.bfloat16, 96, False), (torch.bfloat16, 32, False),
         (torch.bfloat16, 200, False), (torch.bfloat16, 128, True), (torch.float32, 128, True)]
SHAPES = {"split": ([40, 7], 33, 4, 2), "unsplit": ([300, 230], 97, 64, 16)}  # prefix and leaves end inside a tile


def _same(got, want, bound, name):
    got, want = got.double().cpu(), want.double().cpu()
    for what in (torch.isnan, torch.isposinf, torch.isneginf):
        assert torch.equal(what(got), what(want)), (name, what.__name__)
    finite = torch.isfinite(want)
    assert rel_l2(got[finite], want[finite]) <= bound, name


@pytest.mark.parametrize("dtype, d, masked", KINDS, ids=[f"{str(t).split('.')[1]}_d{d}{'_mask' * m}" for t, d, m in KINDS])
@pytest.mark.parametrize("shape", list(SHAPES))
@pytest.mark.parametrize("where", ["value", "dout"])
def test_infinities_stay_infinities(where, shape, dtype, d, masked, cuda_device):
    from bridge_amd import TPRPrefixMeta, prefix_attention_backward, prefix_attention_forward
    lens, prefix, hq, hkv = SHAPES[shape]
    meta = TPRPrefixMeta.shared_prefix(prefix, lens)
    scale = 1.0 / math.sqrt(d)
    bound = FP32_REL if dtype == torch.float32 else BF16_REL
    mask = torch.zeros(meta.total_q, meta.max_keys(), dtype=torch.bool) if masked else None
    on_gpu = None if mask is None else mask.to(cuda_device)
    q, k, v, pk, pv, dout = make_inputs(meta, hq, hkv, d, dtype, seed=3 + d, device=cuda_device)
    if where == "value":
        pv[-1, 0, 3], pv[-1, 1, d - 1] = math.inf, -math.inf
    else:
        last = meta.cu_seqlens_q[1] - 1
        dout[last, 0, 5], dout[last, hq - 1, d - 1] = math.inf, -math.inf
    print(f"[infinity {where} {shape} {dtype} d{d} masked={masked}]", flush=True)
    out, lse = prefix_attention_forward(q, k, v, pk, pv, meta, scale, attention_mask=on_gpu)
    grads = prefix_attention_backward(q, k, v, pk, pv, out, lse, dout, meta, scale, attention_mask=on_gpu)
    torch.cuda.synchronize()
    ro, rl, rg = oracle(meta, q, k, v, pk, pv, dout, scale, mask=mask)
    assert rel_l2(lse, rl) <= FP32_REL
    _same(out, ro, bound, "out")
    if where == "value":
        assert torch.isposinf(ro[:, 0, 3]).all()  # every query sees the last prefix row
        names = ("dv", "dprefix_v")               # dS is NaN or infinite in every row: nothing to compare in dq and dk
    else:
        assert torch.isposinf(rg[4][:, 0, 5]).all() and torch.isinf(rg[3]).any()
        names = ("dq", "dk", "dv", "dprefix_k", "dprefix_v")
    for name, got, want in zip(("dq", "dk", "dv", "dprefix_k", "dprefix_v"), grads, rg):
        if name in names:
            _same(got, want, bound, name)


@pytest.mark.parametrize("dtype, d", [(torch.bfloat16, 96), (torch.bfloat16, 200), (torch.float32, 64)])
def test_one_key_returns_its_value(dtype, d, cuda_device):
    """P is exactly 1: the output is the value row, infinities included."""
    from bridge_amd import TPRPrefixMeta, prefix_attention_forward
    meta = TPRPrefixMeta.shared_prefix(0, [1])
    q, k, v, pk, pv, _ = make_inputs(meta, 4, 2, d, dtype, seed=1, device=cuda_device)
    v[0, 0, 0], v[0, 1, 7] = math.inf, -math.inf
    out, _ = prefix_attention_forward(q, k, v, pk, pv, meta)
    assert torch.equal(out, v.repeat_interleave(2, dim=1))
