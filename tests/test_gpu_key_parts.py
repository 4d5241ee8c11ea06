"""GPU: the key parts of calls with few query rows (the forward and dQ cut along
the keys over several workgroups, summed from the caller's workspace), against
the fp64 oracle and against the same call without a workspace.

Bound: the bf16 kernels round P (or dS), one operand and the result to bf16,
three independent errors of at most 2^-9 each: relative L2 at most
sqrt(3) 2^-9 = 3.4e-3. The cut changes the sums' order (fp32) and the maximum
P is rounded against, nothing else."""

from __future__ import annotations

import ctypes
import math
from unittest import mock

import pytest
import torch

from _helpers import make_inputs, oracle, rel_l2

pytestmark = pytest.mark.gpu

BF16_REL = 3.4e-3
PF = dict(N_FPART=36, N_QPART=41)


def _metas():
    from bridge_amd import TPRPrefixMeta as M
    n = 11  # a path laid out leaf first: one key run per node, more than the kernels hold in registers
    lens = [97 + 30 * i for i in range(n)]
    off = [0]
    for x in lens:
        off.append(off[-1] + x)
    return {
        "one_row": M.shared_prefix(1500, [1]),
        "ragged": M.shared_prefix(1601, [70, 0, 33]),
        "suffix_only": M.shared_prefix(0, [900]),
        "run_list": M(cu_seqlens_q=(0, 40, 61), node_offsets=tuple(off),
                      leaf_ancestors=(tuple(range(n - 1, -1, -1)), tuple(range(n - 1, 4, -1)))),
    }


@pytest.mark.parametrize("strided", [False, True], ids=["packed", "strided"])
@pytest.mark.parametrize("d, recompute", [(128, False), (256, False), (256, True), (64, False)],
                         ids=["d128", "d256", "d256_recompute", "d64"])
@pytest.mark.parametrize("name", ["one_row", "ragged", "suffix_only", "run_list"])
def test_key_parts_match_oracle_and_whole_items(name, d, recompute, strided, cuda_device):
    from bridge_amd import _lib, prefix_attention_backward, prefix_attention_forward
    meta = _metas()[name]
    hq, hkv = (4, 2) if name != "ragged" else (6, 2)
    scale = 1.0 / math.sqrt(d)
    plan = meta.plan(hq, hkv, d, torch.bfloat16, cuda_device, recompute_dq=recompute)
    assert plan.host[PF["N_FPART"]] > 0 and plan.fwd_workspace_bytes > 0 and plan.host[PF["N_QPART"]] > 0
    q, k, v, pk, pv, dout = make_inputs(meta, hq, hkv, d, torch.bfloat16, seed=7 + d, device=cuda_device)
    if strided:  # views of wider rows
        q, k, v = (torch.cat([t, t[:, :1]], 1)[:, :t.shape[1]] for t in (q, k, v))
    print(f"[key parts {name} d{d} recompute={recompute} strided={strided}] {int(plan.host[PF['N_FPART']])} forward, "
          f"{int(plan.host[PF['N_QPART']])} dQ parts", flush=True)
    out, lse = prefix_attention_forward(q, k, v, pk, pv, meta, scale)
    grads = prefix_attention_backward(q, k, v, pk, pv, out, lse, dout, meta, scale, recompute_dq=recompute)
    # the same without a workspace: whole items
    whole, whole_lse = torch.empty_like(out), torch.empty_like(lse)
    strides = [0 if t.is_contiguous() else t.stride(0) for t in (q, k, v)]
    params = _lib.TprFwdParams(_lib.ABI_VERSION, 0, scale, 0.0, plan.host.data_ptr(), plan.device.data_ptr(),
                               *(t.data_ptr() if t.numel() else None for t in (q, k, v, pk, pv, whole, whole_lse)),
                               *strides, None, 0)
    stream = ctypes.c_void_p(torch.cuda.current_stream(cuda_device).cuda_stream)
    _lib.check(_lib.load().tpr_attn_fwd(ctypes.byref(params), stream), "tpr_attn_fwd")
    torch.cuda.synchronize()
    ro, rl, rg = oracle(meta, q, k, v, pk, pv, dout, scale)
    assert rel_l2(lse, rl) <= 1e-6 and rel_l2(whole_lse, rl) <= 1e-6
    assert rel_l2(out, ro) <= BF16_REL and rel_l2(whole, ro) <= BF16_REL
    assert rel_l2(grads[0], rg[0]) <= BF16_REL
    # every row on its own: a part added twice or left out hides in a norm over all rows
    err = (out.double().cpu() - ro).norm(dim=2) / ro.norm(dim=2)
    assert err.max().item() <= 3 * BF16_REL


def test_forward_without_memory_for_its_parts_runs_whole_items(cuda_device):
    """The workspace cannot be allocated (host side, forced): the result is that
    of the call without one, bit for bit, with and without a backward to follow."""
    from bridge_amd import TPRPrefixMeta, _lib, prefix_attention_forward, tpr_prefix_attention
    meta, d = TPRPrefixMeta.shared_prefix(1500, [100]), 128
    plan = meta.plan(32, 8, d, torch.bfloat16, cuda_device)
    q, k, v, pk, pv, _ = make_inputs(meta, 32, 8, d, torch.bfloat16, seed=2, device=cuda_device)
    whole, whole_lse = torch.empty_like(q), torch.empty(32, 100, dtype=torch.float32, device=cuda_device)
    params = _lib.TprFwdParams(_lib.ABI_VERSION, 0, 1.0 / math.sqrt(d), 0.0, plan.host.data_ptr(), plan.device.data_ptr(),
                               *(t.data_ptr() for t in (q, k, v, pk, pv, whole, whole_lse)), 0, 0, 0, None, 0)
    stream = ctypes.c_void_p(torch.cuda.current_stream(cuda_device).cuda_stream)
    _lib.check(_lib.load().tpr_attn_fwd(ctypes.byref(params), stream), "tpr_attn_fwd")
    real, asked = torch.empty, []

    def empty(size, *args, **kwargs):
        if kwargs.get("dtype") == torch.uint8:
            asked.append(size)
            raise torch.OutOfMemoryError("no memory")
        return real(size, *args, **kwargs)

    with mock.patch.object(torch, "empty", empty):
        out, lse = prefix_attention_forward(q, k, v, pk, pv, meta)
        leaf = q.clone().requires_grad_(True)
        out2, _ = tpr_prefix_attention(leaf, k, v, pk, pv, meta)
    torch.cuda.synchronize()
    assert asked == [plan.fwd_workspace_bytes] * 2
    assert torch.equal(out, whole) and torch.equal(out2, whole) and torch.equal(lse, whole_lse)


def test_key_parts_are_deterministic_and_replay(cuda_device):
    """Two runs agree bit for bit, and so does a captured forward on each replay."""
    from bridge_amd import TPRPrefixMeta, prefix_attention_forward
    meta = TPRPrefixMeta.shared_prefix(3000, [50])
    q, k, v, pk, pv, _ = make_inputs(meta, 8, 2, 128, torch.bfloat16, seed=3, device=cuda_device)
    first, lse = prefix_attention_forward(q, k, v, pk, pv, meta)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        again, lse2 = prefix_attention_forward(q, k, v, pk, pv, meta)
    for _ in range(3):
        again.zero_()
        graph.replay()
        eager, _ = prefix_attention_forward(q, k, v, pk, pv, meta)
        torch.cuda.synchronize()
        assert torch.equal(again, first) and torch.equal(eager, first) and torch.equal(lse, lse2)
