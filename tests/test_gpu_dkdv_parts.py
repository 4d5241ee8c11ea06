"""GPU: dK/dV with its query ranges cut into parts, against the fp64 oracle and
against the whole items (a workspace without room for the parts).

Bounds. Parts change only the order of fp32 sums (1e-5 of the result's norm)
and, through it, the last bf16 bit of some elements (2^-8 of the element):
parts against whole items, relative L2 at most 2^-8 over all rows and in each.
Against the oracle: P (or dS), one operand and the result are rounded to bf16,
three independent errors of at most 2^-9 each, 3.4e-3 in all; dS also takes
delta from the rounded output, and dP - delta cancels where a row has few keys
(a one-row prefix measured 3.8e-3 of dK): twice that."""

from __future__ import annotations

import math

import pytest
import torch

from _helpers import make_inputs, oracle, rel_l2

pytestmark = pytest.mark.gpu

BF16_REL = 2 * 3.4e-3
ULP = 2.0 ** -8
N_KPART = 46


def _metas():
    from bridge_amd import TPRPrefixMeta as M
    return {
        "one_leaf": M.shared_prefix(1, [1500]),              # tiles cut across their causal diagonal
        "ragged": M.shared_prefix(130, [700, 0, 33, 450]),   # node parts over several leaves
        "no_prefix": M.shared_prefix(0, [1281, 3]),
        "tree": M(cu_seqlens_q=(0, 333, 398, 1138, 1155), node_offsets=(0, 130, 200, 270),
                  leaf_ancestors=((0, 1), (0, 1), (0, 2), (0, 2))),
    }


@pytest.mark.parametrize("relay", [False, True], ids=["bf16", "relay"])
@pytest.mark.parametrize("d, recompute", [(128, False), (128, True), (256, False), (64, False)],
                         ids=["d128", "d128_recompute", "d256", "d64"])
@pytest.mark.parametrize("name", ["one_leaf", "ragged", "no_prefix", "tree"])
def test_dkdv_parts_match_oracle_and_whole_items(name, d, recompute, relay, cuda_device):
    from bridge_amd import prefix_attention_backward, prefix_attention_forward
    meta = _metas()[name]
    hq, hkv = (6, 2) if name == "ragged" else (4, 2)
    scale = 1.0 / math.sqrt(d)
    plan = meta.plan(hq, hkv, d, torch.bfloat16, cuda_device, recompute_dq=recompute)
    assert plan.host[N_KPART] > 0 and plan.workspace_bytes > plan.bwd_min_bytes
    q, k, v, pk, pv, dout = make_inputs(meta, hq, hkv, d, torch.bfloat16, seed=11 + d, device=cuda_device)
    print(f"[dK/dV parts {name} d{d} recompute={recompute} relay={relay}] {int(plan.host[N_KPART])} items, "
          f"{int(plan.host[N_KPART + 4])} slots", flush=True)
    out, lse = prefix_attention_forward(q, k, v, pk, pv, meta, scale)

    def backward(size):
        acc = tuple(torch.full(pk.shape, 0.25, dtype=torch.float32, device=cuda_device) for _ in range(2)) if relay else None
        room = torch.full((size + (1 << 20),), 0x5a, dtype=torch.uint8, device=cuda_device)
        grads = prefix_attention_backward(q, k, v, pk, pv, out, lse, dout, meta, scale, recompute_dq=recompute,
                                          prefix_grad_accumulators=acc, buffers={"workspace": room[:size]})
        assert bool((room[size:] == 0x5a).all()), "written past the workspace"
        return grads

    parts, again = backward(plan.workspace_bytes), backward(plan.workspace_bytes)
    whole = backward(plan.bwd_min_bytes)
    torch.cuda.synchronize()
    _, _, ref = oracle(meta, q, k, v, pk, pv, dout, scale)
    for i, label in enumerate(("dq", "dk", "dv", "dprefix_k", "dprefix_v")):
        assert torch.equal(parts[i], again[i]), label
        if parts[i].numel() == 0:
            continue
        want = ref[i] + 0.25 if relay and i >= 3 else ref[i]
        assert rel_l2(parts[i], want) <= BF16_REL, label
        assert rel_l2(whole[i], want) <= BF16_REL, label
        # rows on their own: a part left out or added twice hides in a norm over all rows
        p, w = parts[i].double().flatten(1), whole[i].double().flatten(1)
        assert rel_l2(p, w) <= ULP, label
        err = (p - w).norm(dim=1) / w.norm(dim=1).clamp_min(1e-2 * w.norm() / math.sqrt(len(w)))
        assert err.max().item() <= ULP, label


@pytest.mark.parametrize("d", [128, 64])
@pytest.mark.parametrize("tiles_full", [True, False], ids=["tiles_full", "tiles_least"])
def test_separate_steps_do_not_depend_on_each_others_workspace(tiles_full, d, cuda_device):
    """The tiles step and the reduction step, enqueued separately with the full
    workspace for one and the least for the other: dK, dV and dQ are those of one
    call with the size that the step which writes them was given, bit for bit."""
    from bridge_amd import _lib, prefix_attention_backward, prefix_attention_forward
    meta, hq, hkv, scale = _metas()["ragged"], 6, 2, 1.0 / math.sqrt(d)
    plan = meta.plan(hq, hkv, d, torch.bfloat16, cuda_device)
    assert plan.host[N_KPART] > 0
    q, k, v, pk, pv, dout = make_inputs(meta, hq, hkv, d, torch.bfloat16, seed=5, device=cuda_device)
    out, lse = prefix_attention_forward(q, k, v, pk, pv, meta, scale)
    size = {True: plan.workspace_bytes, False: plan.bwd_min_bytes}
    print(f"[dK/dV steps d{d} tiles_full={tiles_full}]", flush=True)

    def backward(room, full, **more):
        return prefix_attention_backward(q, k, v, pk, pv, out, lse, dout, meta, scale,
                                         buffers={"workspace": room[:size[full]], **more.pop("buffers", {})}, **more)

    def room():
        return torch.full((plan.workspace_bytes,), 0xff, dtype=torch.uint8, device=cuda_device)  # floats read as NaN

    one = {full: backward(room(), full) for full in (True, False)}
    names = ("dq", "dk", "dv", "dprefix_k", "dprefix_v")
    mine = {n: torch.full_like(t, math.nan) for n, t in zip(names, one[True])}
    ws, mine["delta"] = room(), torch.empty_like(lse)
    for phase, full in ((_lib.TPR_BWD_DELTA, not tiles_full), (_lib.TPR_BWD_DKDV_TILES, tiles_full),
                        (_lib.TPR_BWD_DKDV_REDUCE, not tiles_full), (_lib.TPR_BWD_DQ, tiles_full)):
        backward(ws, full, phases=phase, buffers=mine)
    torch.cuda.synchronize()
    for name, want in zip(names, one[tiles_full]):
        assert torch.equal(mine[name], want), name
