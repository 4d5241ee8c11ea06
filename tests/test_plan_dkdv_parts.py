"""CPU: the planner's dK/dV parts -- every (key tile, KV head) streams exactly
the query blocks of the whole items, in ordered parts with slots of their own
-- and where they are used."""

import ctypes
from collections import defaultdict

import pytest
import torch

from bridge_amd import TPRPrefixMeta, _lib
from test_gpu_random_trees import random_meta
from test_plan import CPU, decode, tiles_of

N_KPART = 46


def parts_of(w):
    rows = lambda n, off: [tuple(w[w[off] + 8 * i: w[off] + 8 * i + 8]) for i in range(w[n])]  # noqa: E731
    return [r for r in rows(N_KPART, N_KPART + 1) if r[0] >= 0], rows(N_KPART + 2, N_KPART + 3), w[N_KPART + 4]


def ranges(items):
    out = defaultdict(list)
    for it in items:
        if it[5] > it[4]:
            out[it[:4]].append((it[4], it[5]))
    return {k: sorted(v) for k, v in out.items()}


def merged(spans):
    assert all(a[1] == b[0] for a, b in zip(spans, spans[1:]))
    return spans[0][0], spans[-1][1]


def check(plan):
    w, _, dkdv, _ = decode(plan)
    items, reds, slots = parts_of(w)
    whole, parts = ranges(tiles_of(dkdv)), ranges(items)
    assert {k: merged(v) for k, v in whole.items()} == {k: merged(v) for k, v in parts.items()}
    assert {it[:4] for it in items} == {it[:4] for it in tiles_of(dkdv)}  # tiles no query sees write zeros
    assert all(it[5] - it[4] <= 256 and it[7] == 0 for it in items)
    by_slot = {it[6]: it for it in items if it[6] >= 0}
    assert sorted(by_slot) == list(range(slots)) and len(by_slot) == sum(it[6] >= 0 for it in items)
    summed = []
    for src, seg, k0, h, slot0, n, _, _ in reds:
        mine = [by_slot[slot0 + i] for i in range(n)]
        assert n > 1 and all(it[:4] == (src, seg, k0, h) for it in mine)
        assert all(a[5] == b[4] for a, b in zip(mine, mine[1:]))
        summed += range(slot0, slot0 + n)
    assert sorted(summed) == list(range(slots))
    # a tile with a slot is never also written directly
    assert not {it[:4] for it in items if it[6] < 0} & {r[:4] for r in reds}
    return len(items)


def tree_plan(seed, d):
    """A random tree with every leaf four times as long, at a few head layouts."""
    m = random_meta(500 + seed, deep=seed % 3 == 2)
    meta = TPRPrefixMeta(tuple(4 * x for x in m.cu_seqlens_q), m.node_offsets, m.leaf_ancestors)
    return meta.plan(*[(32, 8), (16, 4), (16, 2), (12, 3)][seed % 4], d, torch.bfloat16, CPU)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("seed", range(12))
def test_parts_stream_the_whole_items_blocks(seed, d):
    plan = tree_plan(seed, d)
    if not plan.host[N_KPART]:
        pytest.skip("no parts in this plan")
    check(plan)


def test_the_random_trees_have_parts():
    assert sum(int(tree_plan(seed, d).host[N_KPART]) > 0 for seed in range(12) for d in (64, 128, 256)) >= 34


@pytest.mark.parametrize("d, hq, hkv", [(128, 32, 8), (64, 32, 8), (256, 8, 2), (128, 6, 3)])
def test_parts_only_where_the_chip_is_idle(d, hq, hkv):
    def plan(prefix, lens):
        return TPRPrefixMeta.shared_prefix(prefix, lens).plan(hq, hkv, d, torch.bfloat16, CPU)

    few = plan(200, [4000, 50, 0])
    assert check(few) > 0 and few.host[N_KPART + 4] > 0
    if hkv != 3:
        assert plan(4096, [4096] * 4).host[N_KPART] == 0   # the chip is full
    assert plan(64, [64]).host[N_KPART] == 0               # one block per tile
    # fp32 partials: bounded, behind everything the whole items need
    lib, at = _lib.load(), ctypes.c_void_p(few.host.data_ptr())
    slot = (128 if d == 128 else 64) * d * 8
    assert lib.tpr_attn_bwd_workspace_bytes(at) == few.workspace_bytes
    assert few.bwd_min_bytes == lib.tpr_attn_bwd_min_workspace_bytes(at)
    assert 0 < int(few.host[N_KPART + 4]) * slot <= few.workspace_bytes - few.bwd_min_bytes
    assert int(few.host[N_KPART + 4]) * slot <= 135 << 20
    assert lib.tpr_attn_bwd_min_workspace_bytes(None) == 0
