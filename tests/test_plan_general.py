"""CPU: the general kernels' forward / dQ work items on the random prefix trees
of the planner tests -- every (leaf, token, query head) in exactly one row
block -- for both ways a row block is run (one wave, or several that share its
keys), every type and padded head size."""

import math
from collections import Counter

import pytest
import torch

from bridge_amd import TPRPrefixMeta
from test_plan import CPU, PF, decode
from test_plan_random_trees import _case, _leaf_len

PF_SPLIT = 35
SPLIT = {(torch.float32, 64): 8, (torch.float32, 128): 4, (torch.float32, 256): 2, (torch.bfloat16, 32): 8,
         (torch.bfloat16, 96): 8, (torch.bfloat16, 128): 8, (torch.bfloat16, 200): 4}


def check_items(meta, hq, hkv, d, dtype, masked):
    plan = meta.plan(hq, hkv, d, dtype, CPU, masked=masked)
    assert plan.path == "simt"
    w, fwd, _, _ = decode(plan)
    split = w[PF_SPLIT]
    blocks = sum(-(-_leaf_len(meta, s) // 32) for s in range(meta.num_leaves)) * hq
    assert split == (1 if blocks >= 1024 else SPLIT[dtype, d])
    hpw = math.gcd(hq // hkv, 4) if split == 1 else 1
    tokens = 32 * (4 // hpw) if split == 1 else 32
    covered = Counter()
    for leaf, tok0, qh0, kvh in fwd:
        if leaf < 0:
            continue
        assert kvh == qh0 // (hq // hkv) and qh0 % hpw == 0 and tok0 % tokens == 0
        for h in range(qh0, qh0 + hpw):
            for t in range(tok0, min(tok0 + tokens, _leaf_len(meta, leaf)), 32):
                covered[leaf, t, h] += 1
    expected = {(s, t, h) for s in range(meta.num_leaves) for t in range(0, _leaf_len(meta, s), 32) for h in range(hq)}
    assert set(covered) == expected and set(covered.values()) <= {1}
    return split


@pytest.mark.parametrize("dtype, d", list(SPLIT))
@pytest.mark.parametrize("seed", range(6))
def test_row_blocks_of_random_trees(seed, dtype, d):
    meta, hq, hkv = _case(seed)
    for masked in (False, True) if (dtype, d) != (torch.bfloat16, 128) else (True,):
        check_items(meta, hq, hkv, d, dtype, masked)


@pytest.mark.parametrize("lens, split", [([1], False), ([992], False), ([993], True), ([500, 500], True),
                                         ([1024] * 4, True)])
def test_split_by_row_blocks(lens, split):
    meta = TPRPrefixMeta.shared_prefix(100, lens)
    assert (check_items(meta, 32, 8, 64, torch.float32, False) == 1) == split
