"""CPU: the planner's key parts -- every tile of every forward / dQ item in
exactly one part, partial slots used once and summed by one merge, no parts
where whole items fill the chip -- and the forward workspace's checks."""

import ctypes
import random
from collections import defaultdict

import pytest
import torch

from bridge_amd import TPRPrefixMeta, _lib
from test_gpu_random_trees import random_meta
from test_plan import CPU, PF, decode, key_runs

N_FPART, N_QPART = 36, 41


def parts_of(w, at):
    """({(leaf, tok, qh, kvh): [(tile0, tiles, slot)]}, {(...): (slot0, parts)}, slots)"""
    items, merges = defaultdict(list), {}
    for i in range(w[at]):
        leaf, tok, qh, kvh, t0, n, slot, _ = w[w[at + 1] + 8 * i: w[at + 1] + 8 * i + 8]
        if leaf >= 0:
            items[leaf, tok, qh, kvh].append((t0, n, slot))
    for i in range(w[at + 2]):
        leaf, tok, qh, kvh, _, n, slot, _ = w[w[at + 3] + 8 * i: w[at + 3] + 8 * i + 8]
        assert (leaf, tok, qh, kvh) not in merges
        merges[leaf, tok, qh, kvh] = (slot, n)
    return items, merges, w[at + 4]


def check_parts(w, at, expected):
    """expected: {(leaf, tok, qh, kvh): tiles of its key stream}"""
    items, merges, slots = parts_of(w, at)
    assert set(items) == set(expected)
    used = []
    for key, parts in items.items():
        parts.sort()
        assert parts[0][0] == 0 and all(n > 0 for _, n, _ in parts)
        assert all(a + n == b for (a, n, _), (b, _, _) in zip(parts, parts[1:]))
        assert parts[-1][0] + parts[-1][1] == expected[key]
        if len(parts) == 1:
            assert parts[0][2] == -1 and key not in merges
        else:
            slot0, n = merges.pop(key)
            assert n == len(parts) and [s for _, _, s in parts] == list(range(slot0, slot0 + n))
            used += [s for _, _, s in parts]
    assert not merges and sorted(used) == list(range(slots))


def long_meta(seed):
    """A random tree of the planner tests with every node 40 times as long."""
    m = random_meta(300 + seed, deep=seed % 3 == 2)
    return TPRPrefixMeta(m.cu_seqlens_q, tuple(40 * x for x in m.node_offsets), m.leaf_ancestors)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("seed", range(9))
def test_parts_cover_every_tile_once(seed, d):
    meta = long_meta(seed)
    hq, hkv = [(8, 2), (4, 4), (6, 2)][seed % 3]
    for recompute in (False, True):
        plan = meta.plan(hq, hkv, d, torch.bfloat16, CPU, recompute_dq=recompute)
        w, fwd, _, _ = decode(plan)
        _, runs = key_runs(plan)
        g = hq // hkv
        length = [b - a for a, b in zip(meta.cu_seqlens_q, meta.cu_seqlens_q[1:])]

        def tokens(first_two, rows):  # tokens of an item: rows / heads
            heads = max(h for h in range(1, rows[0] + 1) if g % h == 0 and rows[0] % h == 0)
            return rows[1] * (rows[0] // heads)

        def tiles(item, tok_per_item):
            leaf, tok = item[:2]
            own = min(length[leaf], tok + tok_per_item)
            return -(-own // 64) + sum(-(-n // 64) for _, n in runs[leaf])

        if w[N_FPART]:
            per = tokens(None, (8 if d == 128 else 4, 32))
            check_parts(w, N_FPART, {it: tiles(it, per) for it in fwd if it[0] >= 0})
        if w[N_QPART] and plan.dq_from_ds:
            kt = 128 if d == 128 else 64
            per = tokens(None, (8, 64 if d == 128 else 32))
            dqs = [tuple(w[w[PF["OFF_DQS"]] + 4 * i: w[PF["OFF_DQS"]] + 4 * i + 4]) for i in range(w[PF["N_DQS"]])]
            no = meta.node_offsets
            check_parts(w, N_QPART, {
                it: -(-min(length[it[0]], it[1] + per) // kt)
                + sum(-(-(no[n + 1] - no[n]) // kt) for n in meta.leaf_ancestors[it[0]])
                for it in dqs if it[0] >= 0})
        elif w[N_QPART]:
            assert d != 128
            per = tokens(None, (4, 32))
            check_parts(w, N_QPART, {it: tiles(it, per) for it in fwd if it[0] >= 0})


@pytest.mark.parametrize("d, hq, hkv", [(128, 32, 8), (64, 32, 8), (256, 8, 2)])
def test_parts_only_where_rows_are_few(d, hq, hkv):
    def counts(prefix, lens):
        plan = TPRPrefixMeta.shared_prefix(prefix, lens).plan(hq, hkv, d, torch.bfloat16, CPU)
        w = plan.host.tolist()
        assert (plan.fwd_workspace_bytes > 0) == (w[N_FPART] > 0)
        assert plan.fwd_workspace_bytes <= 160 << 20
        return w[N_FPART], w[N_QPART]

    assert counts(4096, [4096] * 4) == (0, 0)           # the chip is full
    assert counts(100, [64]) == (0, 0)                  # too few tiles to cut
    few = counts(16384, [64])
    assert few[0] >= 64 and few[1] >= 64


def test_partial_slots_are_bounded():
    """At most 192 MiB of partial slots in the forward and in dQ, also where the
    items (just under four rounds of the chip) would be cut into many."""
    rng = random.Random(5)
    shapes = [(40, 8, 128, 60000, [5541]), (16, 2, 256, 40000, [6305]), (32, 8, 128, 32768, [7000]), (32, 8, 64, 60000, [20000])]
    for _ in range(40):
        hq, hkv, d = rng.choice([(32, 8, 128), (40, 8, 128), (16, 2, 128), (16, 2, 256), (8, 2, 256), (32, 8, 64)])
        rows = rng.randrange(400, 1024) * 256 // hq  # 400 to 1023 items of 256 rows
        shapes.append((hq, hkv, d, rng.randrange(8192, 65536), [rows // 3, rows - rows // 3]))
    cut = 0
    for hq, hkv, d, prefix, lens in shapes:
        for recompute in (False, True):
            plan = TPRPrefixMeta.shared_prefix(prefix, lens).plan(hq, hkv, d, torch.bfloat16, CPU, recompute_dq=recompute)
            w = plan.host.tolist()
            dq_rows = (512 if d == 128 else 256) if plan.dq_from_ds else 128
            assert plan.fwd_workspace_bytes <= 192 << 20
            assert w[N_QPART + 4] * dq_rows * d * 4 <= 192 << 20
            cut += w[N_FPART] > 0
    assert cut >= 10


def test_forward_workspace_checks():
    plan = TPRPrefixMeta.shared_prefix(8192, [64]).plan(32, 8, 128, torch.bfloat16, CPU)
    lib = _lib.load()
    need = lib.tpr_attn_fwd_workspace_bytes(ctypes.c_void_p(plan.host.data_ptr()))
    assert need == plan.fwd_workspace_bytes > 0 and lib.tpr_attn_fwd_workspace_bytes(None) == 0
    p = _lib.TprFwdParams(_lib.ABI_VERSION, 0, 1.0, 0.0, plan.host.data_ptr(), plan.host.data_ptr(),
                          *([4096] * 7), 0, 0, 0, None, 0)
    for ws, size, status in ((4096, need - 1, _lib.TPR_ERR_BUFFER_TOO_SMALL), (4096 + 16, need, _lib.TPR_ERR_INVALID_ARGUMENT)):
        assert lib.tpr_attn_fwd_ws(ctypes.byref(p), ctypes.c_void_p(ws), size, None) == status
