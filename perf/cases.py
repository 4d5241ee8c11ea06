"""The work that users of this framework have it do, as cases that can be timed
and checked: one attention layer's passes at the sizes of the repository's own
workloads, through the public entry points.

A case's ``kind`` names the entry point:

* ``layer``: ``TPRPrefixAttention`` over all siblings of one shared prefix,
  forward and backward -- a training step's attention layer;
* ``tree``: the same over a rollout tree lowered by ``topology.lower_tree``,
  every segment in one launch;
* ``visit``: the executor's leaf visit, ``TPRKernelBackend`` over a
  ``PrefixKVStack``, forward and backward, the path's gradient added into the
  stack's fp32 rows;
* ``push``: the executor's graph-free forward of a segment (no backward);
* ``rect``: ``rectangular_causal_attention`` on one sequence, forward and
  backward, with or without a physical key mask.

Lengths of siblings are a text of numbers separated by commas.
"""

import math

import torch

from bridge_amd import PrefixKVStack, StackSegment, TPRKernelBackend, TPRPrefixAttention, TPRPrefixMeta
from bridge_amd import rectangular_causal_attention
from bridge_amd.topology import build_trajectory_trees, lower_tree

DTYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _lens(text):
    return [int(x) for x in text.split(",")]


def _join(lens):
    return ",".join(str(n) for n in lens)


def _case(kind, dtype, hq, hkv, d, prefix, suffixes, **more):
    return {"kind": kind, "dtype": dtype, "hq": hq, "hkv": hkv, "d": d, "prefix": prefix,
            "suffixes": _join(suffixes), **more}


def listed():
    # 16 suffix lengths of U[256, 8192], the benchmark's ragged workload
    ragged = torch.randint(256, 8193, (16,), generator=torch.Generator(device="cpu").manual_seed(0)).tolist()
    return [
        # a short turn's leaf visited on its own under a short path: the smallest calls of a schedule
        dict(_case("visit", "bf16", 32, 8, 128, 1500, [100]), name="visit-short"),
        # four ragged siblings visited together under a path of a prompt and several turns
        dict(_case("visit", "bf16", 32, 8, 128, 4096, [1000, 777, 1301, 512]), name="visit-siblings"),
        # the graph-free forward of one turn under a long path (prefill of a segment)
        dict(_case("push", "bf16", 32, 8, 128, 8192, [512]), name="push-turn"),
        # the benchmark's default: the Qwen3-4B layer
        dict(_case("layer", "bf16", 32, 8, 128, 4096, [4096] * 4), name="layer-4k"),
        # the benchmark's long agent session
        dict(_case("layer", "bf16", 32, 8, 128, 32768, [2048] * 8), name="long-session"),
        # the benchmark's ragged batch
        dict(_case("layer", "bf16", 32, 8, 128, 8192, ragged), name="ragged"),
        # the benchmark's rollout tree: 2048 shared, 4 x 1024 shared by 4 rollouts each, 1024 own
        dict(_case("tree", "bf16", 32, 8, 128, 2048, [1024] * 16, branches=4, branch=1024), name="turn-tree"),
        # head_dim 256 and 64 at the benchmark's shapes
        dict(_case("layer", "bf16", 8, 2, 256, 4096, [4096] * 4), name="head256"),
        dict(_case("layer", "bf16", 32, 8, 64, 4096, [4096] * 4), name="head64"),
        # fp32 runs of numerics checks: the benchmark's plumbing shape, and a layer's head layout
        dict(_case("layer", "fp32", 4, 4, 64, 512, [512] * 2), name="fp32-plumbing"),
        dict(_case("layer", "fp32", 32, 8, 128, 1024, [1024] * 2), name="fp32-layer"),
        # one sequence with padded key columns and query rows: the operator's custom-mask mode
        dict(_case("rect", "bf16", 32, 8, 128, 1024, [2048], mask=True, pad_cols=100, pad_rows=60), name="rect-masked"),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


HEADS = [(32, 8), (32, 8), (8, 2), (16, 2), (4, 4), (6, 2)]
MOST_FLOPS = {"mfma": 3.0e13, "other": 3.0e11}  # of a drawn case: below the largest listed one's time


def draw(rng):
    while True:
        kind = rng.choice(["layer", "layer", "layer", "visit", "visit", "push", "rect", "tree"])
        dtype = rng.choice(["bf16", "bf16", "bf16", "fp32"]) if kind in ("layer", "rect") else "bf16"
        hq, hkv = rng.choice(HEADS)
        d = rng.choice([64, 128] if dtype == "fp32" else [64, 96, 128, 128, 128, 256])
        prefix = _log_int(rng, 64, 32768)
        if kind in ("push", "rect"):
            suffixes = [_log_int(rng, 16, 8192)]
        else:
            high = _log_int(rng, 64, 8192)
            suffixes = [_log_int(rng, max(16, high // 16), high) for _ in range(rng.choice([1, 2, 3, 4, 8, 16]))]
        case = _case(kind, dtype, hq, hkv, d, prefix, suffixes)
        if kind == "tree":
            case.update(branches=rng.choice([1, 2, 3, 4]), branch=_log_int(rng, 32, 4096))
        if kind == "rect" and rng.random() < 0.5:
            case.update(mask=True, pad_cols=rng.randrange(0, min(prefix, 200)),
                        pad_rows=rng.randrange(0, min(suffixes[0], 64)))
        slow = dtype == "fp32" or d == 96 or case.get("mask")
        if work(case)["flops"] <= MOST_FLOPS["other" if slow else "mfma"]:
            return case


# ---- the shapes of a case --------------------------------------------------------
def _tree_rows(case):
    """Token rows of the tree's rollouts: root, one of the branches, own tokens; the
    tokens differ from the first one on, so every part is a segment of its own."""
    lens, b = _lens(case["suffixes"]), case["branches"]
    rows = []
    for i, n in enumerate(lens):
        j = i * b // len(lens)
        rows.append(torch.cat([torch.full((case["prefix"],), 1), torch.full((case["branch"],), 100 + j),
                               torch.full((n,), 1000 + i)]))
    return rows


def _launch(case):
    rows = _tree_rows(case)
    (tree,) = build_trajectory_trees([f"u_s_{i}" for i in range(len(rows))], {"input_ids": rows})
    return lower_tree(tree)


def _segments(case):
    """[(query rows a, b, [(first row, last row + 1) of the keys before them])] in the
    packed q rows (and, for the kinds with a prefix of its own, "p" rows)."""
    if case["kind"] != "tree":
        out, a = [], 0
        for n in _lens(case["suffixes"]):
            out.append((a, a + n, [(0, case["prefix"])] if case["prefix"] else []))
            a += n
        return out
    meta, index = _launch_parts(case)
    out = []
    for s, anc in enumerate(meta.leaf_ancestors):
        spans = []
        for n in anc:
            lo, hi = meta.node_offsets[n], meta.node_offsets[n + 1]
            first = int(index[lo])
            spans.append((first, first + hi - lo))  # a node's rows are one segment's packed rows
        out.append((meta.cu_seqlens_q[s], meta.cu_seqlens_q[s + 1], spans))
    return out


def _launch_parts(case):
    launch = _launch(case)
    return launch.meta, launch.prefix_index.tolist()


def _mask(case, device):
    s, p = _lens(case["suffixes"])[0], case["prefix"]
    rows = torch.arange(s, device=device)[:, None]
    cols = torch.arange(p + s, device=device)[None, :]
    hidden = cols > p + rows                                  # right-down causal
    hidden |= (cols >= p - case["pad_cols"]) & (cols < p)     # padded prefix columns
    hidden |= rows >= s - case["pad_rows"]                    # padded query rows
    return hidden


def _pairs(case):
    if case["kind"] == "tree":
        # the branches that some rollout takes (a branch of one rollout alone is part of that leaf)
        lens, b, p, n1 = _lens(case["suffixes"]), case["branches"], case["prefix"], case["branch"]
        own = lambda n, before: n * before + n * (n + 1) // 2  # noqa: E731
        used = sorted({i * b // len(lens) for i in range(len(lens))})
        return own(p, 0) + sum(own(n1, p) for _ in used) + sum(own(n, p + n1) for n in lens)
    p = case["prefix"]
    if case.get("mask"):
        n = _lens(case["suffixes"])[0] - case["pad_rows"]
        return n * (p - case["pad_cols"]) + n * (n + 1) // 2
    return sum(n * p + n * (n + 1) // 2 for n in _lens(case["suffixes"]))


def _rows(case):
    """(query rows, prefix rows that are tensors of their own)"""
    tq = sum(_lens(case["suffixes"]))
    if case["kind"] == "tree":
        used = {i * case["branches"] // len(_lens(case["suffixes"])) for i in range(len(_lens(case["suffixes"])))}
        return tq + case["prefix"] + case["branch"] * len(used), 0
    return tq, case["prefix"]


def work(case):
    es = 2 if case["dtype"] == "bf16" else 4
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    tq, tp = _rows(case)
    if case["kind"] == "push":
        return {"bytes": es * d * (2 * tq * hq + 2 * (tq + tp) * hkv), "flops": 4.0 * hq * d * _pairs(case)}
    # q, dout, k, v, the prefix read; out and every gradient written
    prefix_grad = 2 * 8 if case["kind"] == "visit" else 2 * es  # fp32 rows read and added to
    mask = tq * (tq + tp) if case.get("mask") else 0
    return {"bytes": es * d * (4 * tq * hq + 4 * tq * hkv + 2 * tp * hkv) + prefix_grad * tp * hkv * d + mask,
            "flops": 14.0 * hq * d * _pairs(case)}


# ---- inputs ----------------------------------------------------------------------
def _inputs(case, seed):
    """q, k, v, dout of the packed rows, and the prefix K/V (empty for a tree)."""
    hq, hkv, d, dtype = case["hq"], case["hkv"], case["d"], DTYPES[case["dtype"]]
    tq, tp = _rows(case)
    gen = torch.Generator(device="cuda").manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, device="cuda", generator=gen).to(dtype)

    return [normal(tq, hq, d), normal(tq, hkv, d), normal(tq, hkv, d), normal(tq, hq, d),
            normal(tp, hkv, d), normal(tp, hkv, d)]


def prepare(case, seed):
    q, k, v, dout, pk, pv = _inputs(case, seed)
    kind, scale = case["kind"], 1.0 / math.sqrt(case["d"])
    state = {"kind": kind, "scale": scale, "dout": dout}
    if kind == "layer":
        meta = TPRPrefixMeta.shared_prefix(case["prefix"], _lens(case["suffixes"]))
        return dict(state, meta=meta, leaves=[t.requires_grad_(True) for t in (q, k, v, pk, pv)])
    if kind == "tree":
        launch = _launch(case)
        return dict(state, meta=launch.meta, index=launch.prefix_index.to("cuda"),
                    leaves=[t.requires_grad_(True) for t in (q, k, v)])
    if kind == "rect":
        key, value = torch.cat([pk, k])[:, None], torch.cat([pv, v])[:, None]
        leaves = [t.requires_grad_(True) for t in (q[:, None].contiguous(), key, value)]
        return dict(state, leaves=leaves, mask=_mask(case, "cuda") if case.get("mask") else None,
                    dout=dout.reshape(dout.shape[0], 1, -1))
    p = case["prefix"]
    half = p // 2  # the path: two segments
    stack = PrefixKVStack(p)
    for i, (a, b) in enumerate([(0, half), (half, p)]):
        stack.push(StackSegment(i, i - 1 if i else None, b - a, a, a), {1: (pk[a:b, None], pv[a:b, None])})
    backend = TPRKernelBackend.from_stack(stack, tuple(_lens(case["suffixes"])))
    leaves = [t[:, None] for t in (q, k, v)]
    if kind == "visit":
        leaves = [t.requires_grad_(True) for t in leaves]
    return dict(state, stack=stack, backend=backend, leaves=leaves, dout=dout.reshape(dout.shape[0], 1, -1))


def run(state):
    kind, leaves = state["kind"], state["leaves"]
    if kind == "push":
        with torch.no_grad():
            return state["backend"].attention(1, *leaves, softmax_scale=state["scale"])
    if kind == "visit":
        out = state["backend"].attention(1, *leaves, softmax_scale=state["scale"])
        grads = torch.autograd.grad(out, leaves, state["dout"])
        return (out, *grads, *state["stack"].past_gradient_accumulators()[1])
    if kind == "rect":
        out = rectangular_causal_attention(*leaves, softmax_scale=state["scale"], attention_mask=state["mask"])
        return (out, *torch.autograd.grad(out, leaves, state["dout"]))
    if kind == "tree":
        q, k, v = leaves
        index = state["index"]
        out, lse = TPRPrefixAttention.apply(q, k, v, k.index_select(0, index), v.index_select(0, index),
                                            state["meta"], state["scale"])
    else:
        out, lse = TPRPrefixAttention.apply(*leaves, state["meta"], state["scale"])
    return (out, lse, *torch.autograd.grad(out, leaves, state["dout"]))


# ---- the same in 64 bits ------------------------------------------------------------
def exact(case, seed):
    tensors = _inputs(case, seed)
    q, k, v, dout, pk, pv = (t.double() for t in tensors)
    del tensors
    hq, hkv = case["hq"], case["hkv"]
    group, scale = hq // hkv, 1.0 / math.sqrt(case["d"])
    backward = case["kind"] != "push"
    hidden = _mask(case, "cuda") if case.get("mask") else None
    out, lse = torch.zeros_like(q), q.new_zeros((hq, q.shape[0]))
    dq, dk, dv, dpk, dpv = (torch.zeros_like(t) for t in (q, k, v, pk, pv))
    own = case["kind"] == "tree"  # the keys before a segment are rows of k and v themselves
    before_k, before_v, before_dk, before_dv = (k, v, dk, dv) if own else (pk, pv, dpk, dpv)
    for a, b, spans in _segments(case):
        for h in range(hkv):
            keys = torch.cat([before_k[x:y, h] for x, y in spans] + [k[a:b, h]])
            values = torch.cat([before_v[x:y, h] for x, y in spans] + [v[a:b, h]])
            n_before = keys.shape[0] - (b - a)
            gk, gv = torch.zeros_like(keys), torch.zeros_like(values)
            for g in range(h * group, (h + 1) * group):
                for r0 in range(a, b, 2048):
                    r1 = min(b, r0 + 2048)
                    last = n_before + r1 - a if hidden is None else keys.shape[0]
                    ks, vs = keys[:last], values[:last]
                    s = (q[r0:r1, g] @ ks.T).mul_(scale)
                    if hidden is not None:
                        hide = hidden[r0 - a:r1 - a]
                    else:
                        hide = (torch.arange(last, device="cuda")[None, :]
                                > n_before + torch.arange(r0 - a, r1 - a, device="cuda")[:, None])
                    s.masked_fill_(hide, -math.inf)
                    norm = torch.logsumexp(s, 1, keepdim=True)
                    p = s.sub_(norm.masked_fill(norm == -math.inf, 0.0)).exp_()
                    o = p @ vs
                    out[r0:r1, g] = o
                    lse[g, r0:r1] = norm[:, 0]
                    if not backward:
                        continue
                    do = dout[r0:r1, g]
                    gv[:last] += p.T @ do
                    ds = (do @ vs.T).sub_((do * o).sum(1, keepdim=True)).mul_(p).mul_(scale)
                    dq[r0:r1, g] = ds @ ks
                    gk[:last] += ds.T @ q[r0:r1, g]
            at = 0
            for x, y in spans:
                before_dk[x:y, h] += gk[at:at + y - x]
                before_dv[x:y, h] += gv[at:at + y - x]
                at += y - x
            dk[a:b, h] += gk[at:]
            dv[a:b, h] += gv[at:]
    if case["kind"] == "push":
        return out.reshape(out.shape[0], 1, -1)
    if case["kind"] == "visit":
        return (out.reshape(out.shape[0], 1, -1), dq[:, None], dk[:, None], dv[:, None], dpk, dpv)
    if case["kind"] == "rect":
        return (out.reshape(out.shape[0], 1, -1), dq[:, None], torch.cat([dpk, dk])[:, None],
                torch.cat([dpv, dv])[:, None])
    return (out, lse, dq, dk, dv) if own else (out, lse, dq, dk, dv, dpk, dpv)


def tolerance(case):
    if case["dtype"] == "fp32":
        return {"rel": 1e-5}
    return {"rel": 1e-2}
