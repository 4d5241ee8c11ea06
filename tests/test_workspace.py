"""CPU: the backward's workspace on the host -- a caller's buffer counts with
the bytes it has, one too small is refused before a launch, and where the
allocator fails the smaller sizes are tried in turn and nothing is kept alive."""

import ctypes
import gc
import weakref
from unittest import mock

import pytest
import torch

from bridge_amd import TPRPrefixMeta, _lib
from bridge_amd.prefix_attention import _workspace

CPU = torch.device("cpu")


def _inputs():
    """A plan with dQ and dK/dV parts: its full workspace is larger than the least."""
    meta = TPRPrefixMeta.shared_prefix(1, [1500])
    q, k = (torch.empty(1500, h, 128, dtype=torch.bfloat16) for h in (4, 2))
    plan = meta.plan(4, 2, 128, torch.bfloat16, CPU)
    assert 0 < plan.bwd_min_bytes < plan.workspace_bytes
    return meta, q, k, plan


def test_a_given_workspace_counts_with_its_own_bytes():
    meta, q, k, plan = _inputs()
    for size in (plan.workspace_bytes, plan.bwd_min_bytes, plan.bwd_min_bytes - 256, 0):
        room = torch.empty(plan.workspace_bytes + 4096, dtype=torch.uint8)
        for ws in (room[:size], room[256:256 + size], torch.empty(size // 4, dtype=torch.float32)):
            got = _workspace(meta, q, k, None, ws)
            assert got[1] is ws and got[2] == size
    # no more than the storage holds, whatever the view's shape says
    assert _workspace(meta, q, k, None, torch.empty(16, dtype=torch.uint8).expand(1 << 20, 16))[2] == 16


@pytest.mark.parametrize("short", [0, 1, 256])
def test_less_than_the_least_is_refused_before_a_launch(short):
    *_, plan = _inputs()
    at = plan.host.data_ptr()
    b = _lib.TprBwdParams(_lib.ABI_VERSION, 0, 1.0, 0.0, at, at, *([4096] * 14), 4096, plan.bwd_min_bytes - short,
                          0, 0, 0, None, 0)
    if short == 0:
        b.workspace = 4096 + 16  # enough, but misaligned: the next check
    status = _lib.load().tpr_attn_bwd(ctypes.byref(b), None)
    assert status == (_lib.TPR_ERR_BUFFER_TOO_SMALL if short else _lib.TPR_ERR_INVALID_ARGUMENT)


def _failing_empty(fails):
    """torch.empty that runs out of memory on its first ``fails`` calls; the sizes asked for."""
    real, asked = torch.empty, []

    def empty(size, *args, **kwargs):
        asked.append(size)
        if len(asked) <= fails:
            raise torch.OutOfMemoryError("no memory")
        return real(size, *args, **kwargs)

    return mock.patch.object(torch, "empty", empty), asked


@pytest.mark.parametrize("fails", range(5))
def test_out_of_memory_tries_smaller_sizes_and_keeps_nothing_alive(fails):
    meta, q, k, plan = _inputs()
    flat = meta.plan(4, 2, 128, torch.bfloat16, CPU, ds_store_budget=0)
    sizes = [plan.workspace_bytes, plan.bwd_min_bytes, flat.workspace_bytes, flat.bwd_min_bytes]
    assert plan.dq_from_ds and not flat.dq_from_ds and len(set(sizes)) == 4

    def caller():
        """(weak references to a caller's tensors, what it got or raised)"""
        mine = torch.zeros(8)
        patch, asked = _failing_empty(fails)
        with patch:
            try:
                got_plan, ws, size = _workspace(meta, q, k, None, None)
            except torch.OutOfMemoryError:
                return [weakref.ref(mine)], None, asked
        assert size == ws.numel() == sizes[fails]
        return [weakref.ref(mine), weakref.ref(ws)], got_plan, asked

    gc.collect()
    gc.disable()
    try:
        refs, got_plan, asked = caller()
        alive = [r() is not None for r in refs]
    finally:
        gc.enable()
    assert asked == sizes[:fails + 1]
    assert got_plan is ([plan, plan, flat, flat] + [None])[fails]
    assert not any(alive)
