"""Which memory the expert product works in: the shared workspace that graphs
bake, and a long call's own.  On the CPU, with the library's entries recorded
instead of run."""

import pytest
import torch

from sluice_amd import ops

CPU = torch.device("cpu")
H, I, E, K = 64, 64, 8, 4
CHUNK = 4096 // K


class _Calls:
    """The entries fused_experts uses; records (entry, tokens, workspace, bytes)."""

    def __init__(self):
        self.seen = []

    @staticmethod
    def sluice_fused_experts_workspace(T, H, I, k, shared_I):
        return 4096 * T

    def sluice_fused_experts_bf16(self, *a):
        self.seen.append(("bf16", a[6], a[17], a[18]))
        return 0

    def sluice_fused_experts_prefill(self, *a):
        self.seen.append(("prefill", a[8], a[21], a[22]))
        return 0


@pytest.fixture
def calls(monkeypatch):
    lib = _Calls()
    lib.capturing = False
    monkeypatch.setattr(ops._lib, "load", lambda: lib)
    monkeypatch.setattr(ops, "_stream", lambda device: 0)
    monkeypatch.setattr(ops, "_WS", ops._Workspace())
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: lib.capturing)
    return lib


def _call(T):
    z = dict(dtype=torch.bfloat16)
    return ops._fused_experts_impl(
        torch.zeros((T, H), **z), torch.zeros((E, 2 * I, H), **z), torch.zeros((E, H, I), **z),
        torch.zeros((T, K)), torch.zeros((T, K), dtype=torch.int32), "silu", E, None, None, None,
        None, 1.0, None)


@pytest.mark.parametrize("T", [CHUNK + 1, 3 * CHUNK + 5])
def test_a_long_call_leaves_the_shared_workspace(calls, T):
    """A workspace reserved for one launch stays where it is, whatever the
    length of later calls: graphs captured over it hold its address."""
    ops.reserve_workspace(CPU, CHUNK, H, I, K)
    shared = ops._WS.get(CPU, 1)
    _call(T)
    assert ops._WS.get(CPU, 1) is shared
    assert [(e, n) for e, n, _, _ in calls.seen] == [("prefill", T)]
    assert calls.seen[0][2] != shared.data_ptr() and calls.seen[0][3] >= 4096 * T


def test_a_long_call_uses_a_workspace_reserved_for_it(calls):
    ops.reserve_workspace(CPU, 3 * CHUNK, H, I, K)
    shared = ops._WS.get(CPU, 1)
    _call(3 * CHUNK)
    assert calls.seen == [("prefill", 3 * CHUNK, shared.data_ptr(), shared.numel())]


def test_a_captured_workspace_outlives_its_successor(calls):
    ops.reserve_workspace(CPU, 512, H, I, K)
    shared = ops._WS.get(CPU, 1)
    calls.capturing = True
    _call(500)
    calls.capturing = False
    _call(CHUNK)  # grows the shared one
    assert ops._WS.get(CPU, 1) is not shared
    assert any(t is shared for t in ops._WS.kept)


def test_slices_while_capturing_and_without_memory(calls, monkeypatch):
    """Slices of one launch's tokens; memory that was out is not tried again
    while it is still short."""
    ops.reserve_workspace(CPU, CHUNK, H, I, K)
    shared = ops._WS.get(CPU, 1)
    sliced = [("bf16", n, shared.data_ptr(), shared.numel()) for n in (CHUNK, CHUNK, 7)]
    calls.capturing = True
    _call(2 * CHUNK + 7)
    assert calls.seen == sliced
    calls.capturing = False

    tries, free = [], [0]

    def empty(n, **kw):
        tries.append(n)
        raise torch.OutOfMemoryError("out")

    real = torch.empty
    monkeypatch.setattr(ops, "_PREFILL_OOM", {})
    monkeypatch.setattr(torch.cuda, "memory_reserved", lambda d: 0)
    monkeypatch.setattr(torch.cuda, "memory_allocated", lambda d: 0)
    monkeypatch.setattr(torch.cuda, "mem_get_info", lambda d: (free[0], 1 << 40))
    monkeypatch.setattr(torch, "empty", empty)
    for _ in range(3):
        calls.seen.clear()
        _call(2 * CHUNK + 7)
        assert calls.seen == sliced
    assert len(tries) == 1
    monkeypatch.setattr(torch, "empty", real)
    free[0] = 1 << 40
    calls.seen.clear()
    _call(2 * CHUNK + 7)
    assert [(e, n) for e, n, _, _ in calls.seen] == [("prefill", 2 * CHUNK + 7)]
