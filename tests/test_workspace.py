"""Growth and retention policy of the per-device scratch buffer
(``kairyu_amd._native.WorkspacePool``), with host tensors standing in for
device memory."""

from __future__ import annotations

import torch

from kairyu_amd._native import WorkspacePool


def _pool(minimum=16):
    state = {"capturing": False, "syncs": 0, "allocs": []}

    def allocate(index, nbytes):
        state["allocs"].append(nbytes)
        return torch.empty(nbytes, dtype=torch.uint8)

    def synchronize(index):
        state["syncs"] += 1

    return WorkspacePool(allocate, lambda index: state["capturing"], synchronize, minimum), state


def test_growth_is_geometric():
    pool, state = _pool()
    for need in range(1, 5000, 7):   # ever larger calls
        assert pool.get(0, need).numel() >= need
    # 16 -> 32 -> ... -> 8192: one allocation per doubling, not one per call
    assert state["allocs"] == [16 * 2 ** i for i in range(10)]
    assert state["syncs"] == len(state["allocs"]) - 1
    assert pool.retained == []           # nothing was captured: all released
    assert WorkspacePool.grown_size(100, 1000, 16) == 1000
    assert WorkspacePool.grown_size(100, 150, 16) == 200


def test_buffers_used_by_a_captured_graph_are_retained_and_bounded():
    pool, state = _pool()
    first = pool.get(0, 10)
    state["capturing"] = True
    assert pool.get(0, 10) is first       # handed to a graph
    state["capturing"] = False
    second = pool.get(0, 100)             # outgrows the captured buffer
    assert pool.retained == [first]
    assert state["syncs"] == 0            # never synchronizes a buffer a graph may use
    third = pool.get(0, 1000)             # `second` was never captured: released
    assert pool.retained == [first]
    assert state["syncs"] == 1
    assert sum(t.numel() for t in pool.retained) < third.numel()
    assert second.numel() == 100


def test_devices_are_independent():
    pool, _ = _pool()
    a, b = pool.get(0, 64), pool.get(1, 128)
    assert a is not b and pool.get(0, 1) is a and pool.get(1, 1) is b


def test_block_fp8_calls_have_scratch_of_their_own(monkeypatch):
    """Block-FP8 linears take the room for their quantized rows from torch's
    allocator, per call: two calls whose scratch is alive at once (two streams,
    two threads) share no byte, and none of the device's shared buffer."""

    from types import SimpleNamespace

    from kairyu_amd import _native
    from kairyu_amd.kernels import quant_gemm_hip as hip

    spans, shared = [], torch.empty(1 << 16, dtype=torch.uint8)
    alive = []

    def call(name, *args):
        at, nbytes = args[-3], args[-2]
        assert nbytes >= 32 * 256 + 32 * 2 * 4
        spans.append((at, at + nbytes))

    empty = torch.empty

    def keep(*args, **kwargs):
        alive.append(empty(*args, **kwargs))
        return alive[-1]

    monkeypatch.setattr(_native, "call", call)
    monkeypatch.setattr(_native, "workspace", lambda device, nbytes=0: shared)
    monkeypatch.setattr(_native, "stream_handle", lambda device: 0)
    monkeypatch.setattr(hip, "_device_index", lambda device: 0)
    monkeypatch.setattr(hip, "_workspace_bytes", lambda entry, index, m, k: m * k + m * k // 32)
    monkeypatch.setattr(hip, "_prepare", lambda x, module, scheme, **kw: (x, empty(32, 64, dtype=x.dtype)))
    monkeypatch.setattr(torch, "empty", keep)
    module = SimpleNamespace(weight=empty(64, 256, dtype=torch.uint8), weight_scale_inv=empty(1, 2), bias=None,
                             in_features=256, out_features=64, _add_local_bias=lambda: True)
    x = empty(32, 256, dtype=torch.bfloat16)
    hip.block_fp8_linear_forward(x, module)
    hip.block_fp8_linear_forward(x, module)
    hip.block_fp8_swiglu_forward(x, module, module)
    spans.append((shared.data_ptr(), shared.data_ptr() + shared.numel()))
    spans.sort()
    assert len(spans) == 4 and all(a[1] <= b[0] for a, b in zip(spans, spans[1:]))
