"""The Python wrappers' workspace pool (ops._Workspace) and stream capture, with
a stand-in allocator (no GPU): a buffer that a captured launch was given must
not reach any other call, as the graph goes on writing to it."""

from __future__ import annotations

import pytest
import torch

from vllm_fastdecoder_amd import ops

DEV = torch.device("cuda", 0)


@pytest.fixture
def pool(monkeypatch):
    """A pool on one stream, and the switch that says whether it captures."""
    state = {"capturing": False}
    monkeypatch.setattr(ops, "_current_stream", lambda idx: 7)
    monkeypatch.setattr(ops, "_capturing", lambda: state["capturing"])
    monkeypatch.setattr(ops._Workspace, "_allocate",
                        staticmethod(lambda key, n: torch.empty(n, dtype=torch.uint8)))
    return ops._Workspace(), state


def _ptrs(ws):
    return {b.data_ptr() for b in ws._bufs.values()}


def test_captured_buffers_reach_no_other_call(pool):
    ws, state = pool
    eager = ws.get(DEV, 100)
    state["capturing"] = True
    first, second = ws.get(DEV, 100), ws.get(DEV, 100)  # two graphs of one stream
    assert len({t.data_ptr() for t in (eager, first, second)}) == 3
    state["capturing"] = False
    grown = ws.get(DEV, 1000)  # replaces the eager buffer alone
    assert ws.get(DEV, 100) is grown and _ptrs(ws) == {grown.data_ptr()}


def test_a_first_call_under_capture_leaves_nothing_behind(pool):
    ws, state = pool
    state["capturing"] = True
    held = ws.get(DEV, 100)
    assert held.numel() >= 100 and not ws._bufs
    state["capturing"] = False
    assert ws.get(DEV, 100).data_ptr() != held.data_ptr()


def test_a_reserved_stream_captures_with_its_reservation(pool):
    ws, state = pool
    reserved = ws.get(DEV, 100, pin=True)
    state["capturing"] = True
    assert ws.get(DEV, 60) is reserved
    grown = ws.get(DEV, 200)  # too small a reservation: kept as well
    state["capturing"] = False
    assert [t.data_ptr() for t in ws._pinned[(0, 7)]] == [reserved.data_ptr(), grown.data_ptr()]
