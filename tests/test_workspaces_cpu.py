"""Scratch buffers of the typed wrappers: who shares one, on CPU tensors."""
import threading
import types

import pytest
import torch

from pyemma_amd import _native


@pytest.fixture
def on_cpu(monkeypatch):
    state = dict(capturing=False, stream=0, device=0)
    monkeypatch.setattr(_native, "device", lambda: torch.device("cpu"))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: types.SimpleNamespace(cuda_stream=state["stream"],
                                                                                    device_index=state["device"]))
    return state


def test_captured_call_keeps_its_buffer(on_cpu):
    """What a graph captured stays in place when a later call needs more."""
    eager = _native.workspace(1000, "captured")
    on_cpu["capturing"] = True
    held = _native.workspace(1000, "captured")
    on_cpu["capturing"] = False
    assert held.data_ptr() != eager.data_ptr()
    assert _native.workspace(1000, "captured").data_ptr() == eager.data_ptr()
    assert _native.workspace(5000, "captured").data_ptr() != held.data_ptr()


def test_own_buffers_are_not_replaced_by_other_calls(on_cpu):
    own = _native.Workspaces()
    a = _native.workspace(1000, "own", own)
    on_cpu["capturing"] = True
    assert _native.workspace(900, "own", own) is a
    on_cpu["capturing"] = False
    big = _native.workspace(10 ** 6, "own")
    assert big is not a and own.buffers["own"] is a
    assert _native.workspace(1000, "own", own) is a


def test_streams_devices_and_threads_have_their_own(on_cpu):
    a = _native.workspace(1000, "shared")
    assert _native.workspace(500, "shared") is a
    for key, value in (("stream", 77), ("device", 1)):
        old, on_cpu[key] = on_cpu[key], value
        b = _native.workspace(1000, "shared")
        assert b is not a and _native.workspace(1000, "shared") is b
        on_cpu[key] = old
        assert _native.workspace(1000, "shared") is a
    got = []
    th = threading.Thread(target=lambda: got.append(_native.workspace(1000, "shared")))
    th.start()
    th.join()
    assert got[0] is not a
    assert _native.workspace(1000, "shared") is a


def test_number_of_streams_with_buffers_is_bounded(on_cpu):
    first = {}
    for s in range(1000, 1100):
        on_cpu["stream"] = s
        first[s] = _native.workspace(300, "bounded")
    assert len(_native._shared.sets) == _native._SharedWorkspaces.MAX_STREAMS
    assert _native.workspace(300, "bounded") is first[1099]
    on_cpu["stream"] = 1000
    assert _native.workspace(300, "bounded") is not first[1000]
