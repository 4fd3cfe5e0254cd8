"""Scratch buffers of the typed wrappers: who shares one, on CPU tensors."""
import pytest
import torch

from pyemma_amd import _native


@pytest.fixture
def on_cpu(monkeypatch):
    state = dict(capturing=False)
    monkeypatch.setattr(_native, "device", lambda: torch.device("cpu"))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state["capturing"])
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
