"""W4A8Linear's repacked copy is ordered for the stream that uses it (fake
streams and events; the rule itself, without a GPU)."""

import pytest
import torch

from cider_amd import nn, ops


class _Stream:
    def __init__(self, handle):
        self.cuda_stream = handle
        self.waited = []

    def wait_event(self, e):
        self.waited.append(e)


class _Event:
    def record(self, stream):
        self.on = stream


class _Copy:
    def __init__(self):
        self.used_on = []

    def record_stream(self, s):
        self.used_on.append(s)


@pytest.mark.parametrize("capturing", [False, True])
def test_copy_waits_unless_its_stream_ran_it(monkeypatch, capturing):
    lin = nn.W4A8Linear.__new__(nn.W4A8Linear)
    torch.nn.Module.__init__(lin)
    lin.register_buffer("packed_weight", torch.zeros(32, 8, dtype=torch.uint8))
    lin._w4_nk = lin._w4_sig = lin._w4_done = None
    now = {"stream": _Stream(1), "capturing": capturing}
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: now["stream"])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: now["capturing"])
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(ops, "repack_w4_ref", lambda w: _Copy())

    copy = lin._packed_nk()
    made, now["capturing"] = now["stream"], False
    assert lin._packed_nk() is copy
    # made under capture, the copy is not there until a replay: the wait on the
    # captured event refuses the eager call
    assert bool(made.waited) == capturing
    now["stream"] = other = _Stream(2)
    assert lin._packed_nk() is copy
    assert other.waited == [lin._w4_done] and copy.used_on[-1] is other
