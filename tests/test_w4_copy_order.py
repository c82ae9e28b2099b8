"""W4A8Linear's repacked copy is ordered for the stream that uses it (fake
streams and events; the rule itself, without a GPU)."""

import sys

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


class _MadeOn(_Copy):
    def __init__(self, stream):
        super().__init__()
        self.stream = stream


# Two threads that repack at once: the second one's whole call runs at each line of
# the first one's in turn.  Whichever copy is kept, a later use on a stream that
# did not make it waits.
@pytest.mark.parametrize("line", range(16))
def test_two_repacks_at_once(monkeypatch, line):
    lin = nn.W4A8Linear.__new__(nn.W4A8Linear)
    torch.nn.Module.__init__(lin)
    lin.register_buffer("packed_weight", torch.zeros(32, 8, dtype=torch.uint8))
    lin._w4_nk = lin._w4_sig = lin._w4_done = None
    one, two = _Stream(1), _Stream(2)
    now = [one]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: now[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(ops, "repack_w4_ref", lambda w: _MadeOn(now[0]))
    left = [line]

    def local(frame, event, arg):
        if event == "line":
            left[0] -= 1
            if left[0] == 0:
                sys.settrace(None)
                frame.f_trace = None
                now[0] = two
                lin._packed_nk()
                now[0] = one
        return local

    old = sys.gettrace()
    sys.settrace(lambda frame, event, arg:
                 local if frame.f_code is nn.W4A8Linear._packed_nk.__code__ else None)
    try:
        lin._packed_nk()
    finally:
        sys.settrace(old)
    for s in (one, two):
        now[0] = s
        del s.waited[:]
        copy = lin._packed_nk()
        assert copy.stream is s or [e.on for e in s.waited] == [copy.stream]


def test_copy_of_a_foreign_stream_is_always_waited_for(monkeypatch):
    # a destroyed stream's handle may be a new stream's: the wait stays
    lin = nn.W4A8Linear.__new__(nn.W4A8Linear)
    torch.nn.Module.__init__(lin)
    lin.register_buffer("packed_weight", torch.zeros(32, 8, dtype=torch.uint8))
    lin._w4_nk = lin._w4_sig = lin._w4_done = None
    foreign, later = _Stream(64), _Stream(64)
    foreign.stream_id = later.stream_id = 64
    now = [foreign]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: now[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(ops, "repack_w4_ref", lambda w: _Copy())
    copy = lin._packed_nk()
    now[0] = later
    assert lin._packed_nk() is copy
    assert len(later.waited) == 1 and copy.used_on == [later]
