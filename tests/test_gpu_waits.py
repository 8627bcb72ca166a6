"""Which waits of one stream for another a schedule issues: none twice, and at its end one per stream."""
import pytest
import torch

from dynaflow_amd.runtime.device import HipDevice

pytestmark = pytest.mark.gpu


class Counted(torch.cuda.Event):
    waits = 0

    def wait(self, stream=None):
        Counted.waits += 1
        super().wait(stream)


def test_waits_are_not_repeated(monkeypatch):
    monkeypatch.setattr(torch.cuda, "Event", Counted)
    monkeypatch.setattr(Counted, "waits", 0)
    device = HipDevice()
    first, second = device.new_stream(), device.new_stream()
    (start, other) = device.starts(2)
    assert start is other
    start.wait(first), start.wait(first), start.wait(second), start.wait(first)
    assert Counted.waits == 2
    start.wait()                                     # the stream that it was recorded on
    assert Counted.waits == 2
    start.record(first)                              # recorded again: to be waited for again
    start.wait(second), start.wait(first)
    assert Counted.waits == 3


def test_the_last_event_of_a_stream_stands_for_those_before_it():
    device = HipDevice()
    streams = [device.new_stream(), device.new_stream()]
    events = [device.new_event() for _ in range(4)]
    for event, stream in zip((events[2], events[0], events[1], events[3]), (streams[0], streams[1], streams[0], streams[0])):
        event.record(stream)
    assert device.tails(events[:1]) == events[:1]
    assert device.tails(events) == [events[0], events[3]]
    assert device.tails([events[1], events[2]]) == [events[1]]


def test_results_are_there_after_the_forward():
    """The caller's stream reads what both nano-batches wrote behind long kernels on the other streams."""
    device = HipDevice()
    streams = [device.new_stream(), device.new_stream()]
    x, out = torch.randn(4096, 4096, device="cuda"), [torch.zeros(4096, device="cuda") for _ in range(3)]
    want = (x @ x @ x)[0]
    starts = device.starts(3)
    events = []
    for i, start in enumerate(starts):
        stream = streams[i % 2]
        with device.stream(stream):
            start.wait(stream)
            out[i].copy_((x @ x @ x)[0])
            events.append(device.new_event())
            events[-1].record()
    for event in device.tails(events):
        event.wait()
    for got in out:
        assert torch.equal(got, want)
