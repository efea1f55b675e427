"""Which handle a call of autograd.tendencies runs on and how the calls are
ordered, on the CPU with stand-ins for the handle, streams and events."""
import threading

import pytest
import torch

from mam4xx_amd import autograd as ag


class Event:
    def __init__(self):
        self.at = None  # the call this event was recorded after

    def record(self, stream):
        self.at = stream.calls[-1] if stream.calls else None


class Stream:
    def __init__(self, gpu):
        self.gpu, self.calls, self.waited, self.capturing = gpu, [], [], False
        self.cuda_stream = id(self)

    def wait_event(self, event):
        self.waited.append(event.at)


class Gpu:
    """per thread a current stream, as torch has it"""

    def __init__(self):
        self.local, self.made, self.streams, self.ncalls = threading.local(), [], [], 0

    def stream(self):
        self.streams.append(Stream(self))
        return self.streams[-1]

    def chain(self, **kw):
        assert not self.local.stream.capturing, "a handle made during a capture"
        self.made.append(kw)
        return ("chain", len(self.made), kw)


@pytest.fixture
def gpu(monkeypatch):
    g = Gpu()
    g.local.stream = g.stream()
    monkeypatch.setattr(torch.cuda, "current_device", lambda: 0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: g.local.stream)
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing",
                        lambda: g.local.stream.capturing)
    monkeypatch.setattr(ag, "Chain", g.chain)
    monkeypatch.setattr(ag, "_handles", {})
    return g


def call(g, ncell=None):
    with ag._handle(ncell) as ch:
        g.ncalls += 1
        g.local.stream.calls.append(g.ncalls)
        return ch


def test_one_handle_for_all_streams_each_call_after_the_last(gpu):
    chains = set()
    for i in range(200):
        gpu.local.stream = gpu.stream()
        chains.add(id(call(gpu)))
        assert gpu.local.stream.waited == [i or None]
    assert len(chains) == 1 and len(gpu.made) == 2  # it and the captures' one


def test_a_capture_finds_the_handles_of_the_warm_up(gpu):
    eager = call(gpu, 1152)
    gpu.local.stream = gpu.stream()
    gpu.local.stream.capturing = True
    from mam4xx_amd import _abi
    assert call(gpu, 1152)[2] == dict(schedule=_abi.SCHED_FUSED)  # no workspace
    assert call(gpu, 20000) is eager and call(gpu) is eager
    assert gpu.local.stream.waited == []  # events from outside a capture are not waited for
    gpu.local.stream.capturing = False
    gpu.local.stream = gpu.stream()
    call(gpu, 1152)
    assert gpu.local.stream.waited == [1]  # nor are a capture's recorded


def test_a_failed_call_still_orders_the_next(gpu):
    with pytest.raises(ValueError):
        with ag._handle():
            gpu.local.stream.calls.append("failed")
            raise ValueError
    gpu.local.stream = gpu.stream()
    call(gpu)
    assert gpu.local.stream.waited == ["failed"]


def test_threads_share_the_handle_one_call_at_a_time(gpu):
    inside, seen, lock = [], set(), threading.Lock()

    def work():
        gpu.local.stream = gpu.stream()
        for _ in range(50):
            with ag._handle() as ch:
                inside.append(1)
                assert len(inside) == 1
                seen.add(id(ch))
                with lock:
                    gpu.ncalls += 1
                gpu.local.stream.calls.append(gpu.ncalls)
                inside.pop()

    errors = []

    def guarded():
        try:
            work()
        except Exception as e:  # an assertion in a thread
            errors.append(e)

    ts = [threading.Thread(target=guarded) for _ in range(4)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors and len(seen) == 1 and len(gpu.made) == 2
    order = sorted(w for s in gpu.streams for w in s.waited if w is not None)
    assert order == list(range(1, 200))  # every call but the last was waited for, once
