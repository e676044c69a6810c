"""How recorded decode steps go away, with stand-ins for the device: at once when they are dropped, by whomever, and after
a wait for the device, which may still be running them."""
import gc
from types import SimpleNamespace as NS

import pytest
import torch

from ferrox_amd.engine.runner import DecodeGraph, ModelRunner


@pytest.fixture
def made(monkeypatch):
    """(makes a runner with n recorded steps, what happened to them in order); the cycle collector does not run."""
    log, zeros = [], torch.zeros
    monkeypatch.setattr(torch, "zeros", lambda *a, pin_memory=False, **kw: zeros(*a, **kw))
    monkeypatch.setattr(torch.cuda, "Event", lambda: NS(record=lambda: None))
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: log.append("wait"))

    class Recorded:
        def __init__(self, n):
            self.n = n

        def reset(self):
            log.append(self.n)

    def make(n):
        runner = ModelRunner.__new__(ModelRunner)
        runner.device = torch.device("cpu")
        runner.manager = NS(groups={}, blocks_for=lambda positions: 1, step_words=lambda *a: 8)
        runner._graphs = {}
        for i in range(n):
            runner._graphs[i] = DecodeGraph(runner, 1, 64)
            runner._graphs[i].graph = Recorded(i)
        return runner

    collecting = gc.isenabled()
    gc.disable()
    yield make, log
    if collecting:
        gc.enable()


def test_a_dropped_runner_lets_go_of_its_recorded_steps(made):
    make, log = made
    runner = make(2)
    assert log == []
    del runner
    assert log == ["wait", 0, "wait", 1]


def test_recorded_steps_that_are_dropped_one_by_one_or_together(made):
    make, log = made
    runner = make(3)
    runner._graphs.pop(1)                    # as for the oldest of too many
    assert log == ["wait", 1]
    runner._graphs.clear()                   # as when recording fails
    assert log == ["wait", 1, "wait", 0, "wait", 2]


def test_a_step_that_was_never_recorded_waits_for_nothing(made):
    make, log = made
    runner = make(0)
    DecodeGraph(runner, 1, 64)
    assert log == []


def test_events_of_a_step_live_until_its_recording_has_ended(made, monkeypatch):
    """What a part leaves in the context's events, the events of launches on another stream, is there when the recording ends, and gone once the step is recorded."""
    import contextlib
    import weakref
    make, log = made

    class Event:
        pass

    class Graph:
        def capture_begin(self):
            log.append("begin")

        def capture_end(self):
            log.append(("end", seen[-1]() is not None))

        def reset(self):
            pass

    seen = []

    def forward(ctx, caches):
        event = Event()
        ctx.events.append(event)
        seen.append(weakref.ref(event))
        return torch.zeros(1, 4)

    stream = NS(wait_stream=lambda s: None)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", Graph)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "Event", lambda: NS(record=lambda: None, synchronize=lambda: None))
    runner = make(0)
    runner.manager.pack_decode = lambda *a, **kw: None
    runner.storage = NS(pad_pages=[], pad_slot=0, caches=None)
    runner.model, runner.vocab_size, runner.before_launch, runner.capture_stream = NS(forward=forward), 4, None, stream
    runner.act_dtype, runner.block_size = torch.float32, 64
    step = DecodeGraph(runner, 1, 64)
    step.run(runner, [NS(want=[0], tokens=[1], req="a")])
    assert log == ["wait", "begin", ("end", True)] and step.graph is not None
    assert seen[-1]() is None and seen[0]() is None
