"""Host logic of the recorded-call inputs (``tybok_amd.graph.StaticCall``): no GPU, no recording."""
import contextlib
import gc
import weakref

import pytest
import torch

from tybok_amd.graph import CaptureSession, GraphRunner, StaticCall


def _call():
    return StaticCall(torch.zeros(1), noise=torch.full((1, 4, 8), 7.0), state=torch.zeros(1, 8), images=[torch.zeros(2), torch.zeros(2)])


def test_store_leading_keeps_the_zero_padding_of_a_padded_store():
    # a value narrower than its static tensor lands in the leading columns; what lies behind it reads as zeros,
    # whatever an earlier request (a wider value, noise drawn in place, a plain store) left there
    call = _call()
    a = torch.arange(12.0).view(1, 4, 3) + 1
    call.store_leading(noise=a)  # the first store clears what recording left behind the value
    want = torch.nn.functional.pad(a, (0, 5))
    assert torch.equal(call.inputs["noise"], want)
    wide = torch.ones(1, 4, 6) * 3
    call.store_leading(noise=wide)
    assert torch.equal(call.inputs["noise"], torch.nn.functional.pad(wide, (0, 2)))
    call.store_leading(noise=a)  # narrower than the last one: columns 3..5 must be cleared again
    assert torch.equal(call.inputs["noise"], want)
    call.inputs["noise"].fill_(9.0)  # (noise drawn in place)
    call.forget_leading("noise")
    call.store_leading(noise=a)
    assert torch.equal(call.inputs["noise"], want)
    call.store(noise=torch.full((1, 4, 8), 5.0))  # a plain store forgets the width as well
    call.store_leading(noise=a)
    assert torch.equal(call.inputs["noise"], want)
    full = torch.randn(1, 4, 8)
    call.store_leading(noise=full)
    assert torch.equal(call.inputs["noise"], full)


def test_store_leading_refuses_what_does_not_fit():
    call = _call()
    with pytest.raises(ValueError):
        call.store_leading(state=torch.zeros(1, 9))
    with pytest.raises(ValueError):
        call.store_leading(state=torch.zeros(2, 4))
    with pytest.raises(ValueError):
        call.store(images=[torch.zeros(2)])


def test_store_owned_copies_only_new_objects():
    call = _call()
    t = torch.ones(1, 8)
    call.store_owned(state=t)
    call.inputs["state"].zero_()
    call.store_owned(state=t)  # the very object stored last time: not copied again
    assert torch.count_nonzero(call.inputs["state"]) == 0
    call.forget_owned("state")
    call.store_owned(state=t)
    assert torch.equal(call.inputs["state"], t)


class _Stream:
    device_index = 0

    def __init__(self, log, name):
        self.log, self.name = log, name

    def wait_event(self, event):
        self.log.append((self.name, "waits for", event.at))


class _Event:
    at = None

    def record(self, stream):
        self.at = (stream.name, len(stream.log))
        stream.log.append((stream.name, "done", self.at))


def test_turns_wait_for_the_last_grid_and_for_nothing_behind_it(monkeypatch):
    from tybok_amd import graph

    log: list = []
    a, b = _Stream(log, "a"), _Stream(log, "b")
    current = [a]
    monkeypatch.setattr(graph, "_turn_done", {})
    monkeypatch.setattr(torch.cuda, "Event", _Event)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: current[0])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    graph.launch_alone(lambda: log.append(("a", "grid")), "cuda")
    log.append(("a", "unrelated work"))
    current[0] = b
    graph.launch_alone(lambda: log.append(("b", "grid")), "cuda")
    first = ("a", 2)
    assert log == [("a", "waits for", None), ("a", "grid"), ("a", "done", first), ("a", "unrelated work"),
                   ("b", "waits for", first), ("b", "grid"), ("b", "done", ("b", 6))]  # fmt: skip


def test_only_a_recording_that_holds_such_a_grid_takes_turns(monkeypatch):
    from tybok_amd import graph

    class Session:  # records nothing: runs the body as a capture would
        def prime_and_capture(self, fn):
            fn()
            return type("Graph", (), {"replay": lambda self: None})()

    turns: list = []

    @graph.contextmanager
    def turn(device=None):
        turns.append(device)
        yield

    monkeypatch.setattr(graph, "launch_turn", turn)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: None)
    plain = StaticCall(torch.zeros(1), x=torch.ones(1)).record(Session(), lambda x: x)
    plain.replay()
    assert turns == [] and not plain.takes_turn

    def body(x):
        graph.launch_alone(lambda: None, "cuda")
        return x

    loop = StaticCall(torch.zeros(1), x=torch.ones(1)).record(Session(), body)
    assert turns == [] and loop.takes_turn
    loop.replay()
    assert turns == [torch.device("cpu")]


class _Cycle:
    def __init__(self, on_death):
        self.me = self
        weakref.finalize(self, on_death)


def test_nothing_is_garbage_collected_while_a_graph_is_recorded(monkeypatch):
    # a dead graph in a reference cycle (an engine that was replaced) would be destroyed inside the recording
    recording, died_inside = [False], []

    @contextlib.contextmanager
    def graph(recorded):
        recording[0] = True
        yield
        recording[0] = False

    monkeypatch.setattr(torch.cuda, "CUDAGraph", object)
    monkeypatch.setattr(torch.cuda, "graph", graph)
    before = gc.get_threshold()
    gc.set_threshold(1, 1, 1)

    def body():
        for _ in range(50):
            _Cycle(lambda: died_inside.append(recording[0]))

    try:
        CaptureSession("cpu").capture(body)
        assert gc.isenabled()
    finally:
        gc.set_threshold(*before)
    gc.collect()
    assert len(died_inside) == 50 and not any(died_inside)


def test_a_dropped_engine_is_freed_at_once():
    class Engine:
        def __init__(self):
            self.runner = GraphRunner(self._record, "cpu")

        def _record(self, key, request):
            return (key, request)

    engine = Engine()
    assert engine.runner.entry("a", 1) == ("a", 1) and engine.runner.precapture(["b"]) and engine.runner.entry("b") == ("b", None)
    assert GraphRunner(lambda key, request: key, "cpu").entry("c") == "c"
    gone = weakref.ref(engine)
    gc.disable()
    try:
        del engine
        assert gone() is None
    finally:
        gc.enable()
