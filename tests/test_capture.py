"""What a capture must not meet (no GPU: the graph and the streams are stand-ins)."""
import contextlib
import gc
import threading
from types import SimpleNamespace

import pytest
import torch

from dinfer_amd.engine import runner as runner_module
from dinfer_amd.engine.runner import ModelRunner


class Graph:
    def capture_begin(self, **kw):
        pass

    def capture_end(self):
        pass

    def pool(self):
        return 1


@pytest.fixture
def capture(monkeypatch):
    stream = SimpleNamespace(wait_stream=lambda s: None)
    for name, value in (("synchronize", lambda: None), ("CUDAGraph", Graph), ("Stream", lambda device: stream), ("current_stream", lambda: stream),
                        ("stream", lambda s: contextlib.nullcontext())):
        monkeypatch.setattr(torch.cuda, name, value)
    r = SimpleNamespace(batch=SimpleNamespace(lengths_known=False), device="cuda", _capture_stream=None, _graph_pool=None)
    return lambda forward: ModelRunner._capture(r, forward)


class Holder:
    """What owns a graph, in a cycle of references."""

    def __init__(self, freed):
        self.itself, self.freed = self, freed

    def __del__(self):
        self.freed.append(1)


def test_no_garbage_is_collected_inside_a_capture(capture):
    freed, inside = [], []

    def forward():
        Holder(freed)
        for _ in range(3000):       # far more new containers than any threshold
            [[] for _ in range(3)]
        inside.append((len(freed), gc.isenabled()))

    old = gc.get_threshold()
    gc.collect()
    gc.set_threshold(1, 1, 1)
    try:
        capture(forward)
        assert inside == [(0, False)] and gc.isenabled()
        with pytest.raises(ZeroDivisionError):
            capture(lambda: 1 / 0)
        assert gc.isenabled()
    finally:
        gc.set_threshold(*old)
    gc.collect()
    assert freed == [1]


def test_captures_of_two_threads_and_a_process_that_collects_by_itself():
    first_in, second_out = threading.Event(), threading.Event()
    states = []

    def first():
        with runner_module._uncollected:
            first_in.set()
            second_out.wait(10)
            states.append(gc.isenabled())

    t = threading.Thread(target=first)
    t.start()
    assert first_in.wait(10)
    with runner_module._uncollected:
        states.append(gc.isenabled())
    states.append(gc.isenabled())     # the other thread is still inside
    second_out.set()
    t.join()
    assert states == [False, False, False] and gc.isenabled()
    gc.disable()
    try:
        with runner_module._uncollected:
            pass
        assert not gc.isenabled()
    finally:
        gc.enable()
