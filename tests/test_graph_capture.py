"""A graph capture runs with the cyclic collector off: a dropped model is a
cycle that owns graphs, and destroying a graph during a capture aborts."""
from __future__ import annotations

import contextlib
import gc
import threading
import weakref

import pytest
import torch


class _Node:
    pass


def _dead_cycle():
    a, b = _Node(), _Node()
    a.other, b.other = b, a
    return weakref.ref(a)


@pytest.fixture
def capture(monkeypatch):
    from rwkv7mi import model

    monkeypatch.setattr(torch.cuda, "graph", lambda graph: contextlib.nullcontext())
    old = gc.get_threshold()
    yield model.graph_capture
    gc.set_threshold(*old)
    gc.enable()


def test_no_collection_during_a_capture(capture):
    with capture(None):
        gc.set_threshold(1, 1, 1)  # collect at every allocation
        dead = _dead_cycle()
        keep = [[i] for i in range(2000)]
        assert dead() is not None and not gc.isenabled()
    assert gc.isenabled()
    gc.collect()
    assert dead() is None and len(keep) == 2000


@pytest.mark.parametrize("was_on", [True, False])
def test_collector_state_is_restored(capture, was_on):
    (gc.enable if was_on else gc.disable)()
    with pytest.raises(RuntimeError, match="body"):
        with capture(None):
            raise RuntimeError("body")
    assert gc.isenabled() is was_on


def test_overlapping_captures_of_two_threads(capture):
    inside, leave = threading.Event(), threading.Event()

    def other():
        with capture(None):
            inside.set()
            leave.wait(10)

    t = threading.Thread(target=other)
    with capture(None):
        t.start()
        assert inside.wait(10)
    assert not gc.isenabled()  # the other one is still capturing
    leave.set()
    t.join()
    assert gc.isenabled()
