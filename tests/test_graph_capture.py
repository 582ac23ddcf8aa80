"""A dropped model and its runners are a cycle that owns graphs, and destroying
a graph while a stream captures aborts the process: the graph of a runner that
dies during a capture is destroyed after it, and the collector is left alone."""
from __future__ import annotations

import contextlib
import gc
import threading
import weakref

import numpy as np
import pytest
import torch


@pytest.fixture
def env(monkeypatch):
    """(graph_capture, make, gone, busy): ``make(name)`` drops a runner inside a
    cycle; ``busy[0]`` says that this thread's stream captures."""
    from rwkv7mi import model

    busy, gone = [False], []
    monkeypatch.setattr(torch.cuda, "graph", lambda graph: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: busy[0])

    def make(name, cls=model.NativeGraphRunner):
        r = cls.__new__(cls)
        # (an array: like a graph, it goes with its last reference, not with the cycle's collection)
        r.graph, r.model = np.zeros(1), [r]
        weakref.finalize(r.graph, gone.append, name)

    yield model.graph_capture, make, gone, busy
    busy[0] = False
    gc.enable()
    gc.collect()
    model._drop_graphs()
    assert not model._dead_graphs


def test_graphs_that_die_in_a_capture_outlive_it(env):
    from rwkv7mi.model import NativePrefillGraphRunner

    capture, make, gone, _ = env
    with capture(None):
        make("decode")
        make("prefill", NativePrefillGraphRunner)
        gc.collect()
        assert gone == []
    assert sorted(gone) == ["decode", "prefill"]
    make("later")
    gc.collect()
    assert gone[2:] == ["later"]


def test_graphs_that_die_in_a_plain_capture_wait_for_the_next_chance(env):
    capture, make, gone, busy = env
    busy[0] = True
    make("a")
    gc.collect()
    assert gone == []
    busy[0] = False
    make("b")
    gc.collect()
    assert sorted(gone) == ["a", "b"]
    busy[0] = True
    make("c")
    gc.collect()
    busy[0] = False
    with capture(None):
        assert "c" not in gone
    assert "c" in gone


@pytest.mark.parametrize("was_on", [True, False])
def test_a_capture_leaves_the_collector_alone(env, was_on):
    capture = env[0]
    (gc.enable if was_on else gc.disable)()
    with pytest.raises(RuntimeError, match="body"):
        with capture(None):
            assert gc.isenabled() is was_on
            gc.disable()  # a caller's own choice, kept
            raise RuntimeError("body")
    assert not gc.isenabled()


def test_overlapping_captures_of_two_threads(env):
    capture, make, gone, _ = env
    inside, leave = threading.Event(), threading.Event()

    def other():
        with capture(None):
            inside.set()
            leave.wait(10)

    t = threading.Thread(target=other)
    with capture(None):
        t.start()
        assert inside.wait(10)
        make("x")
        gc.collect()
    assert gone == []  # the other one is still capturing
    leave.set()
    t.join()
    assert gone == ["x"]


@pytest.mark.gpu
def test_a_model_collected_during_a_capture():
    """The graphs of a dropped model that the collector finds inside another
    capture are kept until it has ended, and that capture is intact."""
    from rwkv7mi import model as M

    cfg = M.NativeRWKV7Config(vocab_size=512, hidden_size=256, num_hidden_layers=2, intermediate_size=1024,
                              decay_low_rank_dim=16, a_low_rank_dim=16, gate_low_rank_dim=32, v_low_rank_dim=16)
    m = M.NativeRWKV7ForCausalLM.from_random(cfg, seed=0, device="cuda", dtype=torch.float16)
    m.graph_runner(2)
    m.prefill_graph_runner(1, 16)
    x, y = torch.ones(64, device="cuda"), torch.zeros(64, device="cuda")
    torch.cuda.synchronize()
    gc.collect()
    M._drop_graphs()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        torch.add(x, x, out=y)
        del m
        gc.collect()
        assert len(M._dead_graphs) == 2
    for i in range(3):
        x.fill_(i)
        g.replay()
        torch.cuda.synchronize()
        assert bool((y == 2 * i).all())
    M._drop_graphs()
    assert not M._dead_graphs
