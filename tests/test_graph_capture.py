"""Captures of the package count the capturing thread's calls alone: a process group's own thread may ask events in the middle of one."""
import contextlib
import os
import re
import threading
from types import SimpleNamespace

import pytest
import torch

from nano_vllm_amd import ops
from nano_vllm_amd.engine.runner import ModelRunner

PACKAGE = os.path.dirname(ops.__file__)


def test_every_capture_of_the_engine_is_of_its_own_thread(monkeypatch):
    modes = []

    @contextlib.contextmanager
    def graph(graph, pool=None, stream=None, capture_error_mode="global"):
        modes.append(capture_error_mode)
        yield
    monkeypatch.setattr(torch.cuda, "graph", graph)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: SimpleNamespace(pool=lambda: 7))
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    r = ModelRunner.__new__(ModelRunner)
    r.max_bs, r.share_prefix, r.world_size, r.graphs, r.sgraphs, r.graphs_px, r._sgraph_pool = 2, True, 1, {}, {}, {}, None
    r.sstage = SimpleNamespace(upload=lambda: None)
    r.prepare_portions = r._decode_body = r._forward_decode = lambda *a, **k: None
    r.capture_graphs()                              # two buckets, the larger one with a shared prefix too
    r._capture_decode(1)
    assert modes == ["thread_local"] * 4


def test_no_capture_goes_another_way():
    for folder, _, files in os.walk(PACKAGE):
        for name in files:
            if name.endswith(".py"):
                with open(os.path.join(folder, name)) as fh:
                    found = re.findall(r"torch\.cuda\.graph\(.*", fh.read())
                assert len(found) == (2 if os.path.join(folder, name) == ops.__file__ else 0), (name, found)        # (its one call, and its docstring)


@pytest.mark.gpu
def test_a_capture_beside_a_thread_that_asks_events():
    x, stop, failed = torch.ones(1 << 20, device="cuda"), threading.Event(), []

    def ask():
        try:
            s, event = torch.cuda.Stream(), torch.cuda.Event()
            while not stop.is_set():
                event.record(s)
                event.query()
        except Exception as e:  # noqa: BLE001
            failed.append(e)
    other = threading.Thread(target=ask)
    other.start()
    try:
        for i in range(20):
            graph = torch.cuda.CUDAGraph()
            with ops.capture(graph):
                y = x
                for _ in range(50):
                    y = y + 1
            graph.replay()
            torch.cuda.synchronize()
            assert bool((y == 51).all())
    finally:
        stop.set()
        other.join()
    assert not failed
