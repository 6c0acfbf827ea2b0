"""Captures run with Python's cyclic collector paused (smlm_hip.capture)."""
import contextlib
import gc
import os
import re
import threading

import pytest
import torch

from conftest import PKG_ROOT, REPO
from smlm_hip import capture


@pytest.fixture(params=[True, False], ids=["collector-on", "collector-off"])
def collector(request):
    was = gc.isenabled()
    (gc.enable if request.param else gc.disable)()
    yield request.param
    (gc.enable if was else gc.disable)()


def test_the_collector_is_off_inside_and_as_before_after(collector, monkeypatch):
    seen = []

    @contextlib.contextmanager
    def graph_capture(graph):
        seen.append((graph, gc.isenabled()))
        yield
        seen.append(gc.isenabled())

    monkeypatch.setattr(torch.cuda, "graph", graph_capture)
    with capture.capture("graph"):
        seen.append(gc.isenabled())
    assert seen == [("graph", False), False, False] and gc.isenabled() == collector


def test_the_collector_returns_after_an_exception(collector):
    with pytest.raises(KeyError):
        with capture.collector_paused():
            raise KeyError
    assert gc.isenabled() == collector


def test_overlapping_pauses_of_two_threads(collector):
    """The first to begin ends first: the collector stays off for the other one."""
    inside, leave, seen = threading.Event(), threading.Event(), []

    def other():
        with capture.collector_paused():
            inside.set()
            leave.wait(30)
            seen.append(gc.isenabled())

    with capture.collector_paused():
        thread = threading.Thread(target=other)
        thread.start()
        assert inside.wait(30)
    seen.append(gc.isenabled())
    leave.set()
    thread.join(30)
    assert seen == [False, False] and gc.isenabled() == collector


def test_every_capture_goes_through_the_helper():
    package = os.path.join(PKG_ROOT, "smlm_hip")
    files = [os.path.join(REPO, "bench.py")] + [os.path.join(package, f) for f in sorted(os.listdir(package))
                                                if f.endswith(".py") and f != "capture.py"]
    direct = [f for f in files if re.search(r"torch\.cuda\.graph\(|capture_begin\(", open(f).read())]
    assert direct == []
