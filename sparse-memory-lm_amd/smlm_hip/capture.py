"""HIP graph capture, the way every captured graph of this package is made."""
import contextlib
import gc
import threading

import torch

_lock = threading.Lock()
_captures = 0          # captures that hold the collector off, over all threads
_resume = False        # whether it ran before the first of them


@contextlib.contextmanager
def collector_paused():
    """Python's cyclic collector held off: it may destroy a captured graph that some cycle kept, which is not permitted
    while a stream is capturing and ends the process.  What it was, on or off, it is again after the last of overlapping
    pauses, also when one ends with an exception."""
    global _captures, _resume
    with _lock:
        if _captures == 0:
            _resume = gc.isenabled()
            gc.disable()
        _captures += 1
    try:
        yield
    finally:
        with _lock:
            _captures -= 1
            if _captures == 0 and _resume:
                gc.enable()


@contextlib.contextmanager
def capture(graph):
    """torch.cuda.graph(graph) with the cyclic collector paused."""
    with collector_paused(), torch.cuda.graph(graph):
        yield
