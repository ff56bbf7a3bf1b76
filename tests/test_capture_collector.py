"""The cyclic garbage collector and a capture: it does not run while any thread captures, and is as it was afterwards.  On the CPU, with
stand-ins for what captures."""
import collections
import contextlib
import gc
import threading
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from bare_cuda_4gib_amd.engine import executor


def test_off_while_any_thread_is_inside_and_restored():
    was = gc.isenabled()
    try:
        for on in (True, False):
            (gc.enable if on else gc.disable)()
            inside, leave = threading.Event(), threading.Event()

            def other():
                with executor.collector_off():
                    inside.set()
                    leave.wait(10)

            thread = threading.Thread(target=other)
            with pytest.raises(ValueError):
                with executor.collector_off(), executor.collector_off():
                    thread.start()
                    assert inside.wait(10) and not gc.isenabled()
                    raise ValueError
            assert not gc.isenabled()                     # (the other thread is still inside)
            leave.set()
            thread.join()
            assert gc.isenabled() == on
    finally:
        (gc.enable if was else gc.disable)()


def test_a_step_is_captured_without_the_collector(monkeypatch):
    """A cycle that is garbage when a step is captured is not collected inside the capture, however eager the collector is."""
    events, capturing = [], []

    class Old:
        def __init__(self):
            self.me = self

        def __del__(self):
            events.append("destroyed inside" if capturing else "destroyed outside")

    @contextlib.contextmanager
    def graph(*a, **k):
        capturing.append(1)
        yield
        capturing.pop()

    def forward(ctx):
        if capturing:
            Old()
            [[] for _ in range(2000)]                     # (containers enough for a collection)
        return torch.zeros(1)

    monkeypatch.setattr(torch.cuda, "graph", graph)
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: None)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda *a: None)
    monkeypatch.setattr(torch.cuda, "Event", lambda: SimpleNamespace(record=lambda: None))
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    cache = SimpleNamespace(save_slots=lambda s: None, restore_slots=lambda s: None)
    fake = SimpleNamespace(_graphs=collections.OrderedDict(), MAX_GRAPHS=2, rt=SimpleNamespace(device="cpu"), _capture_parts=[], captures=0, cache=cache,
                           model=SimpleNamespace(forward=forward), _context_from=lambda *a: SimpleNamespace(made={}))
    was, threshold = gc.isenabled(), gc.get_threshold()
    gc.enable()
    gc.set_threshold(5, 2, 2)
    try:
        executor.Executor._capture(fake, (1, 256), np.zeros(4, dtype=np.int32), [("token_ids", 4)], [], dict(seq_slots=[0], T=1), 256)
    finally:
        gc.set_threshold(*threshold)
        (gc.enable if was else gc.disable)()
    gc.collect()
    assert fake.captures == 1 and events == ["destroyed outside"]
