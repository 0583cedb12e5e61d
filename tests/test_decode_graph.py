"""The host's side of a captured decode step (engine/decode_graph.py) without a GPU: what it does before it writes the pinned layout
that the kernels of the step read."""
import contextlib
from types import SimpleNamespace

import pytest
import torch

from rbitnet_amd.cache import Cache
from rbitnet_amd.engine import decode_graph
from rbitnet_amd.parts.base import CacheRequest


class Weak(SimpleNamespace):
    """(an engine is held by a weak reference)"""


@pytest.mark.parametrize("interrupted", ["first", "replayed"])
def test_a_step_after_an_interrupted_one_waits_before_it_writes_the_layout(monkeypatch, interrupted):
    events, failing = [], set()

    def wait(kind):
        events.append(kind)
        if kind in failing:
            raise KeyboardInterrupt

    stream = SimpleNamespace(wait_stream=lambda other: None)
    graph = SimpleNamespace(replay=lambda: events.append("replay"))
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda t: t)
    monkeypatch.setattr(torch.cuda, "Stream", lambda device=None: stream)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda: stream)
    monkeypatch.setattr(torch.cuda, "stream", lambda s: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "graph", lambda g: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "CUDAGraph", lambda: graph)
    monkeypatch.setattr(torch.cuda, "synchronize", lambda: wait("synchronize"))
    lib = SimpleNamespace(n_compute_units=256, fetch_words=lambda *a: None, sample=lambda *a: None, wait=lambda: wait("wait"))
    model = SimpleNamespace(forward=lambda ctx, cache, rows: events.append("launch") or torch.zeros(1, 7))
    cache = Cache([CacheRequest("kv", heads=1, head_dim=8)], 1, 128, torch.float32, "cpu")
    engine = Weak(device=torch.device("cpu"), lib=lib, model=model, cache=cache, max_seq_len=128)
    step = decode_graph.DecodeGraph(engine, 1, 1)
    for name in ("fill", "refill_single"):
        real = getattr(step.ctx, name)
        monkeypatch.setattr(step.ctx, name, lambda *a, real=real, **kw: (events.append("write"), real(*a, **kw))[1])
    slot = cache.alloc_slot()
    run = lambda: step.run([slot], [cache.length(slot)], [3])
    if interrupted == "replayed":
        run()
    del events[:]
    failing = {"synchronize" if interrupted == "first" else "wait"}
    before = cache.length(slot)
    with pytest.raises(KeyboardInterrupt):
        run()
    assert events[0] == "write" and cache.length(slot) == before
    failing, done = set(), len(events)
    run()
    assert events[done:done + 2] == ["synchronize", "write"] and cache.length(slot) == before + 1
    done = len(events)
    run()                                                     # and steps that nothing interrupted wait for nobody
    assert events[done] == "write"
