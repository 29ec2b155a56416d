"""The renderers' cell map cache, its streams and events replaced by host objects."""
import contextlib
import threading
from collections import OrderedDict

import pytest
import torch

from svox2_amd import _C


class FakeStream:
    def __init__(self, name):
        self.name, self.waited = name, []

    def wait_event(self, event):
        self.waited.append(event)


class FakeMap:
    def __init__(self, stream):
        self.built_on, self.used_by = stream, []

    def record_stream(self, stream):
        self.used_by.append(stream)


class FakeEvent:
    recorded = None

    def record(self, stream):
        self.recorded = stream


@pytest.fixture
def cache(monkeypatch):
    """The cache with `state.stream` as the current stream, `state.capturing`, and
    the maps built so far."""
    class State:
        stream, capturing = FakeStream("a"), False
    state = State()
    state.built = []

    def build(links, rows):
        state.built.append(FakeMap(state.stream))
        return state.built[-1]

    monkeypatch.setattr(_C, "_CELL_MAPS", OrderedDict())
    monkeypatch.setattr(_C, "_ACCEL_EPOCH", {})
    monkeypatch.setattr(_C, "build_cell_map", build)
    monkeypatch.setattr(_C, "_on_device", lambda t: contextlib.nullcontext())
    monkeypatch.setattr(torch.cuda, "current_device", lambda: None)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: state.capturing)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: state.stream)
    monkeypatch.setattr(torch.cuda, "Event", FakeEvent)
    return state


def _links(k=0):
    return torch.full((4, 4, 4), k, dtype=torch.int32)


def test_capture_leaves_the_cache_alone(cache):
    """While capturing, no map is built, kept or taken."""
    links = _links()
    cache.capturing = True
    assert _C._cached_cell_map(links, 3) is None
    assert not cache.built and not _C._CELL_MAPS
    cache.capturing = False
    cmap = _C._cached_cell_map(links, 3)
    assert _C._cached_cell_map(links, 3) is cmap and len(cache.built) == 1
    cache.capturing = True
    assert _C._cached_cell_map(links, 3) is None and len(_C._CELL_MAPS) == 1


def test_two_threads(cache, monkeypatch):
    """A thread that fills the cache while another looks a map up does not take
    the found entry away under it."""
    links = [_links(k) for k in range(6)]
    fill = threading.Thread(target=lambda: [_C._cached_cell_map(x, 3) for x in links[1:]])

    class Interrupted(OrderedDict):
        def get(self, *args):
            found = super().get(*args)
            if found is not None and fill.ident is None:
                fill.start()
                fill.join(0.3)  # waits for as long as the other thread is kept out
            return found

    monkeypatch.setattr(_C, "_CELL_MAPS", Interrupted())
    cmap = _C._cached_cell_map(links[0], 3)
    assert _C._cached_cell_map(links[0], 3) is cmap
    fill.join()
    assert len(cache.built) == 6 and len(_C._CELL_MAPS) == _C._CELL_MAP_CACHE


def test_streams_share_a_map(cache):
    """A map is built once; every other stream waits for its build and keeps its
    memory until that stream's work is done."""
    links = _links()
    a, b = FakeStream("a"), FakeStream("b")
    cache.stream = a
    cmap = _C._cached_cell_map(links, 3)
    assert _C._cached_cell_map(links, 3) is cmap and not a.waited and not cmap.used_by
    cache.stream = b
    assert _C._cached_cell_map(links, 3) is cmap and len(cache.built) == 1
    assert [e.recorded for e in b.waited] == [a] and cmap.used_by == [b]
