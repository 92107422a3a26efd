"""What ExpertSlotCache issues, and on which stream, without a GPU: the library, the streams
and the events are stand-ins that record the calls."""
from __future__ import annotations

from contextlib import nullcontext
from types import SimpleNamespace

import pytest
import torch

from vllm_expert_cache import cache as cache_mod
from vllm_expert_cache.cache import ExpertSlotCache

CURRENT, SIDE = 11, 22


@pytest.fixture
def calls(monkeypatch):
    """[(entry point or event, stream)] in order; `calls.capturing` is the capture state."""
    class Calls(list):
        capturing = False

    log = Calls()

    def stream(handle):
        def wait_event(ev):
            log.append(("wait", handle))
        return SimpleNamespace(cuda_stream=handle, wait_event=wait_event)

    class Event:
        def record(self, s):
            log.append(("record", s.cuda_stream))

    class Lib:
        def __getattr__(self, name):
            def call(*args):
                s = args[-1]
                log.append((name.replace("expert_cache_", ""), getattr(s, "value", s)))
                return 0
            return call

    monkeypatch.setattr(cache_mod, "lib", Lib)
    monkeypatch.setattr(cache_mod, "device_address", lambda t: t.data_ptr())
    monkeypatch.setattr(cache_mod, "_side_stream", lambda dev: stream(SIDE))
    monkeypatch.setattr(torch.cuda, "current_stream", lambda dev=None: stream(CURRENT))
    monkeypatch.setattr(torch.cuda, "Event", Event)
    monkeypatch.setattr(torch.cuda, "device", lambda dev: nullcontext())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: log.capturing)
    return log


def _caches(n=2, tensors=1):
    owner = SimpleNamespace(**{f"w{i}": torch.zeros(8, 16) for i in range(tensors)})
    return [ExpertSlotCache(owner, list(vars(owner)), 8, 4, "cpu") for _ in range(n)]


IDS = torch.tensor([1, 2], dtype=torch.int32)


def test_refresh_is_one_call(calls):
    cache, = _caches(1)
    cache.refresh(IDS)
    assert calls == [("refresh", CURRENT)]


def test_refresh_gathers_the_tensors_past_six(calls):
    cache, = _caches(1, tensors=7)
    cache.refresh(IDS)
    assert calls == [("refresh", CURRENT), ("gather", CURRENT)]


def test_prefetch_forks_its_copy(calls):
    cache, = _caches(1)
    cache.prefetch(IDS)
    cache.refresh(IDS)
    cache.refresh(IDS)
    assert calls == [("prefetch", CURRENT), ("record", CURRENT), ("wait", SIDE),
                     ("gather_live", SIDE), ("record", SIDE), ("manage_remap", CURRENT),
                     ("wait", CURRENT), ("gather", CURRENT), ("refresh", CURRENT)]


@pytest.mark.parametrize("along", [False, True])
def test_captured_prefetch_does_not_fork(calls, along):
    """Several steps of two layers in one capture: no event, nothing on the side stream."""
    a, b = _caches()
    calls.capturing = True
    for _ in range(3):
        b.prefetch(IDS, along=a if along else None)
        a.refresh(IDS)
        b.refresh(IDS)
    b.join()
    first = [("manage_remap_prefetch", CURRENT), ("gather", CURRENT), ("gather", CURRENT)] \
        if along else [("prefetch", CURRENT), ("gather", CURRENT), ("refresh", CURRENT)]
    assert calls == 3 * (first + [("refresh", CURRENT)])
