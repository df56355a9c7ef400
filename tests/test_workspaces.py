"""The launcher's workspaces per (device, stream): which ones are kept."""

from __future__ import annotations

import collections
from types import SimpleNamespace

import torch

import flydsl_amd.pa_decode as pd


class FakeWorkspace:
    def __init__(self, dev, stream, nbytes, pairs):
        self.slots, self.counters = torch.empty(nbytes, dtype=torch.uint8), torch.zeros(pairs, dtype=torch.int32)

    def pointers(self):
        return (self.slots.data_ptr(), self.slots.numel(), self.counters.data_ptr(), self.counters.numel())


def test_the_least_recently_used_workspace_goes(monkeypatch):
    monkeypatch.setattr(pd, "_workspaces", collections.OrderedDict())
    monkeypatch.setattr(pd, "_SplitWorkspace", FakeWorkspace)
    monkeypatch.setattr(pd, "_workspace_used", None)
    current = SimpleNamespace(stream_id=0)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda index: current)

    def use(stream_id, nbytes=64):
        current.stream_id = stream_id
        return pd._native_workspace(0, stream_id, 4, nbytes)[-1]

    busy = use(1)
    others = [3 + 2 * i for i in range(pd._WORKSPACES_KEPT + 5)]  # torch's own stream ids are odd
    for i in others:
        use(i)
        assert use(1) is busy, i  # used throughout: kept
    assert len(pd._workspaces) == pd._WORKSPACES_KEPT
    assert {k[1] for k in pd._workspaces} == {1, *others[-(pd._WORKSPACES_KEPT - 1):]}
    grown = use(1, 4096)
    assert grown is not busy and grown.slots.numel() >= 4096 and use(1) is grown
    # a workspace dropped between its lookup and its refresh still serves the call
    class Racing(collections.OrderedDict):
        def move_to_end(self, key):
            self.pop(key, None)
            super().move_to_end(key)

    racing = Racing(pd._workspaces)
    monkeypatch.setattr(pd, "_workspaces", racing)
    last = racing[0, others[-1]]
    assert use(others[-1]) is last and (0, others[-1]) not in racing
