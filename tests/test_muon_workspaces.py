"""Muon workspaces under several streams and threads: what a call waits for before it reuses one,
with a library and streams that only record (the results on the GPU: tests/test_gpu_muon.py)."""
import contextlib
import copy
import threading
import time

import pytest
import torch

from morph_amd import muon


class Stream:
    def __init__(self, name, log):
        self.name, self.log, self.capturing = name, log, False

    def wait_stream(self, other):
        self.log.append((self.name, other.name))


@pytest.fixture
def streams(monkeypatch):
    log, current = [], []

    @contextlib.contextmanager
    def use(stream):
        current.append(stream)
        yield
        current.pop()

    monkeypatch.setattr(torch.cuda, "stream", use)
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: current[-1])
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: current[-1].capturing)
    return Stream("a", log), Stream("b", log), log


def test_another_stream_waits_for_the_last_one(streams):
    a, b, log = streams
    ws = muon.Workspaces()
    first = ws.get(64, 64, 1, "cpu", 0, a)
    assert ws.get(64, 64, 1, "cpu", 0, a) is first and log == []
    assert ws.get(64, 64, 1, "cpu", 0, b) is first and log == [("b", "a")]
    assert ws.get(64, 64, 1, "cpu", 0, b) is first and log == [("b", "a")]
    with torch.cuda.stream(a):  # the current one, by default
        assert ws.get(64, 64, 1, "cpu") is first and log == [("b", "a"), ("a", "b")]
    assert ws.get(64, 64, 1, "cpu", 1, b) is not first and len(log) == 2  # another workspace


def test_a_capture_waits_for_nothing(streams):
    """A stream under capture may not wait for one that is not, nor the other way round."""
    a, b, log = streams
    ws = muon.Workspaces()
    ws.get(64, 64, 1, "cpu", 0, a)
    b.capturing = True
    ws.get(64, 64, 1, "cpu", 0, b)
    b.capturing = False
    ws.get(64, 64, 1, "cpu", 0, a)
    a.capturing = True
    ws.get(64, 64, 1, "cpu", 0, b)
    assert log == []


class Library:
    """Records each entry's name, slowly, as launches of a full queue return."""

    def __init__(self):
        self.calls = []

    def __getattr__(self, name):
        def call(*args):
            if name == "morph_muon_workspace_bytes":
                return 256
            self.calls.append((threading.get_ident(), name))
            time.sleep(2e-3)
            return 0
        return call


@pytest.mark.parametrize("call", ["orthogonalize", "muon_step"])
def test_threads_do_not_mix_their_launches(streams, monkeypatch, call):
    """Two threads on one stream with the shared workspaces: each call's launches are together."""
    lib = Library()
    monkeypatch.setattr(muon, "lib", lambda: lib)
    monkeypatch.setattr(muon, "stream_handle", lambda s=None: None)
    monkeypatch.setattr(muon, "_check_matrix", lambda t, name: None)
    monkeypatch.setattr(muon, "_check_items", lambda *a: list(zip(*a[:3], [None] * len(a[0]))))
    ts = [torch.zeros(n, 40) for n in (8, 16, 24)]
    ws = muon.Workspaces()

    def run():
        for _ in range(4):
            if call == "orthogonalize":
                muon.orthogonalize(ts, stream=streams[0], workspaces=ws)
            else:
                muon.muon_step(ts, ts, ts, .02, .01, stream=streams[0], workspaces=ws)

    threads = [threading.Thread(target=run) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    per_call = 3 if call == "orthogonalize" else 6  # a launch per shape, or prepare and chain
    owners = [who for who, _ in lib.calls]
    assert len(owners) == 8 * per_call
    for k in range(0, len(owners), per_call):
        assert len(set(owners[k:k + per_call])) == 1, k


def test_workspaces_can_be_copied(streams):
    ws = muon.Workspaces()
    ws.get(64, 64, 1, "cpu", 0, streams[0])
    assert copy.deepcopy(ws)._ws == {}
