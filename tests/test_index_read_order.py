"""The order that reads and writes of an index put their streams in, nested ones among them: on the CPU, with streams that only
count what each has done and knows of the others."""
from types import SimpleNamespace

import pytest
import torch

from docagents_amd.index.flat import FlatIndex


class Stream:
    def __init__(self, handle):
        self.cuda_stream, self.seen = handle, {}

    def work(self):
        self.seen[self.cuda_stream] = self.seen.get(self.cuda_stream, 0) + 1

    def learn(self, seen):
        for s, n in seen.items():
            self.seen[s] = max(n, self.seen.get(s, 0))

    def wait_event(self, ev):
        self.learn(ev.seen)

    def wait_stream(self, other):
        self.learn(other.seen)

    def after(self, other):
        return self.seen.get(other.cuda_stream, 0) >= other.seen.get(other.cuda_stream, 0)


class Event:
    def __init__(self):
        self.seen = {}

    def record(self, stream):
        self.seen = dict(stream.seen)


@pytest.fixture
def index(monkeypatch):
    idx = FlatIndex(8, "cpu", capacity=64)
    idx.device = SimpleNamespace(type="cuda")
    now = [None]
    monkeypatch.setattr(torch.cuda, "current_stream", lambda device=None: now[0])
    monkeypatch.setattr(torch.cuda, "Event", Event)

    def on(stream, what):
        class At:
            def __enter__(self):
                self.before, now[0] = now[0], stream
                self.inner = what()
                self.inner.__enter__()

            def __exit__(self, *e):
                self.inner.__exit__(*e)
                now[0] = self.before
        return At()
    return SimpleNamespace(read=lambda s: on(s, idx.reading), write=lambda s: on(s, idx.writing))


def streams():
    return Stream(0), Stream(7), Stream(9)  # (the default stream's handle is 0)


def test_write_after_nested_reads(index):
    a, b, w = streams()
    with index.read(a):
        a.work()
        with index.read(a):
            a.work()
        with index.read(b):
            b.work()
            with index.read(a):
                a.work()
        a.work()
    with index.write(w):
        assert w.after(a) and w.after(b)


def test_write_after_each_of_two_reads(index):
    a, _, w = streams()
    for _ in range(2):  # (the second read's event is the first one's, recorded again)
        with index.read(a):
            a.work()
    with index.write(w):
        assert w.after(a)
        w.work()
    with index.read(a):
        assert a.after(w)
        a.work()
    with index.write(w):
        assert w.after(a)


def test_write_on_another_stream_inside_a_read(index):
    a, b, w = streams()
    with index.read(a):
        a.work()
        with index.read(b):
            b.work()
            with index.write(w):
                assert w.after(a) and w.after(b)


@pytest.mark.parametrize("same", [False, True])
def test_nested_read_after_a_write_on_another_stream(index, same):
    a, b, w = streams()
    with index.read(a):
        with index.write(w):
            w.work()
        with index.read(a if same else b):
            assert (a if same else b).after(w)
            (a if same else b).work()
        a.work()
    with index.write(w):
        assert w.after(a) and w.after(b)


def test_read_on_the_outer_stream_after_a_write_inside_another_read(index):
    a, b, w = streams()
    with index.read(a):
        with index.read(b):
            with index.write(w):
                w.work()
        with index.read(a):
            assert a.after(w)
