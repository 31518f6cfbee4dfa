"""What a write replaces stays out of the allocator's hands until the searches that may still read it have run."""
import numpy as np
import torch

from docagents_amd.index import flat, ivf


class Spy:
    """Stands for a device tensor: notes the streams that it is recorded on."""

    def __init__(self):
        self.streams = []

    def record_stream(self, st):
        self.streams.append(st)


def test_lists_of_a_retrained_index(monkeypatch):
    index = ivf.IVFFlatIndex(8, "cpu", lists=2)
    old = index.list_off_t = Spy()
    monkeypatch.setattr(index, "device", torch.device("cuda"))
    monkeypatch.setattr(ivf, "h2d", lambda a, dev: torch.from_numpy(a))
    monkeypatch.setattr(flat.torch.cuda, "current_stream", lambda dev=None: "writer")
    index._set_lists(np.array([0, 3, 5]))
    assert old.streams == ["writer"]
    assert index.list_off_t.tolist() == [0, 3, 5] and index.most_rows.tolist() == [0, 3, 5]


def test_centroids_of_a_retrained_index(monkeypatch):
    index = ivf.IVFFlatIndex(8, "cpu", lists=2)
    index.add("d", np.arange(6), torch.nn.functional.normalize(torch.randn(6, 8), dim=-1))
    assert index.train(iters=1)
    seen = []
    monkeypatch.setattr(index, "_retire", lambda *t: seen.extend(t))
    old = index.centroids, index.list_off_t
    assert index.train(iters=1)
    assert all(any(o is s for s in seen) for o in old)
