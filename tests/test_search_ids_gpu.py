"""Searches that look up the external ids themselves, and filters whose row ranges ride in the launch's arguments."""
import numpy as np
import pytest
import torch

from docagents_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _data(N, d, Q, seed):
    g = torch.Generator().manual_seed(seed)
    X = torch.nn.functional.normalize(torch.randn(N, d, generator=g), dim=-1).to(torch.bfloat16)
    q = torch.nn.functional.normalize(torch.randn(Q, d, generator=g), dim=-1).to(torch.bfloat16)
    ids = torch.randint(0, 1 << 60, (N,), generator=g)
    return X.to(DEV), q.to(DEV), ids.to(DEV)


@pytest.mark.parametrize("N,d,Q,K", [(3, 384, 2, 5), (5000, 768, 1, 5), (5000, 768, 70, 20), (900, 64, 3, 32)])
def test_ids_of_a_dense_search(N, d, Q, K):
    from docagents_amd.ops import kernels as ops
    X, q, ids = _data(N, d, Q, 1)
    thr = 0.02  # (some of the K places stay empty)
    s, rows = ops.topk_dense(X, q, K, thr)
    s2, got = ops.topk_dense(X, q, K, thr, ids=ids)
    assert got.dtype == torch.int64 and torch.equal(s, s2) and torch.equal(got.cpu(), R.gather_ids(rows.cpu(), ids.cpu()))
    # rows past a shorter table have no id
    _, got = ops.topk_dense(X, q, K, thr, ids=ids[:N // 2 + 1])
    assert torch.equal(got.cpu(), R.gather_ids(rows.cpu(), ids[:N // 2 + 1].cpu()))
    parts = torch.stack([s, s]), torch.stack([rows, rows])
    ms, mi = ops.topk_merge(*parts, K)
    ms2, mg = ops.topk_merge(*parts, K, ids=ids)
    assert torch.equal(ms, ms2) and torch.equal(mg.cpu(), R.gather_ids(mi.cpu(), ids.cpu()))


# numbers in a table: Q + 1 offsets and two a range; 512 ride in the arguments
@pytest.mark.parametrize("Q,per", [(1, 0), (1, 1), (1, 255), (1, 256), (3, 17), (7, 36), (128, 2), (300, 3)])
def test_ranges_from_the_host(Q, per):
    from docagents_amd.ops import kernels as ops
    N, d, K = 4000, 384, 7
    X, q, ids = _data(N, d, Q, 2)
    rng = np.random.default_rng(Q * 1000 + per)
    a = np.stack([rng.choice(N // 8, per, replace=False) for _ in range(Q)]).reshape(-1) * 8
    ranges = np.stack([a, a + rng.integers(0, 9, a.size)], 1).astype(np.int32)
    off = (np.arange(Q + 1) * per).astype(np.int32)
    most = int((ranges[:, 1] - ranges[:, 0]).reshape(Q, per).sum(1).max()) if per else 0
    want = ops.topk_ranges(X, q, torch.from_numpy(ranges).to(DEV), torch.from_numpy(off).to(DEV), K, -1.0, max_rows=most)
    got = ops.topk_ranges(X, q, ranges, off, K, -1.0, max_rows=most)
    assert all(torch.equal(x, y) for x, y in zip(want, got))
    s, g = ops.topk_ranges(X, q, ranges, off, K, -1.0, max_rows=most, ids=ids)
    assert torch.equal(s, want[0]) and torch.equal(g.cpu(), R.gather_ids(want[1].cpu(), ids.cpu()))
