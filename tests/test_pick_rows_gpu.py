"""The rows of a scan's best groups, scored again from registers (up to 8 tiles) or through LDS (more), bit for bit."""
import math

import pytest
import torch

from docagents_amd.ops import kernels as K
from docagents_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.mark.parametrize("d", [384, 768, 1024])
# tiles of a query: 1, 8, 9 and 32; groups of two tiles: 8 and 10; the last group is short
@pytest.mark.parametrize("N,Kk", [(16_017, 1), (30_001, 8), (30_001, 9), (60_007, 32), (1_060_001, 4), (1_060_001, 5)])
def test_rows_of_the_best_groups(d, N, Kk):
    g = torch.Generator(device=DEV).manual_seed(N + d + Kk)
    X, q = (torch.randint(-1, 2, (n, d), device=DEV, generator=g, dtype=torch.int8).bfloat16() for n in (N, 19))
    X[N - 1] = q[0]
    X[N - 17] = math.nan
    slots = torch.arange(N, device=DEV, dtype=torch.int32)
    slots[::9] = -1
    for sl in (None, slots):
        got, want = K.topk_dense(X, q, Kk, -math.inf, slots=sl), R.topk_dense(X, q, Kk, -math.inf, slots=sl)
        assert torch.equal(got[1], want[1]) and torch.equal(got[0], want[0])


@pytest.mark.parametrize("N,Kk", [(60_007, 32), (1_060_001, 5), (30_001, 8)])
@pytest.mark.parametrize("n", [0, 1, 7, 30])
def test_few_groups_with_rows(N, Kk, n):
    """Fewer groups than K that have rows: as many as rows reach the least similarity, and none."""
    d = 384
    g = torch.Generator(device=DEV).manual_seed(N + n)
    X, q = (torch.randint(-1, 2, (m, d), device=DEV, generator=g, dtype=torch.int8).bfloat16() for m in (N, 19))
    X[torch.randperm(N, device=DEV, generator=g)[:n]] = q[3]
    thr = float(q[3].float().square().sum()) if n else 1e6
    got, want = K.topk_dense(X, q, Kk, thr), R.topk_dense(X, q, Kk, thr)
    assert torch.equal(got[1], want[1]) and torch.equal(got[0], want[0])
    assert int((got[1][3] >= 0).sum()) == min(n, Kk)
