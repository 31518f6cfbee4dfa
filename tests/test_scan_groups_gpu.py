"""The whole-shard scan's groups and the pick of their best, with exact scores: entries of -1, 0 and 1, whose products sum to
whole numbers in any order, so rows and their order are compared bit for bit, ties (to the smaller row) included."""
import math

import pytest
import torch

from docagents_amd.ops import kernels as K
from docagents_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# cols: columns that are not zero; few of them: thousands of equal scores, more than the pick collects in one pass
@pytest.mark.parametrize("N,d,Q,Kk,cols", [
    (1_100_003, 384, 20, 5, 384), (1_100_003, 384, 3, 32, 4),  # groups of two tiles
    (66_000, 1024, 70, 8, 1024), (66_000, 768, 129, 20, 3),
    (20_001, 768, 17, 32, 5), (4_100, 384, 16, 20, 6), (70_001, 1024, 1, 5, 2), (17_499, 384, 20, 5, 5), (17_501, 384, 20, 5, 5), (9_000, 768, 33, 3, 2), (100, 768, 65, 32, 768), (17, 1024, 64, 1, 4),
    (20_000, 384, 5, 20, 0), (2_100, 768, 2, 32, 0), (70_001, 768, 18, 5, 1), (300_000, 1024, 66, 32, 0)])  # (0: all rows equal)
def test_groups_and_ties(N, d, Q, Kk, cols):
    g = torch.Generator(device=DEV).manual_seed(N + d + Q)
    rand = lambda n: torch.randint(-1, 2, (n, d), device=DEV, generator=g, dtype=torch.int8).to(torch.bfloat16)  # noqa: E731
    X, Qv = rand(N), rand(Q)
    Qv[:, cols:] = 0
    X[N - 1] = Qv[0]  # (the best row of the first query: the last row of the last group)
    X[N // 2] = math.nan
    slots = torch.arange(N, device=DEV, dtype=torch.int32) // 3
    slots[::5] = -1
    slots[N - 1] = N // 3
    bitmap = torch.randint(-2**31, 2**31 - 1, (Q, N // 96 + 1), device=DEV, dtype=torch.int32, generator=g)
    for sl, bm, thr in ((None, None, -math.inf), (slots, None, 1.0), (slots, bitmap, -2.0), (slots, bitmap, 2.0 * d)):
        got_s, got_i = K.topk_dense(X, Qv, Kk, thr, slots=sl, bitmap=bm)
        want_s, want_i = R.topk_dense(X, Qv, Kk, thr, slots=sl, bitmap=bm)
        assert torch.equal(got_i, want_i) and torch.equal(got_s, want_s)
