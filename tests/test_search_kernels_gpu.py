"""The vector index's kernels at the edges of their steps, splits and lists, against 64-bit products and plain sorts."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from docagents_amd.ops import kernels as K  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("d,Kk,rows", [(8, 1, None), (264, 5, None), (384, 32, 64), (768, 5, None), (1024, 20, 100),
                                       (1032, 7, None), (4096, 3, None)])
def test_topk_ranges_edges(d, Kk, rows):
    """Steps of 64 rows and what is left of them, splits that end inside a range, empty ranges and queries, a range
    named twice, removed rows and a document filter, every count of 16-B chunks per lane."""
    torch.manual_seed(d)
    N, Q = 1500, 6
    X = torch.nn.functional.normalize(torch.randn(N, d, device=DEV), dim=-1).to(torch.bfloat16)
    Qv = torch.nn.functional.normalize(torch.randn(Q, d, device=DEV), dim=-1).to(torch.bfloat16)
    rg = [[0, 1], [3, 3], [10, 74], [100, 165], [1499, 1500], [200, 263], [200, 263], [0, 1500], [7, 7]]
    ro = [0, 2, 5, 7, 8, 9, 9]
    ranges = torch.tensor(rg, dtype=torch.int32, device=DEV)
    roff = torch.tensor(ro, dtype=torch.int32, device=DEV)
    slots = (torch.arange(N, device=DEV, dtype=torch.int32) // 4).contiguous()
    slots[::5] = -1
    bitmap = torch.randint(-2**31, 2**31 - 1, (Q, N // 128 + 1), device=DEV, dtype=torch.int32)
    dots = Qv.double().cpu() @ X.double().cpu().T
    tol = d * 2.0 ** -23  # d terms summed in fp32, sum of |terms| at most about 1
    for sl, bm in ((None, None), (slots, None), (slots, bitmap)):
        s, i = K.topk_ranges(X, Qv, ranges, roff, Kk, -1.0, max_rows=1500, slots=sl, bitmap=bm, rows_per_split=rows)
        for q in range(Q):
            named = [r for a, b in rg[ro[q]:ro[q + 1]] for r in range(a, b)]
            if sl is not None:
                named = [r for r in named if sl[r] >= 0]
            if bm is not None:
                named = [r for r in named if (int(bm[q, int(sl[r]) >> 5]) >> (int(sl[r]) & 31)) & 1]
            want = sorted((float(dots[q, r]) for r in named), reverse=True)[:Kk]
            got = i[q].tolist()
            assert got[len(want):] == [-1] * (Kk - len(want)) and bool((s[q, len(want):] == -math.inf).all())
            assert all(g in named for g in got[:len(want)])
            assert all(got.count(g) <= named.count(g) for g in got[:len(want)])
            assert torch.allclose(s[q, :len(want)].double().cpu(), torch.tensor(want, dtype=torch.float64), rtol=0, atol=tol)
            at = torch.tensor([float(dots[q, g]) for g in got[:len(want)]], dtype=torch.float64)
            assert torch.allclose(s[q, :len(want)].double().cpu(), at, rtol=0, atol=tol)


@pytest.mark.parametrize("P,Kk", [(1, 1), (1, 32), (3, 5), (13, 5), (52, 20), (300, 32)])
def test_topk_merge_orders(P, Kk):
    """Empty places, ties (the smaller id first, a repeated one kept twice), one list and many: exactly a sort."""
    torch.manual_seed(P)
    Q = 3
    s = (torch.randint(-40, 40, (P, Q, Kk), device=DEV).float() / 8).contiguous()
    i = torch.randint(-2, 500, (P, Q, Kk), device=DEV, dtype=torch.int32).clamp_min(-1)
    i[:, 2] = -1
    os_, oi = K.topk_merge(s, i, Kk)
    for q in range(Q):
        c = sorted((-float(a), int(b)) for a, b in zip(s[:, q].flatten(), i[:, q].flatten()) if b >= 0)[:Kk]
        c += [(math.inf, -1)] * (Kk - len(c))
        assert [(-float(a), int(b)) for a, b in zip(os_[q], oi[q])] == c


@pytest.mark.parametrize("N,d,Q,Kk", [(1, 768, 17, 3), (15, 1024, 65, 32), (512, 384, 24, 8), (513, 768, 16, 5),
                                      (4097, 1024, 128, 5), (4100, 768, 129, 20), (20011, 384, 70, 1), (70001, 1024, 256, 5)])
def test_topk_dense_whole_shard(N, d, Q, Kk):
    """Last tiles and workgroups that are not full, one or two query blocks per wave, query groups that are not full,
    removed rows and a document filter (slots at an odd address)."""
    torch.manual_seed(N)
    X = torch.nn.functional.normalize(torch.randn(N, d, device=DEV), dim=-1).to(torch.bfloat16)
    Qv = torch.nn.functional.normalize(torch.randn(Q, d, device=DEV), dim=-1).to(torch.bfloat16)
    slots = torch.empty(N + 1, dtype=torch.int32, device=DEV)[1:]
    slots.copy_(torch.arange(N, device=DEV) // 3)
    slots[::5] = -1
    bitmap = torch.randint(-2**31, 2**31 - 1, (Q, N // 96 + 1), device=DEV, dtype=torch.int32)
    dots = Qv.double() @ X.double().T
    tol = d * 2.0 ** -23  # d terms summed in fp32, sum of |terms| at most about 1
    bits = (bitmap[:, (slots.clamp_min(0) >> 5).long()] >> (slots & 31)) & 1
    for sl, bm, thr in ((None, None, -1.0), (slots, None, 0.0), (slots, bitmap, -1.0)):
        s, i = K.topk_dense(X, Qv, Kk, thr, slots=sl, bitmap=bm)
        ok = torch.ones_like(dots, dtype=torch.bool)
        if sl is not None:
            ok &= slots >= 0
        if bm is not None:
            ok &= bits.bool()
        want = dots.masked_fill(~ok, -math.inf).masked_fill(dots < thr - tol, -math.inf)
        want = torch.nn.functional.pad(want, (0, Kk), value=-math.inf).topk(Kk).values
        near = (want - thr).abs() <= tol  # a score at the floor may fall on either side
        real = i >= 0
        assert bool((real == (want > -math.inf)).logical_or(near).all())
        assert bool((s[~real] == -math.inf).all()) and bool((i[~real] == -1).all())
        both = real & (want > -math.inf)
        assert bool(((s.double() - want).abs() <= tol)[both].all())
        at = dots.gather(1, i.clamp_min(0).long())
        assert bool(((s.double() - at).abs() <= tol)[real].all()) and bool(ok.gather(1, i.clamp_min(0).long())[real].all())
        assert all(len(set(r)) == len(r) for r in ([j for j in row if j >= 0] for row in i.tolist()))
