"""Inverted lists scanned on the device, and row indices turned into ids there, against 64-bit products and indexing."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K
    from docagents_amd.ops import reference as R

DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.int32, torch.int64, torch.int16])
def test_gather_ids(dtype):
    ids = torch.randint(-2 ** 62, 2 ** 62, (300,), dtype=torch.int64, device=DEV)
    rows = [0, 1, 299, 300, -1, -2, 150, 2 ** 15 - 1, -2 ** 15]
    if dtype != torch.int16:
        rows += [2 ** 31 - 1, -2 ** 31]
    if dtype == torch.int64:  # (their low 32 bits name rows)
        rows += [2 ** 32, 2 ** 32 + 5, -2 ** 32, 2 ** 62, -2 ** 63]
    want = [int(ids[r]) if 0 <= r < 300 else -1 for r in rows]
    rt = torch.tensor(rows, dtype=dtype, device=DEV)
    got = K.gather_ids(rt, ids)
    assert got.dtype == torch.int64 and got.tolist() == want
    assert torch.equal(K.gather_ids(rt[None].expand(3, -1).t(), ids), got[:, None].expand(-1, 3))  # any shape and stride
    assert torch.equal(got.cpu(), R.gather_ids(rt.cpu(), ids.cpu()))
    assert K.gather_ids(rt, ids[:0]).tolist() == [-1] * len(rows)
    assert K.gather_ids(rt[:0], ids).shape == (0,)
    assert K.gather_ids(torch.arange(1000, dtype=torch.int32, device=DEV), ids).tolist() == ids.tolist() + [-1] * 700


LENGTHS = [0, 1, 64, 65, 4200, 0, 130, 63, 700, 1]


def _check(s, i, dots, named, Kk, tol):
    """Scores and rows of one query against every row that it names (dots: 64-bit scores)."""
    named = torch.tensor(named, dtype=torch.long)
    want = dots[named].sort(descending=True).values[:Kk]
    n = len(want)
    assert i[n:].tolist() == [-1] * (Kk - n) and bool((s[n:] == -float("inf")).all())
    got = i[:n].long()
    assert got.unique().numel() == n and bool(torch.isin(got, named).all())
    assert torch.allclose(s[:n].double(), want, rtol=0, atol=tol)
    assert torch.allclose(s[:n].double(), dots[got], rtol=0, atol=tol)


@pytest.mark.parametrize("d,Kk", [(128, 5), (768, 32), (1024, 1)])
@pytest.mark.parametrize("mean_rows", [1, 500, 5300])
def test_topk_lists(d, Kk, mean_rows):
    """Empty lists, lists of a step of the kernel and one row more, one much longer than all others, places that name no
    list, queries of different lists and of none, splits that end inside a later list; with removed rows and a filter; the
    expected count of rows, which only shapes the launch, wrong by far in both directions."""
    torch.manual_seed(d + mean_rows)
    off = torch.tensor([0] + LENGTHS).cumsum(0)
    N = int(off[-1])
    X = torch.nn.functional.normalize(torch.randn(N, d, device=DEV), dim=-1).bfloat16()
    lists = [[0, 1, 2, 3], [4, -1, 6, 8], [-1, -1, -1, -1], [9, 3, 4, 7], [-1, 5, 0, -1], [8, 4, 2, 6], [1, -1, 9, -1]]
    Q = len(lists)
    Qv = torch.nn.functional.normalize(torch.randn(Q, d, device=DEV), dim=-1).bfloat16()
    lt, ot = torch.tensor(lists, dtype=torch.int32, device=DEV), off.int().to(DEV)
    max_rows = int(sum(sorted(LENGTHS)[-4:]))
    slots = (torch.arange(N, device=DEV, dtype=torch.int32) // 4).contiguous()
    slots[::5] = -1
    bitmap = torch.randint(-2 ** 31, 2 ** 31 - 1, (Q, N // 128 + 1), device=DEV, dtype=torch.int32)
    dots = Qv.double().cpu() @ X.double().cpu().T
    sc, bc = slots.long().cpu(), bitmap.cpu()
    for sl, bm in ((None, None), (slots, None), (slots, bitmap)):
        s, i = K.topk_lists(X, Qv, lt, ot, Kk, -1.0, mean_rows=mean_rows, max_rows=max_rows, slots=sl, bitmap=bm)
        for q in range(Q):
            named = [r for x in lists[q] if x >= 0 for r in range(int(off[x]), int(off[x + 1]))]
            if sl is not None:
                named = [r for r in named if sc[r] >= 0]
            if bm is not None:
                named = [r for r in named if (int(bc[q, sc[r] >> 5]) >> (int(sc[r]) & 31)) & 1]
            _check(s[q].cpu(), i[q].cpu(), dots[q], named, Kk, d * 2.0 ** -23)
    s, i = K.topk_lists(X, Qv[:0], lt[:0], ot, Kk, -1.0, mean_rows=mean_rows, max_rows=max_rows)
    assert s.shape == i.shape == (0, Kk)


@pytest.mark.parametrize("probes", [1, 33, 200])
def test_many_lists(probes):
    """More lists named than a wave has lanes; every list empty but one; a threshold that most rows miss."""
    torch.manual_seed(probes)
    L, d, Q, Kk = 400, 384, 5, 7
    n = torch.randint(0, 90, (L,))
    off = torch.cat([torch.zeros(1, dtype=torch.long), n.cumsum(0)])
    N = int(off[-1])
    X = torch.nn.functional.normalize(torch.randn(N, d, device=DEV), dim=-1).bfloat16()
    Qv = torch.nn.functional.normalize(torch.randn(Q, d, device=DEV), dim=-1).bfloat16()
    lt = torch.stack([torch.randperm(L)[:probes] for _ in range(Q)]).int()
    dots = Qv.double().cpu() @ X.double().cpu().T
    longest = int(n.sort(descending=True).values[:probes].sum())
    for thr in (-1.0, 0.1):
        s, i = K.topk_lists(X, Qv, lt.to(DEV), off.int().to(DEV), Kk, thr, mean_rows=-(-probes * N // L), max_rows=longest)
        for q in range(Q):
            named = [r for x in lt[q].tolist() for r in range(int(off[x]), int(off[x + 1])) if dots[q, r] >= thr]
            _check(s[q].cpu(), i[q].cpu(), dots[q], named, Kk, d * 2.0 ** -23)
    one = torch.zeros(L + 1, dtype=torch.long)
    one[L // 2 + 1:] = N
    s, i = K.topk_lists(X, Qv, lt.to(DEV), one.int().to(DEV), Kk, -1.0, mean_rows=1, max_rows=N)
    for q in range(Q):
        _check(s[q].cpu(), i[q].cpu(), dots[q], list(range(N)) if L // 2 in lt[q].tolist() else [], Kk, d * 2.0 ** -23)


@pytest.mark.parametrize("count", [16, 17, 63, 64, 65, 128, 1000])
@pytest.mark.parametrize("by_list", [False, True])
def test_splits_that_begin_behind_many_ranges(count, by_list):
    """A query's later splits find the range that they begin in by sums over 64 ranges a step: empty ranges, ranges that
    end where a split begins, places that name no list, a query without rows beside ones with many."""
    torch.manual_seed(count)
    d, Q, Kk = 256, 3, 32
    n = torch.randint(0, 12, (Q, count))
    n[0, ::3] = 64  # (splits of 64 rows: some begin exactly at a range)
    n[1, count // 2:] = 0
    n[2] = 0
    N = int(n.sum())
    off = torch.cat([torch.zeros(1, dtype=torch.long), n.flatten().cumsum(0)])
    X = torch.nn.functional.normalize(torch.randn(N, d, device=DEV), dim=-1).bfloat16()
    Qv = torch.nn.functional.normalize(torch.randn(Q, d, device=DEV), dim=-1).bfloat16()
    order = torch.stack([torch.randperm(count) for _ in range(Q)])
    lists = torch.gather(torch.arange(Q * count).view(Q, count), 1, order)
    most = int(n.sum(1).max())
    if by_list:
        lists[torch.rand(Q, count) < 0.2] = -1
        s, i = K.topk_lists(X, Qv, lists.int().to(DEV), off.int().to(DEV), Kk, -1.0, mean_rows=1, max_rows=most)
    else:
        ranges = torch.stack([off[lists], off[lists + 1]], -1).view(-1, 2).int().to(DEV)
        ro = (torch.arange(Q + 1) * count).int().to(DEV)
        s, i = K.topk_ranges(X, Qv, ranges, ro, Kk, -1.0, max_rows=most, rows_per_split=64)
    dots = Qv.double().cpu() @ X.double().cpu().T
    for q in range(Q):
        named = [r for x in lists[q].tolist() if x >= 0 for r in range(int(off[x]), int(off[x + 1]))]
        _check(s[q].cpu(), i[q].cpu(), dots[q], named, Kk, d * 2.0 ** -23)


def test_index_without_questions():
    """A batch that holds no question, before and after training, with rows added since and with a filter."""
    from docagents_amd.index import make_index
    index = make_index("ivfflat", 384, DEV, lists=4, probes=2)
    g = torch.Generator().manual_seed(1)
    for n in (40, 5):
        x = torch.nn.functional.normalize(torch.randn(n, 384, generator=g), dim=-1)
        index.add(f"d{n}", torch.arange(n).numpy(), x)
        if n == 40:
            assert index.train(iters=1)
        for filters in (None, []):
            s, i = index.search(torch.empty(0, 384, device=DEV), 3, -1.0, filters)
            assert s.shape == i.shape == (0, 3)
