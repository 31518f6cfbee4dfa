"""Range searches whose workgroups' lists meet in the launch: the edges of its steps, of its rule and of the counters' use."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K

DEV = "cuda"


@pytest.mark.parametrize("d", [384, 1024])
@pytest.mark.parametrize("rows,Kk", [(1, 5), (31, 32), (32, 1), (33, 32), (64, 5), (65, 32), (256, 32), (257, 32), (700, 5), (512, 32), (513, 32)])
def test_lists_that_meet_in_the_launch(d, rows, Kk):
    """One row, half a step, a step and one row more, one workgroup, 256 candidates and one list more; queries with fewer
    rows, and none; by ranges of the host and by lists, with removed rows; the same launch again finds its counters at zero."""
    g = torch.Generator(device=DEV).manual_seed(rows + d)
    N, Q = 4000, 5
    X, q = (torch.nn.functional.normalize(torch.randn(n, d, device=DEV, generator=g), dim=-1).bfloat16() for n in (N, Q))
    slots = torch.arange(N, device=DEV, dtype=torch.int32)
    slots[::7] = -1
    ids = torch.arange(N, device=DEV) * 3 + 1
    n = [rows, rows // 2, 0, max(1, rows - 1), rows]  # rows of each query, in two ranges
    first = [17, 900, 0, 1800, 2500]
    ranges = np.array([[a, a + m // 3, a + m // 3 + 5, a + m + 5] for a, m in zip(first, n)], dtype=np.int32).reshape(-1, 2)
    off = 2 * np.arange(Q + 1, dtype=np.int32)
    # as lists: list 2 i is the gap before range i, list 2 i + 1 the range
    order = np.lexsort((ranges[:, 1], ranges[:, 0]))
    edges = torch.tensor([0] + [x for r in order for x in ranges[r].tolist()], dtype=torch.int32, device=DEV)
    lists = torch.tensor([[2 * int(np.where(order == 2 * i + j)[0][0]) + 1 for j in (0, 1)] for i in range(Q)],
                         dtype=torch.int32, device=DEV)
    dots = q.double() @ X.double().T
    for by_list in (False, True):
        for _ in range(2):
            if by_list:
                s, got = K.topk_lists(X, q, lists, edges, Kk, -1.0, mean_rows=rows, max_rows=rows, slots=slots, ids=ids)
            else:
                s, got = K.topk_ranges(X, q, ranges, off, Kk, -1.0, max_rows=rows, slots=slots, ids=ids)
            for i in range(Q):
                r = torch.cat([torch.arange(*ranges[2 * i + j].tolist(), device=DEV) for j in (0, 1)])
                r = r[slots[r] >= 0]
                want, at = dots[i, r].sort(descending=True)
                m = min(Kk, len(r))
                assert torch.allclose(s[i, :m].double(), want[:m], rtol=0, atol=d * 2.0 ** -23)
                assert torch.allclose(dots[i, (got[i, :m] - 1) // 3], want[:m], rtol=0, atol=d * 2.0 ** -22)
                assert got[i, :m].unique().numel() == m and bool(torch.isin(got[i, :m], ids[r]).all())
                assert got[i, m:].tolist() == [-1] * (Kk - m) and bool((s[i, m:] == -float("inf")).all())


@pytest.mark.parametrize("rows,Q,Kk,split", [(512, 1, 32, 32), (513, 1, 32, 64), (6400, 1, 32, 64), (1600, 3, 10, 32), (10240, 1, 1, 32), (10241, 1, 1, 64),
                                             (10240, 1, 2, 64), (2000, 10, 5, 64), (65536, 1, 5, 64), (65537, 1, 5, 128)])
def test_half_steps(rows, Q, Kk, split):
    """Half steps for few rows in all, and no more candidates of them than are soon put together."""
    assert K._rows_per_split(rows, Q, Kk) == split


def test_streams_have_counters_of_their_own():
    """Searches on two streams at once, in eager mode and replayed, give what each gives alone."""
    g = torch.Generator(device=DEV).manual_seed(3)
    X = torch.randint(-2, 3, (20000, 384), device=DEV, generator=g, dtype=torch.int8).bfloat16()
    q = X[:8].contiguous()
    off = np.arange(9, dtype=np.int32)
    parts = [np.array([[a, a + 250]] * 8, dtype=np.int32) for a in (0, 9000)]
    want = [K.topk_ranges(X, q, r, off, 10, -1e9, max_rows=250) for r in parts]
    streams = [torch.cuda.Stream() for _ in parts]
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        kept = K.topk_ranges(X, q, parts[0], off, 10, -1e9, max_rows=250)
    for _ in range(3):
        got = [[], []]
        for _ in range(20):
            for i, st in enumerate(streams):
                with torch.cuda.stream(st):
                    got[i].append(K.topk_ranges(X, q, parts[i], off, 10, -1e9, max_rows=250))
            graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for i in (0, 1) for one in got[i] for a, b in zip(one, want[i]))
        assert all(torch.equal(a, b) for a, b in zip(kept, want[0]))
