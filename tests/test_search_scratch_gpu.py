"""A search leaves the workspace of its role alone: decode graphs captured in that role keep writing to it."""
import pytest
import torch

from docagents_amd.ops import kernels as K
from docagents_amd.ops import reference as R

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# the streaming scan's group maxima and its scores, the query-major scan, and ranges: all past the megabyte reserved here
@pytest.mark.parametrize("kind,N,Q,Kk", [("dense", 300_000, 64, 5), ("dense", 9_000, 64, 5), ("blocks", 300_000, 64, 5),
                                         ("ranges", 60_000, 64, 32)])
def test_role_workspace_stays(kind, N, Q, Kk):
    g = torch.Generator(device=DEV).manual_seed(N + Q)
    X, q = (torch.randint(-1, 2, (n, 384), device=DEV, generator=g, dtype=torch.int8).bfloat16() for n in (N, Q))
    ranges = torch.tensor([[0, N]], dtype=torch.int32, device=DEV).repeat(Q, 1)
    off = torch.arange(Q + 1, dtype=torch.int32, device=DEV)

    def search(ops):
        if kind == "ranges":
            return ops.topk_ranges(X, q, ranges, off, Kk, -1e9, max_rows=N)
        return ops.topk_dense(X, q, Kk, -1e9, rows_per_block=64 if kind == "blocks" else None)

    want = search(R)
    with K.workspace_role(f"search scratch {kind} {N}"):
        K.reserve_workspace(1 << 20, DEV)
        before = K.workspace_buffer(DEV)
        graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        got = search(K)
        with torch.cuda.graph(graph, stream=side):
            captured = search(K)
        for _ in range(2):
            graph.replay()
            again = search(K)
            torch.cuda.synchronize()
            for a, b, c, d in zip(want, got, captured, again):
                assert torch.equal(a, b) and torch.equal(a, c) and torch.equal(a, d)
        assert K.workspace_buffer(DEV) is before
