"""Prefill products whose last round of tiles is shared out along K: against 64-bit products and the whole-tile form."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from docagents_amd.ops import kernels as K  # noqa: E402

DEV = "cuda"


def _operands(M, N, Kd, dtype, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    a = torch.randn(M, Kd, device=DEV, generator=g).to(dtype)
    w = (torch.randn(N, Kd, device=DEV, generator=g) * Kd ** -0.5).to(dtype)
    bias = torch.randn(N, device=DEV, generator=g).to(dtype)
    return a, w, bias, torch.randn(M, N, device=DEV, generator=g).to(dtype)


# tiles of 256 x 256: fewer than a round (9 in 4 slices, 1 in 8), a round and some (300, 5 slices), slices of unequal
# length (33 K-tiles in 4), a last row and column tile that are not full; tiles of 128 rows; exactly a round (whole)
@pytest.mark.parametrize("M,N,Kd,tile", [(700, 768, 1024, 7), (256, 256, 4096, 7), (6244, 3072, 2048, 7),
                                         (700, 776, 64 * 33, 7), (1000, 520, 2048, 10), (6400, 3072, 2048, 10),
                                         (4096, 4096, 1024, 7)])
@pytest.mark.parametrize("epi", [K.EPI_NONE, K.EPI_BIAS, K.EPI_GELU, K.EPI_RESID, K.EPI_SWIGLU])
def test_tail(M, N, Kd, tile, epi, monkeypatch):
    a, w, bias, resid = _operands(M, N, Kd, torch.bfloat16, M + N)
    if epi == K.EPI_SWIGLU and N % 32:
        pytest.skip("gated products need whole groups")
    kw = dict(epi=epi, tile=tile, bias=None if epi in (K.EPI_NONE, K.EPI_SWIGLU) else bias,
              resid=resid if epi == K.EPI_RESID else None)
    got = K.gemm(a, w, **kw)
    again = [K.gemm(a, w, **kw) for _ in range(3)]  # the counters are back at zero, the sums in one order
    assert all(torch.equal(got, x) for x in again)
    with monkeypatch.context() as m:
        m.setattr(K, "_gemm_tail", lambda *_: (None, None))
        whole = K.gemm(a, w, **kw)
    want = a.double() @ w.double().T + (bias.double() if kw["bias"] is not None else 0)
    if epi == K.EPI_GELU:
        want = torch.nn.functional.gelu(want)
    elif epi == K.EPI_RESID:
        want = want.bfloat16().double() + resid.double()
    elif epi == K.EPI_SWIGLU:
        g = want.view(M, N // 32, 2, 16)
        want = (torch.nn.functional.silu(g[:, :, 0]) * g[:, :, 1]).reshape(M, N // 2)

    def rel(x):
        return float((x.double() - want).norm() / want.norm())
    assert rel(got) <= 1.01 * rel(whole) + 1e-6  # as near as the whole tiles are


@pytest.mark.parametrize("M,N,Kd", [(3000, 1024, 4096), (24105, 1024, 4096)])
def test_tail_f16(M, N, Kd, monkeypatch):
    a, w, bias, resid = _operands(M, N, Kd, torch.float16, M)
    got = K.gemm_f16(a, w, bias=bias, epi=K.EPI_RESID, resid=resid)
    with monkeypatch.context() as m:
        m.setattr(K, "_gemm_tail", lambda *_: (None, None))
        whole = K.gemm_f16(a, w, bias=bias, epi=K.EPI_RESID, resid=resid)
    want = a.double() @ w.double().T + bias.double() + resid.double()

    def rel(x):
        return float((x.double() - want).norm() / want.norm())
    assert rel(got) <= 1.01 * rel(whole) + 1e-6


def test_tail_streams():
    """Products beside each other on several streams, more of them than keep scratch, and captured ones: the same bits."""
    a, w, _, _ = _operands(700, 768, 2048, torch.bfloat16, 1)
    want = a.double() @ w.double().T
    first = K.gemm(a, w, tile=7)
    assert float((first.double() - want).norm() / want.norm()) < 2.0 ** -8
    streams = [torch.cuda.Stream() for _ in range(K.TAIL_STREAMS + 2)]
    torch.cuda.synchronize()
    out = []
    for _ in range(4):
        for s in streams:
            with torch.cuda.stream(s):
                out.append(K.gemm(a, w, tile=7))
    torch.cuda.synchronize()
    assert all(torch.equal(x, first) for x in out)
    assert len(K._TAIL) <= K.TAIL_STREAMS
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = [K.gemm(a, w, tile=7) for _ in range(2)]
    for _ in range(3):
        for x in captured:
            x.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert all(torch.equal(x, first) for x in captured)
        assert torch.equal(K.gemm(a, w, tile=7), first)
