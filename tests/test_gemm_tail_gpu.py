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


# tiles of 256 x 256: fewer than a round (9 in 2 and 4 slices, 1 and 12 in 8), a round and some (300, the last 44 in 2),
# slices of unequal length (33 K-tiles in 2, 65 in 4), a last row and column tile that are not full; tiles of 128 rows; too
# short to be cut and exactly a round (whole)
@pytest.mark.parametrize("M,N,Kd,tile", [(700, 768, 2048, 7), (700, 768, 4096, 7), (256, 256, 4096, 7), (1000, 768, 8192, 7),
                                         (6244, 3072, 2048, 7), (700, 776, 64 * 33, 7), (700, 776, 64 * 65, 7),
                                         (1000, 520, 2048, 10), (6400, 3072, 2048, 10), (700, 768, 1024, 7),
                                         (4096, 4096, 1024, 7)])
@pytest.mark.parametrize("epi", [K.EPI_NONE, K.EPI_BIAS, K.EPI_GELU, K.EPI_RESID, K.EPI_SWIGLU])
def test_tail(M, N, Kd, tile, epi, monkeypatch):
    a, w, bias, resid = _operands(M, N, Kd, torch.bfloat16, M + N)
    if epi == K.EPI_SWIGLU and N % 32:
        pytest.skip("gated products need whole groups")
    kw = dict(epi=epi, tile=tile, bias=None if epi in (K.EPI_NONE, K.EPI_SWIGLU) else bias,
              resid=resid if epi == K.EPI_RESID else None)
    cut = K.lib().da_gemm_tail_ws(M, N, Kd, epi, tile) > 0
    assert cut == (epi != K.EPI_GELU and Kd > 1024)  # (else both sides below are one kernel)
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
    assert K.lib().da_gemm_tail_ws(M, N, Kd, K.EPI_RESID, 0) > 0
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


# (M, N, K, tile height's code) -> tiles behind the whole rounds, slices of each; None: left whole
@pytest.mark.parametrize("M,N,Kd,tile,cut", [
    (700, 768, 2048, 7, (9, 2)), (700, 768, 4096, 7, (9, 4)), (256, 256, 4096, 7, (1, 8)), (1000, 768, 8192, 7, (12, 8)),
    (6244, 3072, 2048, 7, (44, 2)), (700, 776, 64 * 33, 7, (12, 2)), (700, 776, 64 * 65, 7, (12, 4)),
    (1000, 520, 2048, 10, (24, 4)), (700, 768, 1024, 7, None), (4096, 4096, 1024, 7, None),
    # within one round a cut has to be worth its allocation: from 28 K-tiles; slices that fill the chip are slower in four
    (3675, 512, 1536, 10, None), (3675, 512, 2048, 10, (58, 2)), (700, 768, 1728, 10, None), (700, 768, 1792, 10, (18, 2))])
@pytest.mark.parametrize("epi", [K.EPI_NONE, K.EPI_GELU, K.EPI_RESID, K.EPI_SWIGLU])
def test_which_rounds_are_cut(M, N, Kd, tile, cut, epi):
    """A product takes scratch for as many partials as it leaves, and none where its tiles stay whole. GELU's always do."""
    height = 128 if tile == 10 else 256
    want = 0 if cut is None or epi == K.EPI_GELU else cut[0] * cut[1] * height * 256 * 4
    assert K.lib().da_gemm_tail_ws(M, N, Kd, epi, tile) == want
    if epi == K.EPI_SWIGLU and N % 32:
        return
    a, w, _, resid = _operands(M, N, Kd, torch.bfloat16, M)
    stream = torch.cuda.current_stream().cuda_stream
    part, cnt = K._gemm_tail(a.device, stream, M, N, Kd, epi, tile)
    assert (part is None and cnt is None) if not want else part.numel() * 4 == want
    got = K.gemm(a, w, epi=epi, tile=tile, resid=resid if epi == K.EPI_RESID else None)
    if cnt is not None:
        assert int(cnt.abs().max()) == 0  # back at zero
    if epi == K.EPI_NONE:
        ref = a.double() @ w.double().T
        assert float((got.double() - ref).norm() / ref.norm()) < 2.0 ** -8


def test_short_products_are_never_cut():
    for Kd in range(128, K.TAIL_MIN_K, 64):
        for M in (256, 700, 1000, 2720, 2797, 3000, 5415, 6244, 24105):
            for N in (256, 768, 1024, 2304, 3072, 4096):
                for tile in (0, 7, 10):
                    assert K.lib().da_gemm_tail_ws(M, N, Kd, K.EPI_NONE, tile) == 0


def test_scratch_is_given_back():
    """Neither a stream that runs a product once nor a whole product keeps partials; a capture has one set of counters,
    cleared once, and they are its own."""
    a, w, _, _ = _operands(700, 768, 2048, torch.bfloat16, 3)
    nbytes = K.lib().da_gemm_tail_ws(700, 768, 2048, K.EPI_NONE, 7)
    assert nbytes == 9 * 2 * 256 * 256 * 4
    out = torch.empty(700, 768, dtype=torch.bfloat16, device=DEV)
    first = K.gemm(a, w, tile=7)
    streams = [torch.cuda.Stream() for _ in range(6)]
    torch.cuda.synchronize()
    held = torch.cuda.memory_allocated()
    for s in streams:
        with torch.cuda.stream(s):
            K.gemm(a, w, tile=7, out=out)
        torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() - held <= 6 * 256 * 8 * 4
    assert torch.equal(out, first)
    side = torch.cuda.Stream()
    graphs = []
    for n in (3, 2):
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=side):
            ys = [K.gemm(a, w, tile=7) for _ in range(n)]
            cnt = K._TAIL_CAPTURED[torch.device(DEV, 0).index, side.cuda_stream][1]
        graphs.append((g, ys, cnt))
    assert graphs[0][2] is not graphs[1][2]
    for _ in range(3):
        for g, ys, cnt in graphs:
            cnt.fill_(1)  # (whatever lies there: the graph's own node clears it)
            for y in ys:
                y.zero_()
            g.replay()
            K.gemm(a, w, tile=7, out=out)
            torch.cuda.synchronize()
            assert all(torch.equal(y, first) for y in ys) and torch.equal(out, first)


def test_more_streams_than_counters(monkeypatch):
    """Counters that make room for another stream's while their product may still run."""
    monkeypatch.setattr(K, "TAIL_STREAMS", 2)
    monkeypatch.setattr(K, "_TAIL", {})
    a, w, _, _ = _operands(700, 768, 2048, torch.bfloat16, 4)
    first = K.gemm(a, w, tile=7)
    streams = [torch.cuda.Stream() for _ in range(5)]
    torch.cuda.synchronize()
    out = []
    for _ in range(6):
        for s in streams:
            with torch.cuda.stream(s):
                out.append(K.gemm(a, w, tile=7))
    torch.cuda.synchronize()
    assert all(torch.equal(x, first) for x in out) and len(K._TAIL) == 2
