"""Wide products of up to 32 rows, on gemm_dk's tiles and on the streaming ones: every epilogue, the rows' norm over few and many parts, ragged edges."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K


# gemm_dk's tiles of 64 columns (the fourth: the streaming ones), one stage and more than the ring holds, parts of the norm past the
# 256 that are added up at once
@pytest.mark.parametrize("M,N,Kd,parts", [(2, 8192 + 16, 256, 1), (17, 8192 + 48, 1024, 300), (32, 16384, 256, 256), (31, 16384 + 32, 768, 511),
                                          (5, 128 * 257, 256, 33), (16, 28672, 1280, 8)])
@pytest.mark.parametrize("epi", ["none", "bias", "swiglu", "reglu", "resid"])
@pytest.mark.parametrize("norm", [False, True])
def test_wide(M, N, Kd, parts, epi, norm):
    wide(M, N, Kd, parts, epi, norm)


# every range that the rule takes to the 128-wide streaming tile: one and most of two rounds of tiles, many of a short K; one
# stage and more than the ring holds, the first and last row count, columns past a tile
@pytest.mark.parametrize("M,N,Kd,parts", [(17, 16384 + 16, 256, 1), (32, 128 * 257, 256, 256), (24, 16384 + 128, 1536, 300), (1, 16384 + 16, 768, 5),
                                          (2, 16384 + 16, 768, 511), (16, 28672 - 32, 1280, 8), (9, 49152 + 16, 256, 3), (16, 61440, 512, 33),
                                          (3, 65536 + 48, 512, 7), (5, 81920 + 16, 1024, 2)])
@pytest.mark.parametrize("epi", ["none", "bias", "swiglu", "reglu", "resid"])
@pytest.mark.parametrize("norm", [False, True])
def test_streaming(M, N, Kd, parts, epi, norm):
    assert K._dk_streams(M, -(-N // 32) * 32 if epi in ("swiglu", "reglu") else N, Kd, Kd + 64)
    wide(M, N, Kd, parts, epi, norm)


def wide(M, N, Kd, parts, epi, norm):
    if epi in ("swiglu", "reglu"):
        N = -(-N // 32) * 32
    if epi == "resid" and norm:
        pytest.skip("residual producers take no norm")
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(M, Kd + 64, device="cuda", generator=g).bfloat16()[:, :Kd]
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).bfloat16()
    bias, r = torch.randn(N, device="cuda", generator=g).bfloat16(), torch.randn(M, N, device="cuda", generator=g).bfloat16()
    code = {"none": K.EPI_NONE, "bias": K.EPI_BIAS, "swiglu": K.EPI_SWIGLU, "reglu": K.EPI_REGLU, "resid": K.EPI_RESID}[epi]
    b, resid = (None if epi == "none" else bias), (r if epi == "resid" else None)
    ssq = torch.rand(parts, 64, device="cuda", generator=g) * Kd / parts * 2
    assert K.dk_wide(M, N, Kd, a.stride(0))
    got = K.gemm_dk(a, w, epi=code, bias=b, resid=resid, norm_in=(ssq, parts, 1e-5) if norm else None).double()
    inv = (ssq[:, :M].double().sum(0) / Kd + 1e-5).rsqrt()[:, None] if norm else 1.0
    ref = (a.double() @ w.double().T) * inv + (0 if b is None else b.double())
    mag = ((a.double().abs() @ w.double().abs().T) * inv).max()
    if epi in ("swiglu", "reglu"):
        x = ref.view(M, N // 32, 2, 16)
        act = torch.nn.functional.silu if epi == "swiglu" else torch.relu
        ref = (act(x[:, :, 0]) * x[:, :, 1]).flatten(1)
    elif epi == "resid":
        ref = ref + r.double()
    # one rounding of the result, and fp32 sums of Kd products and of the parts (times the other gated factor: < 8)
    assert ((got - ref).abs() <= 2.0 ** -8 * ref.abs() + 8 * (Kd + parts) * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("N,Kd", [(4096, 2048), (2048, 2048), (20480, 2048), (4096, 4096), (6144, 4096 + 256), (1024, 14336), (3072, 6144), (640, 5120)])
@pytest.mark.parametrize("M", [3, 32, 40])
def test_rotated_chunks(M, N, Kd):
    """Products of K = 2048 n: tiles begin at a chunk of their own; of other K, and of 2048 by few columns, at the first."""
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(M, Kd, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).bfloat16()
    x = torch.randn(M, N, device="cuda", generator=g).bfloat16()
    ssq = torch.zeros(K.dk_parts(N, M), 64, device="cuda")
    got = K.gemm_dk(a, w, epi=K.EPI_RESID, resid=x, ssq_out=ssq)
    ref = a.double() @ w.double().T + x.double()
    mag = (a.double().abs() @ w.double().abs().T).max()
    assert ((got.double() - ref).abs() <= 2.0 ** -8 * ref.abs() + 8 * Kd * 2.0 ** -24 * mag).all()
    sums = got.double().square().sum(1)
    assert ((ssq[:, :M].double().sum(0) - sums).abs() <= 1e-4 * sums).all()
