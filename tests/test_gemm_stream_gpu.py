"""The weight-streaming 64x128 tile (33..639 rows): every epilogue, K split and ragged edge against 64-bit products."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K

U = 2.0 ** -8  # a bf16 rounding


def _operands(M, N, Kd, lda=0):
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    full = torch.randn(M, lda or Kd, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).bfloat16()
    bias = torch.randn(N, device="cuda", generator=g).bfloat16()
    return full[:, :Kd], w, bias, g


def _swiglu(x):
    M, N = x.shape
    x = x.view(M, N // 32, 2, 16)
    return (torch.nn.functional.silu(x[:, :, 0]) * x[:, :, 1]).reshape(M, N // 2)


# (rows, columns, K, K splits): one K step (fewer than the ring's stages), the ring's length and one more, a last row
# and column tile that are not full, more tiles than workgroups (257 and several rounds of them), several row blocks
@pytest.mark.parametrize("M,N,Kd,splits", [(33, 128, 64, 1), (64, 136, 64 * 10, 1), (63, 96, 64 * 11, 1), (50, 16384 + 40, 64 * 7, 1), (64, 128 * 257, 128, 1),
                                           (65, 32, 128, 2), (200, 128 * 200 + 32, 192, 1), (64, 4096, 2048, 8),
                                           (129, 160, 64 * 12, 4), (639, 1024, 512, 1)])
@pytest.mark.parametrize("epi", ["none", "bias", "gelu", "swiglu", "resid"])
def test_stream_tile(M, N, Kd, splits, epi):
    if epi == "swiglu" and N % 32:
        N += 32 - N % 32
    a, w, bias, g = _operands(M, N, Kd, Kd + 64)
    code = {"none": K.EPI_NONE, "bias": K.EPI_BIAS, "gelu": K.EPI_GELU, "swiglu": K.EPI_SWIGLU, "resid": K.EPI_RESID}[epi]
    resid = torch.randn(M, N, device="cuda", generator=g).bfloat16() if epi == "resid" else None
    b = None if epi == "none" else bias
    got = K.gemm(a, w, b, epi=code, resid=resid, tile=2, splits=splits).double()
    ref = a.double() @ w.double().T + (0 if b is None else b.double())
    ref = {"gelu": torch.nn.functional.gelu, "swiglu": _swiglu}.get(epi, lambda x: x)(ref)
    if resid is not None:
        ref = ref + resid.double()
    # one rounding of the result, and fp32 sums of Kd products of size ~Kd^-1/2 (times the other gated factor: < 8)
    tol = U * ref.abs() + 8 * Kd * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T).max()
    assert ((got - ref).abs() <= tol).all()


@pytest.mark.parametrize("M,N,Kd", [(33, 8192, 512), (64, 8192 + 32, 512), (40, 16384, 256), (48, 128 * 224 + 32, 256),
                                    (33, 8192 + 16, 4352), (64, 16384, 4352), (50, 12288 + 32, 8192), (64, 16384 + 32, 512)])
@pytest.mark.parametrize("epi", ["none", "swiglu"])
def test_row_norm_without_splits(M, N, Kd, epi):
    """Wide products of 33..64 rows: the rows' scale in the epilogue (no partials), of gemm_dk (the first three) and of the streaming
    tiles of 64 and (above 16384 columns) 128."""
    N = -(-N // 32) * 32 if epi == "swiglu" else N
    code = K.EPI_SWIGLU if epi == "swiglu" else K.EPI_NONE
    assert K._dk_whole(M, N, Kd, code, True) == (N <= 16384 and Kd < 4096) and (Kd < 4096 or K._dk_splits(N, Kd) == 1)
    a, w, bias, g = _operands(M, N, Kd)
    parts = 3
    ssq = torch.rand(parts, 64, device="cuda", generator=g) * Kd / parts * 2
    got = K.gemm_dk(a, w, epi=K.EPI_SWIGLU if epi == "swiglu" else K.EPI_NONE, norm_in=(ssq, parts, 1e-5)).double()
    inv = (ssq[:, :M].double().sum(0) / Kd + 1e-5).rsqrt()[:, None]
    ref = (a.double() @ w.double().T) * inv
    mag = ((a.double().abs() @ w.double().abs().T) * inv).max()
    ref = _swiglu(ref) if epi == "swiglu" else ref
    assert ((got - ref).abs() <= U * ref.abs() + 8 * Kd * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("M,N,stages,splits", [(64, 136, 19, 2), (64, 136, 20, 2), (33, 4096 + 8, 28, 3), (48, 320, 4, 32), (64, 136, 5, 4),
                                               (64, 136, 6, 4)])
def test_split_products_either_side_of_the_ring(M, N, stages, splits):
    """K splits of up to 64 rows: 6 stages are the first on the ring, shorter ones are staged through registers."""
    Kd = 64 * stages * splits
    a, w, bias, g = _operands(M, N, Kd, Kd + 64)
    resid = torch.randn(M, N, device="cuda", generator=g).bfloat16()
    got = K.gemm(a, w, bias, epi=K.EPI_RESID, resid=resid, tile=2, splits=splits).double()
    ref = a.double() @ w.double().T + bias.double() + resid.double()
    tol = U * ref.abs() + 8 * Kd * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T).max()
    assert ((got - ref).abs() <= tol).all()


@pytest.mark.parametrize("M,N,stages,splits", [(64, 136, 5, 3), (64, 136, 6, 3), (33, 328, 7, 4)])
def test_partials_either_side_of_the_ring(M, N, stages, splits):
    """Partials that no reduce follows: 6 stages are the first on the ring."""
    Kd = 64 * stages * splits
    a, w, _, _ = _operands(M, N, Kd, Kd + 64)
    ws = torch.empty(splits, M, N, device="cuda")
    K._check(K.lib().da_gemm_partials(K._ptr(a), a.stride(0), K._ptr(w), M, N, Kd, 2, splits, K._ptr(ws), K._stream()), "partials")
    for i, (x, y) in enumerate(zip(a.double().split(64 * stages, 1), w.double().split(64 * stages, 1))):
        tol = 8 * stages * 64 * 2.0 ** -24 * (x.abs() @ y.abs().T).max()
        assert ((ws[i].double() - x @ y.T).abs() <= tol).all()


@pytest.mark.parametrize("Kd", [8192, 8192 + 256])
def test_wide_long_products(Kd):
    """More than 8192 columns: whole to K = 8192, in splits from there."""
    M, N = 40, 8192 + 64
    assert (K._dk_splits(N, Kd) == 1) == (Kd <= 8192) == (K._auto_splits(M, N, Kd) == 1)
    a, w, bias, g = _operands(M, N, Kd)
    ssq = torch.rand(3, 64, device="cuda", generator=g) * Kd / 3 * 2
    got = K.gemm_dk(a, w, epi=K.EPI_SWIGLU, norm_in=(ssq, 3, 1e-5)).double()
    inv = (ssq[:, :M].double().sum(0) / Kd + 1e-5).rsqrt()[:, None]
    ref = _swiglu((a.double() @ w.double().T) * inv)
    mag = ((a.double().abs() @ w.double().abs().T) * inv).max()
    assert ((got - ref).abs() <= U * ref.abs() + 8 * Kd * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("M,N,Kd", [(300, 12288, 256), (129, 320, 4096), (449, 1160, 64), (639, 3072, 512), (200, 2304, 8192), (130, 3072 + 8, 8192)])
@pytest.mark.parametrize("epi", ["none", "gelu", "swiglu", "resid"])
def test_mid_rows(M, N, Kd, epi):
    """129..639 rows as the rule has them: either tile, whole and in splits."""
    if epi == "swiglu" and N % 32:
        N += 32 - N % 32
    a, w, bias, g = _operands(M, N, Kd)
    code = {"none": K.EPI_NONE, "gelu": K.EPI_GELU, "swiglu": K.EPI_SWIGLU, "resid": K.EPI_RESID}[epi]
    resid = torch.randn(M, N, device="cuda", generator=g).bfloat16() if epi == "resid" else None
    b = None if epi == "none" else bias
    got = K.gemm(a, w, b, epi=code, resid=resid).double()
    ref = a.double() @ w.double().T + (0 if b is None else b.double())
    ref = {"gelu": torch.nn.functional.gelu, "swiglu": _swiglu}.get(epi, lambda x: x)(ref)
    if resid is not None:
        ref = ref + resid.double()
    tol = U * ref.abs() + 8 * Kd * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T).max()
    assert ((got - ref).abs() <= tol).all()


@pytest.mark.parametrize("M,N,Kd", [(65, 768, 1024), (200, 320, 512)])
def test_rows_too_long_for_the_streaming_tiles(M, N, Kd):
    """Rows 4 M elements apart: the register-staged tile, in splits."""
    a, w, bias, g = _operands(M, N, Kd)
    apart = torch.empty(M * (1 << 22), device="cuda", dtype=torch.bfloat16).view(M, 1 << 22)[:, :Kd]
    apart.copy_(a)
    assert K._auto_splits(M, N, Kd) > 1
    got = K.gemm(apart, w, bias, epi=K.EPI_BIAS).double()
    ref = a.double() @ w.double().T + bias.double()
    tol = U * ref.abs() + 8 * Kd * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T).max()
    assert ((got - ref).abs() <= tol).all()
