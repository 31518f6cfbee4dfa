"""The weight-streaming tiles of more than 64 rows: every tile, element type, epilogue and ragged edge against 64-bit products."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K

TILES = {14: (128, 128), 15: (128, 64), 16: (64, 64), 17: (64, 128), 18: (192, 128)}


def _swiglu(x):
    x = x.view(x.shape[0], x.shape[1] // 32, 2, 16)
    return (torch.nn.functional.silu(x[:, :, 0]) * x[:, :, 1]).flatten(1)


def _within(got, ref, mag, Kd, f16=False):
    # one rounding of the result, and fp32 sums of Kd products (times the other gated factor: < 8)
    u = 2.0 ** (-11 if f16 else -8)
    return ((got.double() - ref).abs() <= u * ref.abs() + 8 * Kd * 2.0 ** -24 * mag + 2.0 ** -24).all()


# K steps: one, fewer than the ring's stages, more, many units of few (the ring runs across units); splits
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("more_m,more_n,cols,steps,splits", [(1, 8, 1, 2, 1), (-1, 32, 2, 3, 1), (0, 0, 3, 13, 1), (63, 40, 90, 2, 1),
                                                             (17, 64, 2, 12, 4), (1, 8, 1, 16, 2)])
@pytest.mark.parametrize("epi", ["none", "gelu", "swiglu", "resid"])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_tile(tile, more_m, more_n, cols, steps, splits, epi, dtype):
    bm, bn = TILES[tile]
    M, N, Kd = 2 * bm + more_m, cols * bn + more_n, 64 * steps
    f16 = dtype == "fp16"
    if epi == "swiglu":
        if f16:
            pytest.skip("the fp16 encoder has no gated product")
        N = -(-N // 32) * 32
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    t = torch.float16 if f16 else torch.bfloat16
    a = torch.randn(M, Kd + 64, device="cuda", generator=g).to(t)[:, :Kd]
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).to(t)
    b, r = torch.randn(N, device="cuda", generator=g).to(t), torch.randn(M, N, device="cuda", generator=g).to(t)
    code = {"none": K.EPI_NONE, "gelu": K.EPI_GELU, "swiglu": K.EPI_SWIGLU, "resid": K.EPI_RESID}[epi]
    bias, resid = (None if epi == "none" else b), (r if epi == "resid" else None)
    if f16:
        got = torch.empty(M, N, device="cuda", dtype=t)
        ws = torch.empty(splits * M * N, device="cuda")
        K._check(K.lib().da_gemm_f16(K._ptr(a), a.stride(0), K._ptr(w), K._ptr(got), N, K._ptr(bias), K._ptr(resid), N,
                                     M, N, Kd, code, tile, splits, K._ptr(ws), None, None, K._stream()), "gemm_f16")
    else:
        got = K.gemm(a, w, bias, epi=code, resid=resid, tile=tile, splits=splits)
    ref = a.double() @ w.double().T + (0 if bias is None else bias.double())
    ref = {"gelu": torch.nn.functional.gelu, "swiglu": _swiglu}.get(epi, lambda x: x)(ref)
    ref = ref + (0 if resid is None else resid.double())
    assert _within(got, ref, (a.double().abs() @ w.double().abs().T).max(), Kd, f16)


@pytest.mark.parametrize("M,N,Kd", [(65, 768, 768), (128, 1024, 4096), (130, 3072, 1024), (300, 6144, 512), (639, 768, 3072),
                                    (640, 768, 3072), (1279, 384, 1536), (1280, 384, 1536)])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_as_the_rule_has_them(M, N, Kd, dtype):
    """Either side of the rule's lines, whole and in splits, repeated and on another stream at the same time."""
    f16 = dtype == "fp16"
    g = torch.Generator(device="cuda").manual_seed(M + N)
    t = torch.float16 if f16 else torch.bfloat16
    a, r = torch.randn(M, Kd, device="cuda", generator=g).to(t), torch.randn(M, N, device="cuda", generator=g).to(t)
    w, b = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).to(t), torch.randn(N, device="cuda", generator=g).to(t)
    gemm = K.gemm_f16 if f16 else K.gemm
    got = gemm(a, w, b, epi=K.EPI_RESID, resid=r)
    ref = a.double() @ w.double().T + b.double() + r.double()
    # (from 640 rows the phase-split kernel rounds the product before the residual)
    ref_mag = (a.double().abs() @ w.double().abs().T).max()
    u = 2.0 ** (-11 if f16 else -8)
    assert ((got.double() - ref).abs() <= u * (ref.abs() + (ref - r.double()).abs()) + 8 * Kd * 2.0 ** -24 * ref_mag).all()
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    outs = []
    for _ in range(4):
        outs.append(gemm(a, w, b, epi=K.EPI_RESID, resid=r))
        with torch.cuda.stream(side):
            outs.append(gemm(a, w, b, epi=K.EPI_RESID, resid=r))
    torch.cuda.synchronize()
    assert all(torch.equal(o, got) for o in outs)


# (wide: into columns of a wider buffer, which the rotation behind a product does not take)
@pytest.mark.parametrize("M,apart,wide", [(432, True, False), (1280, False, False), (432, True, True)])
def test_qkv_projection_either_way(M, apart, wide):
    H, Hkv, D, Kd = 32, 8, 128, 4096
    N = (H + 2 * Hkv) * D
    assert K._rope_apart(M, N, Kd) == apart
    g = torch.Generator(device="cuda").manual_seed(M)
    a = torch.randn(M, Kd, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).bfloat16()
    pos = torch.arange(M, dtype=torch.int32, device="cuda")
    slot = torch.ones(M, dtype=torch.int32, device="cuda")
    ang = pos.double()[:, None] * 10000.0 ** (-torch.arange(0, D, 2, device="cuda").double() / D)
    cs = torch.stack([ang.cos(), ang.sin()], -1).float().contiguous()
    kc, vc = (torch.zeros(2, Hkv, M, D, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    buf = torch.full((M, N + 64), 7.0, device="cuda", dtype=torch.bfloat16)
    got = K.gemm_rope(a, w, pos, cs, H, Hkv, D, slot, kc, vc, out=buf[:, :N] if wide else None)
    assert (buf[:, N:] == 7).all() and (not wide or got.data_ptr() == buf.data_ptr())
    x = (a.double() @ w.double().T).view(M, H + 2 * Hkv, D)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    turned = torch.stack([x[..., 0::2] * c - x[..., 1::2] * s, x[..., 1::2] * c + x[..., 0::2] * s], -1).flatten(-2)
    ref = torch.cat([turned[:, :H + Hkv], x[:, H + Hkv:]], 1)
    # the product is rounded before it is turned, and after
    tol = 2.0 ** -8 * 3 * x.abs().amax(-1, keepdim=True)
    assert ((got.view_as(ref).double() - ref).abs() <= tol).all()
    assert ((kc[1].transpose(0, 1).double() - ref[:, H:H + Hkv]).abs() <= tol[:, H:H + Hkv]).all()
    assert ((vc[1].transpose(0, 1).double() - ref[:, H + Hkv:]).abs() <= tol[:, H + Hkv:]).all()
    assert not kc[0].any() and not vc[0].any()
