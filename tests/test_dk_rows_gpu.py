"""The barrier-free tiles of more than 64 rows: every tile, element type, epilogue and ragged edge against 64-bit products, and the rule
that takes a product to them."""
import pytest
import torch

from docagents_amd.ops import kernels as K

TILES = {20: (32, 16), 21: (32, 32), 22: (64, 32), 23: (64, 48), 24: (64, 64), 25: (64, 96)}


def _swiglu(x):
    x = x.view(x.shape[0], x.shape[1] // 32, 2, 16)
    return (torch.nn.functional.silu(x[:, :, 0]) * x[:, :, 1]).flatten(1)


# K steps: fewer than the waves, one more than they share evenly, the rotated start's first length; rows and columns past a tile's
# edge by one and short of it, more tiles than CUs
@pytest.mark.gpu
@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("rows,more_m,cols,more_n,steps", [(2, 1, 1, 8, 1), (3, -1, 2, 32, 3), (1, 0, 5, 0, 9), (4, 17, 90, -8, 12),
                                                           (2, 31, 3, 16, 64)])
@pytest.mark.parametrize("epi", ["none", "gelu", "swiglu", "reglu", "resid"])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_tile(tile, rows, more_m, cols, more_n, steps, epi, dtype):
    bm, bn = TILES[tile]
    M, N, Kd, f16 = rows * bm + more_m, max(8, cols * bn + more_n), 64 * steps, dtype == "fp16"
    if epi in ("swiglu", "reglu"):
        if f16 or bn % 32:
            pytest.skip("no such product")
        N = -(-N // 32) * 32
    g = torch.Generator(device="cuda").manual_seed(M * 7 + N)
    t = torch.float16 if f16 else torch.bfloat16
    a = torch.randn(M, Kd + 64, device="cuda", generator=g).to(t)[:, :Kd]
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).to(t)
    b, r = torch.randn(N, device="cuda", generator=g).to(t), torch.randn(M, N + 8, device="cuda", generator=g).to(t)[:, :N]
    code = {"none": K.EPI_NONE, "gelu": K.EPI_GELU, "swiglu": K.EPI_SWIGLU, "reglu": K.EPI_REGLU, "resid": K.EPI_RESID}[epi]
    bias, resid = (None if epi == "none" else b), (r if epi == "resid" else None)
    gated = epi in ("swiglu", "reglu")
    buf = torch.full((M + 1, (N // 2 if gated else N) + 8), 7.0, device="cuda", dtype=t)
    got = K._gemm_dk_rows(a, w, bias, code, resid, buf[:M, :N // 2 if gated else N], tile)
    ref = a.double() @ w.double().T + (0 if bias is None else bias.double())
    if epi == "reglu":
        x = ref.view(M, N // 32, 2, 16)
        ref = (torch.relu(x[:, :, 0]) * x[:, :, 1]).flatten(1)
    else:
        ref = {"gelu": torch.nn.functional.gelu, "swiglu": _swiglu}.get(epi, lambda x: x)(ref)
    ref = ref + (0 if resid is None else resid.double())
    # one rounding of the result, and fp32 sums of Kd products (times the other gated factor: < 8)
    u, mag = 2.0 ** (-11 if f16 else -8), (a.double().abs() @ w.double().abs().T).max()
    assert ((got.double() - ref).abs() <= u * ref.abs() + 8 * Kd * 2.0 ** -24 * mag + 2.0 ** -24).all()
    assert (buf[M] == 7).all() and (buf[:, got.shape[1]:] == 7).all()


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,Kd,tile", [(65, 768, 768, 20), (128, 384, 1536, 20), (256, 1024, 4096, 21), (96, 4096, 4096, 22),
                                         (640, 1024, 1024, 23)])
@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
def test_as_the_rule_has_them(M, N, Kd, tile, dtype):
    """The products that gemm takes to these tiles, the same on every call and beside one another on two streams."""
    f16 = dtype == "fp16"
    assert K._dk_rows_tile(M, N, Kd, K.EPI_RESID, f16) == tile
    g = torch.Generator(device="cuda").manual_seed(M + N)
    t = torch.float16 if f16 else torch.bfloat16
    a, r = torch.randn(M, Kd, device="cuda", generator=g).to(t), torch.randn(M, N, device="cuda", generator=g).to(t)
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).to(t)
    gemm = K.gemm_f16 if f16 else K.gemm
    got = gemm(a, w, epi=K.EPI_RESID, resid=r)
    assert torch.equal(got, K._gemm_dk_rows(a, w, None, K.EPI_RESID, r, torch.empty_like(got), tile))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    outs = []
    for _ in range(4):
        outs.append(gemm(a, w, epi=K.EPI_RESID, resid=r))
        with torch.cuda.stream(side):
            outs.append(gemm(a, w, epi=K.EPI_RESID, resid=r))
    torch.cuda.synchronize()
    assert all(torch.equal(o, got) for o in outs)


@pytest.mark.parametrize("M,N,Kd,epi,want", [(64, 768, 768, K.EPI_BIAS, 0), (1280, 384, 384, K.EPI_BIAS, 0), (768, 320, 8192, K.EPI_NONE, 0),
                                             (512, 28672, 4096, K.EPI_SWIGLU, 0), (256, 4096, 14336, K.EPI_RESID, 0),
                                             (128, 4096, 4096, K.EPI_NONE, 22), (128, 1536, 384, K.EPI_GELU, 21)])
def test_rule(M, N, Kd, epi, want):
    """None up to 64 rows, from 1280 on, and where the other tiles are faster."""
    assert K._dk_rows_tile(M, N, Kd, epi) == want
    assert all(x >= 0 for t in K._DK_TILES.values() for x in t)


@pytest.mark.parametrize("M,N,Kd,epi,f16", [(171, 5920, 2688, K.EPI_SWIGLU, False), (140, 5888, 2432, K.EPI_BIAS, False), (255, 4800, 576, K.EPI_NONE, False),
                                            (777, 1344, 2240, K.EPI_GELU, False), (1022, 1088, 1216, K.EPI_BIAS, False),
                                            (1192, 864, 1216, K.EPI_GELU, True), (494, 2152, 2112, K.EPI_GELU, True), (210, 4336, 832, K.EPI_RESID, True)])
def test_rule_keeps_what_is_faster_elsewhere(M, N, Kd, epi, f16):
    """Products that took 1.05 - 1.3 times as long on the widest tile as on the streaming ones."""
    assert K._dk_rows_tile(M, N, Kd, epi, f16) == 0
