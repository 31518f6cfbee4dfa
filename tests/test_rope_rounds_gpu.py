"""QKV projections by how their tiles fill the chip: one round of 256-row tiles, a short last round shared out, whole rounds."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from docagents_amd.ops import kernels as K  # noqa: E402


# rows of one round of 256-row tiles of more than half of the chip, then rounds with a short and with a long last one
@pytest.mark.parametrize("M,one_round,apart", [(1409, True, False), (2560, True, False), (2817, False, True), (4100, False, False)])
def test_qkv_projection_by_rounds(M, one_round, apart):
    H, Hkv, D, Kd = 32, 8, 128, 4096
    N = (H + 2 * Hkv) * D
    assert K._rope_round(M, N) == one_round and (K._rope_apart(M, N, Kd) and not one_round) == apart
    g = torch.Generator(device="cuda").manual_seed(M)
    a = torch.randn(M, Kd, device="cuda", generator=g).bfloat16()
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).bfloat16()
    pos = torch.arange(M, dtype=torch.int32, device="cuda")
    slot = torch.zeros(M, dtype=torch.int32, device="cuda")
    ang = pos.double()[:, None] * 10000.0 ** (-torch.arange(0, D, 2, device="cuda").double() / D)
    cs = torch.stack([ang.cos(), ang.sin()], -1).float().contiguous()
    kc, vc = (torch.zeros(1, Hkv, M, D, device="cuda", dtype=torch.bfloat16) for _ in range(2))
    got = K.gemm_rope(a, w, pos, cs, H, Hkv, D, slot, kc, vc)
    x = (a.double() @ w.double().T).view(M, H + 2 * Hkv, D)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    turned = torch.stack([x[..., 0::2] * c - x[..., 1::2] * s, x[..., 1::2] * c + x[..., 0::2] * s], -1).flatten(-2)
    ref = torch.cat([turned[:, :H + Hkv], x[:, H + Hkv:]], 1)
    tol = 2.0 ** -8 * 3 * x.abs().amax(-1, keepdim=True)  # the product is rounded before it is turned, and after
    assert ((got.view_as(ref).double() - ref).abs() <= tol).all()
    assert ((kc[0].transpose(0, 1).double() - ref[:, H:H + Hkv]).abs() <= tol[:, H:H + Hkv]).all()
    assert ((vc[0].transpose(0, 1).double() - ref[:, H + Hkv:]).abs() <= tol[:, H + Hkv:]).all()
