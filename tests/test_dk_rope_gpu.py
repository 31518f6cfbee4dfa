"""The decode-sized QKV projection with rotation and cache write inside, against the product and ``rope_cache`` behind it."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K
    from docagents_amd.ops.reference import rope_table

DEV = "cuda"


# heads of 64, 96 and 128; tiles of 16 to 64 columns, a last one that is not full, heads that end inside a tile; every row block
@pytest.mark.parametrize("H,Hkv,D,k", [(4, 2, 64, 256), (8, 8, 96, 512), (32, 8, 128, 1024), (32, 32, 96, 768), (40, 8, 128, 512), (33, 1, 64, 256)])
@pytest.mark.parametrize("M", [2, 16, 17, 33, 48, 49, 64])
def test_rotated_projection(H, Hkv, D, k, M):
    g = torch.Generator(device=DEV).manual_seed(M * 7 + H)
    N, slots, seq = (H + 2 * Hkv) * D, 5, 300
    a = torch.randn(M, k, device=DEV, generator=g).bfloat16()
    w = (torch.randn(N, k, device=DEV, generator=g) * k ** -0.5).bfloat16()
    at = torch.randperm(slots * seq - 1, device=DEV, generator=g)[:M]  # (no two rows at one place)
    at[-1] = slots * seq - 1
    slot, pos = (at // seq).int(), (at % seq).int()
    cs = rope_table(seq, D, 10000.0, torch.device(DEV))
    ssq = torch.rand(3, 64, device=DEV, generator=g) * k
    assert K.dk_rope_fits(M, N, k, k)
    for norm in (None, (ssq, 3, 1e-5)):
        kc, vc = (torch.full((slots, Hkv, seq, D), 7.0, device=DEV, dtype=torch.bfloat16) for _ in range(2))
        want = K.gemm_dk(a, w, norm_in=norm)
        plain = want.clone()
        K.rope_cache(want, pos, cs, H, Hkv, D, slot=slot, k_cache=kc.clone(), v_cache=vc.clone())
        got = K.gemm_dk_rope(a, w, pos, cs, H, Hkv, D, slot, kc, vc, norm_in=norm)
        assert torch.equal(got, want)  # the same rounded values, rotated by the same fused products in fp32
        assert torch.equal(got[:, (H + Hkv) * D:], plain[:, (H + Hkv) * D:])
        for c, o in ((kc, got[:, H * D:(H + Hkv) * D]), (vc, got[:, (H + Hkv) * D:])):
            assert torch.equal(c[slot.long(), :, pos.long()], o.reshape(-1, Hkv, D))
        touched = torch.zeros(slots, seq, dtype=torch.bool, device=DEV)
        touched[slot.long(), pos.long()] = True
        assert bool((kc.transpose(1, 2)[~touched] == 7).all()) and bool((vc.transpose(1, 2)[~touched] == 7).all())
        only_q = torch.full((M, N), 3.0, device=DEV, dtype=torch.bfloat16)
        K.gemm_dk_rope(a, w, pos, cs, H, Hkv, D, slot, kc, vc, norm_in=norm, out=only_q, kv_out=False)
        assert torch.equal(only_q[:, :H * D], got[:, :H * D]) and bool((only_q[:, H * D:] == 3).all())


@pytest.mark.parametrize("N,k", [(6144, 4096), (9216, 3072), (5120, 5120), (10240, 8192)])
def test_which_projections_take_it(N, k):
    """Those of grouped queries, of as many heads of keys, and wider ones: what one plain gemm_dk launch is the faster way for. One row, more than 64
    and a long K of many rows go the other way."""
    for M in (1, 2, 16, 17, 32, 33, 48, 64, 65):
        assert K.dk_rope_fits(M, N, k, k) == (2 <= M <= (64 if k <= 4096 else 32)), M


@pytest.mark.parametrize("M", [1, 65])
def test_what_it_refuses(M):
    D, H, Hkv, k = 64, 4, 2, 256
    a, w = torch.randn(M, k, device=DEV).bfloat16(), torch.randn((H + 2 * Hkv) * D, k, device=DEV).bfloat16()
    slot, pos = torch.zeros(M, device=DEV, dtype=torch.int32), torch.arange(M, device=DEV, dtype=torch.int32)
    kc, vc = torch.zeros(2, 1, Hkv, 128, D, device=DEV, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        K.gemm_dk_rope(a, w, pos, rope_table(128, D, 10000.0, torch.device(DEV)), H, Hkv, D, slot, kc, vc)
