"""Prefill attention with heads of 128 at the lengths and block counts where its workgroups change from four waves to eight."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K

DEV = "cuda"


# one query, a block of 128 and one more, of 256 and one more; four waves to 2048 queries, to 2816 of few blocks, and eight
@pytest.mark.parametrize("H,Hkv,lens,P", [(4, 2, [1], 0), (4, 1, [128, 5, 129], 70), (4, 4, [256, 257], 0), (4, 2, [2048], 33),
                                          (4, 2, [2049, 3], 0), (41, 41, [2100, 9], 0), (4, 1, [2816], 0), (4, 1, [2817], 0),
                                          # behind a long head: one round of blocks (128 x 2 of 256 queries) and more
                                          (64, 8, [507, 130], 759), (64, 8, [507, 130], 760), (64, 64, [1409], 511), (64, 8, [1409], 512)])
def test_prefill_of_heads_of_128(H, Hkv, lens, P):
    g = torch.Generator(device=DEV).manual_seed(sum(lens) + H)
    D, T = 128, sum(lens)
    qkv = torch.randn(T, (H + 2 * Hkv) * D, device=DEV, generator=g).bfloat16()
    pk, pv = (torch.randn(Hkv, P + 8, D, device=DEV, generator=g).bfloat16() for _ in range(2))
    cu = torch.tensor([0] + lens, device=DEV).cumsum(0).int()
    q, k, v = qkv[:, :H * D], qkv[:, H * D:(H + Hkv) * D], qkv[:, (H + Hkv) * D:]
    got = K.flash_attn_varlen(q, k, v, cu, max(lens), H, Hkv, D, causal=True, prefix=(pk, pv, P) if P else None)
    for i, n in enumerate(lens):
        a = int(cu[i])
        for h in range(H):
            s = h // (H // Hkv)
            kk = torch.cat([pk[s, :P], k[a:a + n, s * D:(s + 1) * D]]).float()
            vv = torch.cat([pv[s, :P], v[a:a + n, s * D:(s + 1) * D]]).float()
            sc = q[a:a + n, h * D:(h + 1) * D].float() @ kk.T * D ** -0.5
            sc.masked_fill_(torch.arange(P + n, device=DEV)[None] > torch.arange(n, device=DEV)[:, None] + P, -float("inf"))
            want = torch.softmax(sc, -1) @ vv
            # weights and results rounded to bf16: 2^-9 each of the values, which are of order one
            assert float((got[a:a + n, h * D:(h + 1) * D].float() - want).abs().max()) < 2.0 ** -6
