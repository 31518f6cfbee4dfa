"""fp8 products on tiles of 64 and 128 rows: the same bits as the rows of a product large enough for 256 x 256 tiles (which is
checked against the oracle), ends of tiles in both directions, every epilogue."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K


# rows of the whole product, and of its parts: on tiles of 64, and (the last of them) of 128
@pytest.mark.parametrize("N,Kd,M,parts", [(2304, 768, 4096, [1, 15, 64, 65, 200, 3000]), (200, 128, 32768, [1, 63, 130, 20000]),
                                          (4096, 1024, 4096, [33, 1900])])
@pytest.mark.parametrize("epi", [0, 1, 2, 3, 4])
def test_same_bits(N, Kd, M, parts, epi):
    if epi == 3 and N % 32:
        pytest.skip("halves interleaved by 16")
    g = torch.Generator(device="cuda").manual_seed(N + Kd)
    rand = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()  # noqa: E731
    aq, sa = K.quant_fp8(rand(M, Kd))
    wq, sw = K.quant_weight_fp8(rand(N, Kd))
    bias, resid = (rand(N) if epi in (1, 2, 4) else None), (rand(M, N) if epi == 4 else None)
    assert [K.lib().da_gemm_fp8_tile(m, N) for m in (*parts, M)] == [64] * (len(parts) - 1) + [128, 256]
    want = K.gemm_fp8(aq, sa, wq, sw, bias=bias, epi=epi, resid=resid)
    for m in parts:
        at = (M - m) // 2
        got = K.gemm_fp8(aq[at:at + m], sa[at:at + m], wq, sw, bias=bias, epi=epi, resid=None if resid is None else resid[at:at + m])
        assert torch.equal(got, want[at:at + m]), m
