"""Products of 65 to 128 rows left as fp32 partials by the streaming tile, or the register-staged one."""
import pytest
import torch

from docagents_amd.ops import kernels  # noqa: F401 - first: the two import each other
from docagents_amd.ops import seq_kernels as S


# whole and split K, columns left over, rows on either side of a wave's
@pytest.mark.gpu
@pytest.mark.parametrize("N,Kd", [(200, 64), (200, 192), (200, 256), (1032, 576), (4096, 4096), (264, 14336)])
@pytest.mark.parametrize("M", [65, 92, 97, 128])
def test_partials_of_65_to_128_rows(M, N, Kd):
    g = torch.Generator(device="cuda").manual_seed(M + N)
    a = torch.randn(M, Kd + 8, device="cuda", generator=g).bfloat16()[:, :Kd]
    w = (torch.randn(N, Kd, device="cuda", generator=g) * Kd ** -0.5).bfloat16()
    got = S.gemm_partials(a, w, own=True).double().sum(0)
    mag = (a.double().abs() @ w.double().abs().T).max()
    assert ((got - a.double() @ w.double().T).abs() <= 2 * Kd * 2.0 ** -24 * mag).all()


@pytest.mark.parametrize("M,Kd,lda,tile", [(32, 64, 64, 3), (64, 4096, 4096, 2), (65, 192, 192, 9), (65, 256, 256, 15), (128, 64, 4096, 9),
                                           (128, 14336, 14336, 15), (92, 4096, 1 << 22, 9)])
def test_tile(M, Kd, lda, tile):
    assert S._partials_tile(M, Kd, lda) == tile
