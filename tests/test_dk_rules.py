"""Which decode products gemm_dk takes whole, and whose K workgroups share: either side of every line."""
import pytest

from docagents_amd.ops import kernels as K


@pytest.mark.parametrize("M,N,Kd,epi,norm,whole", [
    (48, 16384, 4096, K.EPI_NONE, False, True), (48, 16400, 4096, K.EPI_NONE, False, False), (48, 8192, 4352, K.EPI_NONE, False, False),
    (64, 1024, 4096, K.EPI_NONE, False, False), (64, 1040, 4096, K.EPI_NONE, False, True), (64, 128, 4096, K.EPI_RESID, False, False),
    (64, 128, 4096, K.EPI_SWIGLU, False, True), (39, 128, 4096, K.EPI_NONE, False, True), (40, 128, 4096, K.EPI_NONE, False, False),
    (57, 128, 4096, K.EPI_NONE, True, True), (58, 128, 4096, K.EPI_NONE, True, False), (57, 256, 3328, K.EPI_NONE, False, True),
    (53, 96, 3072, K.EPI_NONE, False, False), (52, 96, 3072, K.EPI_NONE, False, True), (64, 96, 2048, K.EPI_NONE, False, True)])
def test_whole_products_of_33_rows_and_more(M, N, Kd, epi, norm, whole):
    assert K._dk_whole(M, N, Kd, epi, norm) == whole


@pytest.mark.parametrize("M,N,Kd,splits", [
    (17, 1024, 3072, 4), (16, 1024, 3072, 0), (17, 1024, 3008, 0), (32, 8192, 20480, 2), (32, 8256, 20736, 0), (32, 4096, 10240, 4),
    (32, 4096, 10176, 0), (33, 1024, 8192, 0), (24, 3072, 8192, 5), (24, 3080, 8192, 0),
    (9, 1024, 4096, 4), (8, 1024, 4096, 0), (9, 1024, 4032, 0), (16, 2048, 8192, 4), (16, 2112, 8448, 0), (16, 3072, 14336, 0),
    (8, 256, 4096, 4), (8, 320, 4096, 0), (2, 1024, 16384, 4), (2, 1024, 16320, 0), (1, 320, 8192, 0)])
def test_shared_k(M, N, Kd, splits):
    assert K._dk_split(M, N, Kd, K.EPI_RESID)[1] == splits
    assert K._dk_split(M, N, Kd, K.EPI_SWIGLU) == (0, 0, 0)
