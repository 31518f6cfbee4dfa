"""Which decode products gemm_dk takes whole: either side of every line."""
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
