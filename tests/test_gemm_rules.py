"""Which tile and how many K splits products of 33..639 rows take."""
import pytest

from docagents_amd.ops import kernels as K


@pytest.mark.parametrize("N,Kd,one", [(8192, 4096, False), (8200, 4096, True), (9216, 8192, True), (9216, 8320, False),
                                      (9216, 14336, False), (16384, 14336, False), (28672, 14336, True)])
def test_wide_products_of_up_to_64_rows(N, Kd, one):
    """Whole above 8192 columns, but in two splits where K is long and they fit one round of workgroups."""
    for M in (33, 64):
        assert (K._auto_splits(M, N, Kd) == 1) == one
    if N % 16 == 0:
        assert (K._dk_splits(N, Kd) == 1) == one
        assert K._dk_splits(N, Kd, reduce=True) >= 2
