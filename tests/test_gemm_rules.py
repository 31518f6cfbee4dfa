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


@pytest.mark.parametrize("M,N,Kd,tile", [(300, 12288, 4096, 11), (448, 9216, 3072, 11), (160, 768, 1024, 11), (300, 3072, 8192, 11),
                                         (129, 320, 14336, 11), (512, 4096, 4096, 2), (200, 28672, 4096, 2),
                                         (256, 4096, 14336, 2), (639, 3072, 8192, 2)])
def test_tile_of_129_to_639_rows(M, N, Kd, tile):
    """A last round of 128x128 tiles that is nearly empty, and short products, are for the register-staged tile."""
    got, splits = K._mid_tile(M, N, Kd)
    assert got == tile and (Kd // 64) % splits == 0 and Kd // 64 // splits >= 4
    # (a prefill must not outgrow the workspace of captured decode steps)
    assert splits == 1 or splits * -(-M // 64) * -(-N // 128) <= (1024 if M < 256 else 640)
