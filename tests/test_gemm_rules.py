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


@pytest.mark.parametrize("M,N,Kd,tile", [(300, 12288, 4096, 18), (448, 9216, 3072, 18), (160, 768, 1024, 16), (300, 3072, 8192, 16),
                                         (129, 320, 14336, 16), (512, 4096, 4096, 15), (200, 28672, 4096, 7),
                                         (256, 4096, 14336, 14), (639, 3072, 8192, 10)])
def test_tile_of_129_to_639_rows(M, N, Kd, tile):
    """Few or short rounds on the streaming tiles, long ones of many columns on the phase-split kernel."""
    got, splits = K._row_tile(M, N, Kd)
    assert got == tile and (Kd // 64) % splits == 0 and Kd // 64 // splits >= 4
    # (partials of 32 MB below 256 rows and 20 MB from there)
    assert splits == 1 or splits * -(-M // 64) * -(-N // 128) <= (1024 if M < 256 else 640)


@pytest.mark.parametrize("M", [65, 128, 129, 300, 639])
@pytest.mark.parametrize("N,Kd", [(768, 768), (4096, 4096), (28672, 4096), (64, 1 << 22)])
def test_splits_of_rows_too_long_for_the_streaming_tiles(M, N, Kd):
    """One round of 64 x 128 tiles at most, or four splits up to 128 rows; four K-steps a split."""
    s = K._auto_splits(M, N, Kd)
    assert (Kd // 64) % s == 0 and (s == 1 or Kd // 64 // s >= 4)
    assert s <= 4 if M <= 128 else s == 1 or s * -(-M // 64) * -(-N // 128) <= 256
