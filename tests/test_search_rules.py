"""How many rows a wave of the whole-shard scan takes."""
import pytest

from docagents_amd.ops import kernels as K


@pytest.mark.parametrize("N,rows", [(1, 16), (512, 16), (16384, 16), (16385, 32), (32768, 32), (32769, 48), (60000, 64),
                                    (65536, 64), (262144, 64), (262145, 80), (10_000_000, 2448)])
def test_rows_of_a_wave(N, rows):
    """A round of 256 workgroups to 64 rows a wave, then 64, then as many waves as stay resident."""
    assert K._scan_rows(N) == rows
    if N <= 65536:
        assert -(-N // (4 * rows)) <= 256
