"""Which products of up to 32 rows and more than 16384 columns run on the streaming tiles: either side of every line."""
import pytest

from docagents_amd.ops import kernels as K


@pytest.mark.parametrize("M,N,Kd,streams", [
    (32, 16400, 256, True), (32, 16384, 256, False), (17, 128256, 4096, True), (33, 28672, 2048, False), (24, 28672, 8448, False),
    (16, 17920, 5120, True), (16, 16384, 5120, False), (2, 28656, 1024, True), (2, 28656, 768, False), (16, 28672, 4096, False),
    (8, 32064, 3072, False), (8, 41504, 3584, False), (8, 49152, 2048, False), (8, 49168, 2048, True), (8, 61440, 2048, True),
    (8, 61456, 2048, False), (8, 61456, 512, True), (8, 70464, 1280, False), (8, 81920, 768, False), (8, 81936, 1024, True),
    (8, 128256, 4096, False)])
def test_rule(M, N, Kd, streams):
    assert K._dk_streams(M, N, Kd, Kd) == streams
