"""For how many rows a delta layer's single tokens run in one launch: either side of every line."""
import pytest
import torch

from docagents_amd.ops import kernels as K


@pytest.mark.parametrize("H,Kd,V,ra,rg,rows,one", [
    (32, 128, 128, 128, 128, 300, True), (64, 128, 128, 128, 128, 300, True), (32, 128, 128, 256, 256, 16, True),
    (32, 128, 128, 256, 256, 64, False), (32, 128, 128, 128, 512, 64, False), (8, 128, 128, 512, 512, 16, True), (8, 128, 128, 512, 512, 128, False),
    (16, 96, 96, 64, 256, 128, True), (16, 96, 96, 64, 256, 300, False), (8, 64, 64, 256, 256, 256, False), (1, 128, 128, 1024, 1024, 1, False)])
def test_rows(H, Kd, V, ra, rg, rows, one):
    assert (rows <= K.delta_step_fits(torch.bfloat16, H, H, Kd, V, 4, ra, rg)) == one
