"""Encoder layers launched by one native call each: bit for bit what the operations give one by one."""
import pytest
import torch

from docagents_amd.models.bert import BertEncoder
from docagents_amd.models.configs import EncoderConfig

pytestmark = pytest.mark.gpu


# rows on either side of the few-row products, the row blocks, the split streaming tiles, small results and whole tiles
@pytest.mark.parametrize("rows", [65, 200, 345, 1100, 1700, 3000])
@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("hidden,heads,ffn", [(384, 6, 1536), (1024, 16, 4096)])
def test_layers_are_the_operations(hidden, heads, ffn, dtype, rows, monkeypatch):
    cfg = EncoderConfig(name="layers", vocab=500, hidden=hidden, layers=2, heads=heads, ffn=ffn, max_pos=512)
    enc = BertEncoder(cfg, seed=rows, dtype=dtype)
    lens = [min(300, rows - a) for a in range(0, rows, 300)]
    g = torch.Generator().manual_seed(rows)
    ids = torch.randint(0, 500, (rows,), generator=g, dtype=torch.int32).cuda()
    pos = torch.cat([torch.arange(n, dtype=torch.int32) for n in lens]).cuda()
    cu = torch.tensor([0, *lens], dtype=torch.int32).cumsum(0).int().cuda()
    got = enc.forward(ids, pos, cu, max(lens))
    monkeypatch.setattr(enc.ops, "encoder_layers_fit", lambda n: False)
    want = enc.forward(ids, pos, cu, max(lens))
    assert torch.isfinite(want).all() and torch.equal(got, want)


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp8"])
def test_no_layers(dtype, monkeypatch):
    """Embeddings alone are the result, as for the few rows of a question."""
    cfg = EncoderConfig(name="layers", vocab=500, hidden=384, layers=0, heads=6, ffn=1536, max_pos=512)
    enc = BertEncoder(cfg, seed=2, dtype=dtype)
    ids = torch.arange(80, dtype=torch.int32).cuda()
    cu = torch.tensor([0, 80], dtype=torch.int32).cuda()
    got = enc.forward(ids, ids, cu, 80)
    monkeypatch.setattr(enc.ops, "encoder_layers_fit", lambda n: False)
    assert torch.equal(got, enc.forward(ids, ids, cu, 80))


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp8"])
def test_memory_of_long_batches(dtype, monkeypatch):
    """A long batch's layers hold no more at a time than the operations do one by one."""
    rows = 20000
    cfg = EncoderConfig(name="layers", vocab=500, hidden=1024, layers=3, heads=16, ffn=4096, max_pos=512)
    enc = BertEncoder(cfg, seed=rows, dtype=dtype)
    ids = torch.zeros(rows, dtype=torch.int32).cuda()
    pos = torch.arange(rows, dtype=torch.int32).cuda() % 400
    cu = torch.arange(0, rows + 1, 400, dtype=torch.int32).cuda()

    def peak():
        enc.forward(ids, pos, cu, 400)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        held = torch.cuda.memory_allocated()
        enc.forward(ids, pos, cu, 400)
        return torch.cuda.max_memory_allocated() - held
    got = peak()
    monkeypatch.setattr(enc.ops, "encoder_layers_fit", lambda n: False)
    # (the buffers of a layer are all there at once, not one by one: a width or two of twelve more)
    assert got <= 1.2 * peak()


def test_bad_weights_are_refused():
    cfg = EncoderConfig(name="layers", vocab=500, hidden=384, layers=1, heads=6, ffn=1536, max_pos=512)
    enc = BertEncoder(cfg, seed=1)
    ids = torch.zeros(80, dtype=torch.int32).cuda()
    cu = torch.tensor([0, 80], dtype=torch.int32).cuda()
    layer = enc.w["layers"][0]
    whole = layer["wo"]
    for bad in (whole[:-8], whole.float(), whole.t()):
        layer["wo"] = bad
        with pytest.raises(ValueError, match="wo must be"):
            enc.forward(ids, ids, cu, 80)
