"""Batches of very short texts through captured buckets of 8 and 16 tokens a text."""
import numpy as np
import pytest
import torch

from docagents_amd.models.bert import BertEncoder
from docagents_amd.models.configs import encoder_config

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp8"])
def test_short_batches_match_eager(dtype):
    enc = BertEncoder(encoder_config("tiny-enc"), "cuda", seed=9, dtype=dtype)
    enc.prepare_graphs()
    assert set(enc._gs) == set(BertEncoder.SHORT_BUCKETS)
    rng = np.random.default_rng(4)
    # the first row past a bucket, its last, and one text more than it has
    for nb, T in BertEncoder.SHORT_BUCKETS:
        for n, tot in ((nb, T - 1), (nb, T), (nb // 2 + 1, T - 1), (nb + 1, T - 1)):
            if n > 64 or n > tot:
                continue
            lens = np.full(n, tot // n)
            lens[:tot - lens.sum()] += 1
            seqs = [[int(t) for t in rng.integers(5, 200, size=int(m))] for m in lens]
            got, want = enc.encode_batch(seqs), enc.encode_packed(seqs)
            assert got.shape == want.shape
            cos = torch.nn.functional.cosine_similarity(got.float(), want.float())
            assert float(cos.min()) > 0.999, (nb, T, n, tot)


def test_one_graph_a_row_count():
    """Buckets of as many rows share a graph: no more of them to capture and to keep than the row counts are."""
    enc = BertEncoder(encoder_config("tiny-enc"), "cuda", seed=9)
    enc.prepare_graphs()
    graphs = {id(e[1]) for e in (*enc._gb.values(), *enc._gs.values())}
    assert len(graphs) == len({T for _, T in (*BertEncoder.BATCH_BUCKETS, *BertEncoder.SHORT_BUCKETS)}) == 6


@pytest.mark.parametrize("dtype", ["bf16", "fp16", "fp8"])
def test_a_text_sees_no_other(dtype):
    """Another text in its neighbour's place changes no bit of a text's embedding."""
    enc = BertEncoder(encoder_config("tiny-enc"), "cuda", seed=9, dtype=dtype)
    enc.prepare_graphs()
    rng = np.random.default_rng(5)
    for nb, T in (*BertEncoder.BATCH_BUCKETS, *BertEncoder.SHORT_BUCKETS):
        lens = np.full(nb, (T - 1) // nb)
        lens[: T - 1 - lens.sum()] += 1
        seqs = [[int(t) for t in rng.integers(5, 200, size=int(m))] for m in lens]
        for other in {0, nb // 2, nb - 1}:
            new = list(seqs)
            new[other] = [int(t) for t in rng.integers(5, 200, size=len(seqs[other]))]
            a, b = enc.encode_batch(seqs), enc.encode_batch(new)
            rest = [i for i in range(nb) if i != other]
            assert torch.equal(a[rest], b[rest]) and not torch.equal(a[other], b[other]), (nb, T, other)
