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
