"""Decode attention with a KV head to each query head: tiles of 32 keys and their ends, splits by length, rotated and plain
queries, a shared prefix, against 64-bit attention; no weight is rounded to 16 bits."""
import random

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K
    from docagents_amd.ops import reference as R


def _lens(kind, B, S):
    r = random.Random(B * 31 + S)
    if kind == "edges":
        return [(1, 31, 32, 33, 64, 65, 127, 128, 129, 257, S - 1, S)[i % 12] for i in range(B)]
    return [r.randint(1, S) for _ in range(B)]


# one and many rows; few pairs (the same-XCD exchange) and many; one split and several
@pytest.mark.parametrize("B,H,D,S", [(1, 32, 96, 4096), (2, 16, 96, 1024), (3, 32, 96, 4096), (12, 32, 96, 1024), (40, 32, 96, 512),
                                     (1, 8, 64, 1100), (12, 12, 64, 2048), (1, 16, 128, 4096), (13, 16, 128, 1024)])
@pytest.mark.parametrize("kind", ["edges", "ragged"])
@pytest.mark.parametrize("rope,prefix", [(False, 0), (True, 0), (True, 64)])
def test_rows(B, H, D, S, kind, rope, prefix):
    g = torch.Generator(device="cuda").manual_seed(B + D)
    lens = [max(n, prefix + 1) for n in _lens(kind, B, S)]
    kc, vc = (torch.randn(B + 1, H, S, D, device="cuda", generator=g).bfloat16() for _ in range(2))
    q = torch.randn(B, 3 * H * D, device="cuda", generator=g).bfloat16()
    slot = random.Random(1).sample(range(B), B)
    to = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    pre = to([[prefix, B]] * B) if prefix else None
    rp = (R.rope_table(S, D, 10000.0, device="cuda"), to(lens) - 1) if rope else None
    rk, rv, rq = kc.clone(), vc.clone(), q.clone()
    if rope:
        K.rope_cache(rq, rp[1], rp[0], H, H, D, slot=to(slot), k_cache=rk, v_cache=rv)
    got = K.decode_attn(q, kc, vc, to(lens), to(slot), H, H, D, S, pre=pre, rope=rp)
    assert torch.equal(kc, rk) and torch.equal(vc, rv)
    for b, n in enumerate(lens):
        k, v = rk[slot[b], :, :n].double(), rv[slot[b], :, :n].double()
        if prefix:
            k, v = torch.cat([rk[B, :, :prefix].double(), k[:, prefix:]], 1), torch.cat([rv[B, :, :prefix].double(), v[:, prefix:]], 1)
        s = (k @ rq[b, :H * D].double().view(H, D, 1)).squeeze(-1) * D ** -0.5
        want = (torch.softmax(s, -1).unsqueeze(1) @ v).reshape(-1)
        # the result is rounded to bf16 (by up to 2^-8 of it: 7 bits behind the point); scores of up to 2^5, and with them the
        # weights, are off by some 2^-19 in fp32, and the values are up to 6
        assert ((got[b].double() - want).abs() <= 2.0 ** -8 * want.abs() + 2.0 ** -15).all(), b
    assert torch.equal(K.decode_attn(q, kc, vc, to(lens), to(slot), H, H, D, S, pre=pre, rope=rp), got)


@pytest.mark.parametrize("B", [1, 8])
def test_infinite_value(B):
    """An infinite value under a weight that is not 0 makes its column infinite, whatever the weight's lower bits are."""
    H, D, S = 32, 96, 256
    g = torch.Generator(device="cuda").manual_seed(B)
    kc, vc = (torch.randn(B, H, S, D, device="cuda", generator=g).bfloat16() for _ in range(2))
    vc[:, :, 7, 3] = float("inf")
    vc[:, :, 9, 4] = float("-inf")
    q = torch.randn(B, H * D, device="cuda", generator=g).bfloat16()
    lens, slot = torch.full((B,), 200, dtype=torch.int32, device="cuda"), torch.arange(B, dtype=torch.int32, device="cuda")
    got = K.decode_attn(q, kc, vc, lens, slot, H, H, D, S).view(B, H, D)
    assert (got[..., 3] == float("inf")).all() and (got[..., 4] == float("-inf")).all()
    assert got[..., :3].isfinite().all() and got[..., 5:].isfinite().all()
