"""Grouped-query decode attention with splits by the rows' own length, against fp32."""
import pytest
import torch

pytestmark = pytest.mark.gpu

from docagents_amd.ops import kernels as K  # noqa: E402
from docagents_amd.ops import reference as R  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("H,Hkv,D", [(8, 2, 128), (16, 8, 64), (8, 1, 128)])
@pytest.mark.parametrize("chunk", [0, 64, 512, 640])
def test_rows_of_every_length(H, Hkv, D, chunk, monkeypatch):
    """One key, a split exactly full and one key more, the whole cache; with the merge in the kernel and by itself; the
    tickets are back at zero for the launches that follow; a shared head in another slot."""
    torch.manual_seed(H + chunk)
    S, lens = 1300, [1, 63, 64, 65, 512, 513, 640, 641, 1024, 1025, 1300]
    B = len(lens)
    kc, vc = ((torch.randn(B + 1, Hkv, S, D, device=DEV)).bfloat16() for _ in range(2))
    q = torch.randn(B, H * D, device=DEV).bfloat16()
    lt = torch.tensor(lens, dtype=torch.int32, device=DEV)
    slot = torch.randperm(B, device=DEV).int()
    pre = torch.zeros(B, 2, dtype=torch.int32, device=DEV)
    pre[4:, 0], pre[4:, 1] = 64, B
    kx, vx = kc.clone(), vc.clone()
    for b in range(4, B):
        kx[slot[b], :, :64], vx[slot[b], :, :64] = kc[B, :, :64], vc[B, :, :64]
    for p, k, v in ((None, kc, vc), (pre, kx, vx)):
        want = R.decode_attn(q, k, v, lt, slot, H, Hkv, D).float()
        for fused in (True, False):
            monkeypatch.setattr(K, "_FUSED_COMBINE", fused)
            for _ in range(3):
                got = K.decode_attn(q, kc, vc, lt, slot, H, Hkv, D, max_len=S, chunk=chunk, pre=p).float()
                # weights and result are rounded to bf16: 2^-8 of values of about 1 each
                assert bool(((got - want).abs() <= 2.0 ** -7 * (1 + want.abs())).all())


@pytest.mark.parametrize("H,Hkv,D,B,S,route", [
    (8, 2, 128, 11, 1000, "by_len"), (8, 1, 64, 11, 8200, "by_len"), (16, 8, 64, 11, 1500, "by_len"),
    (16, 8, 128, 24, 333, "rows"), (32, 8, 64, 32, 1027, "rows"), (8, 4, 128, 11, 1300, "even"),
])
def test_automatic_split(H, Hkv, D, B, S, route, monkeypatch):
    """Rows at the edges of a split's 256 keys, one key, the whole cache; splits past a row's keys do nothing."""
    torch.manual_seed(S)
    chunk, nsplit, by_len = K._gqa_split(B, Hkv, S)
    assert route == ("by_len" if by_len else "rows" if nsplit == 1 else "even")
    lens = ([1, 64, 255, 256, 257, 300, 511, 512, 513, S - 1, S] * 3)[:B]
    lens = [min(n, S) for n in lens]
    kc, vc = (torch.randn(B, Hkv, S, D, device=DEV).bfloat16() for _ in range(2))
    q = torch.randn(B, H * D, device=DEV).bfloat16()
    lt, slot = torch.tensor(lens, dtype=torch.int32, device=DEV), torch.randperm(B, device=DEV).int()
    want = R.decode_attn(q, kc, vc, lt, slot, H, Hkv, D).float()
    for fused in (True, False):
        monkeypatch.setattr(K, "_FUSED_COMBINE", fused)
        for _ in range(2):
            got = K.decode_attn(q, kc, vc, lt, slot, H, Hkv, D, max_len=S).float()
            assert bool(((got - want).abs() <= 2.0 ** -7 * (1 + want.abs())).all())


@pytest.mark.parametrize("B,Hkv,G,D,S,chunk", [(22, 12, 1, 96, 1088, 0), (22, 12, 1, 64, 1088, 0), (60, 12, 1, 96, 1088, 64),
                                               (60, 12, 2, 128, 1088, 64)])
def test_merges_see_this_launchs_sums(B, Hkv, G, D, S, chunk):
    """Short rows merge while their neighbours' splits still run, and leave a line of the neighbours' maxima and sums in their CU's
    L1: a merge there afterwards must not read those of the launch before. Questions change from launch to launch."""
    H, g = Hkv * G, torch.Generator(device=DEV).manual_seed(B)
    kc, vc = (torch.randn(B, Hkv, S, D, device=DEV, generator=g).bfloat16() for _ in range(2))
    lens = [1 if i * 7 % 5 < 2 else S if i % 3 else 1 + i * 389 % S for i in range(B)]
    lt, slot = torch.tensor(lens, dtype=torch.int32, device=DEV), torch.arange(B - 1, -1, -1, dtype=torch.int32, device=DEV)
    mask = torch.arange(S, device=DEV) >= lt[:, None]
    cases = []
    for _ in range(4):
        q = torch.randn(B, H * D, device=DEV, generator=g).bfloat16()
        s = (q.float().view(B, Hkv, G, D) @ kc[slot.long()].float().transpose(2, 3).contiguous()) * D ** -0.5
        p = torch.softmax(s.masked_fill(mask[:, None, None], -torch.inf), -1)
        v = vc[slot.long()].float()
        want, mag = (p @ v).reshape(B, -1), (p @ v.abs()).reshape(B, -1)
        # weights and the result are rounded to bf16
        cases.append((q, want, 2.0 ** -8 * (want.abs() + 1.02 * mag) + 2.0 ** -12))
    wrong = torch.zeros((), dtype=torch.int64, device=DEV)
    for i in range(600):
        q, want, tol = cases[i % 4]
        wrong += ((K.decode_attn(q, kc, vc, lt, slot, H, Hkv, D, S, chunk=chunk).float() - want).abs() > tol).sum()
    assert wrong.item() == 0
