"""The encoders' bidirectional attention (D = 64): ends of tiles and query blocks, a moving maximum, fewer KV heads, packed and
separate rows, against 64-bit attention."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K


@pytest.mark.parametrize("dtype,H,Hkv", [(torch.float16, 16, 16), (torch.bfloat16, 12, 12), (torch.bfloat16, 8, 2),
                                         (torch.float16, 8, 4)])
@pytest.mark.parametrize("lens", [[1], [32], [65, 0, 1], [31, 33, 63, 64, 127, 128, 129, 191, 192, 193, 257], [700, 5, 512, 320]])
@pytest.mark.parametrize("rising", [False, True])
def test_rows(dtype, H, Hkv, lens, rising):
    D, T = 64, sum(lens)
    g = torch.Generator(device="cuda").manual_seed(T + H)
    x = torch.randn(T, (H + 2 * Hkv) * D, device="cuda", generator=g)
    at = [0]
    for n in lens:
        if rising:  # scores that grow along the keys: the maximum moves at every tile, weights of all magnitudes
            x[at[-1]:at[-1] + n, H * D:(H + Hkv) * D] *= torch.linspace(0.05, 4, n, device="cuda").view(-1, 1)
        at.append(at[-1] + n)
    x = x.to(dtype)
    q, k, v = x[:, :H * D], x[:, H * D:(H + Hkv) * D], x[:, (H + Hkv) * D:]
    cu = torch.tensor(at, device="cuda", dtype=torch.int32)
    fn = K.flash_attn_f16 if dtype == torch.float16 else K.flash_attn_varlen
    out = torch.full((T + 1, H * D), 7.0, device="cuda", dtype=dtype)
    got = fn(q, k, v, cu, max(lens), H, Hkv, D, False, out=out[:T])
    assert (out[T] == 7).all()
    ulp = 2.0 ** -10 if dtype == torch.float16 else 2.0 ** -7
    for a, n in zip(at, lens):
        r = lambda t, h: t[a:a + n].double().view(n, h, D).transpose(0, 1).repeat_interleave(H // h, 0)  # noqa: E731
        p = torch.softmax(r(q, H) @ r(k, Hkv).transpose(1, 2) * D ** -0.5, -1)
        want, mag = p @ r(v, Hkv), p @ r(v, Hkv).abs()
        err = (got[a:a + n].double().view(n, H, D).transpose(0, 1) - want).abs()
        # weights and the result are rounded to the type (half an ulp each); fp16 weights below 2^-14 of the row's scale to 2^-25
        assert (err <= ulp * (mag + want.abs()) / 2 * 1.01 + 2.0 ** -13).all()


def test_infinite_scores():
    """A query whose first 64 scores are -inf in fp32, beside ordinary ones of its wave."""
    D, H, T = 64, 2, 150
    g = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn(T, H * D, device="cuda", generator=g) for _ in range(3))
    q[:, 0], k[:, 0] = 0, 0
    q[5, 0], k[:64, 0] = 2.0 ** 100, -(2.0 ** 100)
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    cu = torch.tensor([0, T], device="cuda", dtype=torch.int32)
    got = K.flash_attn_varlen(q, k, v, cu, T, H, H, D, False).double().view(T, H, D).transpose(0, 1)
    r = lambda t: t.double().view(T, H, D).transpose(0, 1)  # noqa: E731
    p = torch.softmax(r(q) @ r(k).transpose(1, 2) * D ** -0.5, -1)
    want, mag = p @ r(v), p @ r(v).abs()
    # weights and the result are rounded to the type
    assert ((got - want).abs() <= 2.0 ** -8 * (mag + want.abs()) * 1.01 + 2.0 ** -13).all()


def test_values_near_the_largest():
    """A value of 3e38 under weights of a few per cent, where the scores rise along the keys."""
    D, H, T = 64, 2, 300
    g = torch.Generator(device="cuda").manual_seed(6)
    q, k, v = (torch.randn(T, H * D, device="cuda", generator=g) for _ in range(3))
    k *= torch.linspace(0.05, 2, T, device="cuda").view(-1, 1)
    v[T - 5:, 3] = 3e38
    q, k, v = q.bfloat16(), k.bfloat16(), v.bfloat16()
    cu = torch.tensor([0, T], device="cuda", dtype=torch.int32)
    got = K.flash_attn_varlen(q, k, v, cu, T, H, H, D, False).double().view(T, H, D).transpose(0, 1)
    r = lambda t: t.double().view(T, H, D).transpose(0, 1)  # noqa: E731
    p = torch.softmax(r(q) @ r(k).transpose(1, 2) * D ** -0.5, -1)
    want, mag = p @ r(v), p @ r(v).abs()
    assert ((got - want).abs() <= 2.0 ** -8 * (mag + want.abs()) * 1.01 + 2.0 ** -13).all()
