"""Attention of one text inside the encoder product behind it (up to 32 or 64 rows), against 64-bit arithmetic."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K


def attend(qkv, heads, cu):
    """fp64 attention output, and the sums of weights times |v| that its roundings are relative to."""
    M, h = qkv.shape[0], qkv.shape[1] // 3
    q, k, v = (t.reshape(M, heads, -1).transpose(0, 1) for t in qkv.double().split(h, 1))
    o, m = torch.zeros(2, heads, M, h // heads, dtype=torch.float64, device=qkv.device)
    for a, b in zip(cu, cu[1:]):
        p = ((q[:, a:b] @ k[:, a:b].transpose(1, 2).contiguous()) / math.sqrt(h // heads)).softmax(-1)
        o[:, a:b], m[:, a:b] = p @ v[:, a:b], p @ v[:, a:b].abs()
    return (t.transpose(0, 1).reshape(M, h) for t in (o, m))


# (rows, hidden, heads, text): one row; edges of the 16-row blocks; rows before the text and past it; one unit of K, 12, 13 and 16
@pytest.mark.parametrize("M,h,heads,cu", [
    (1, 768, 12, [0, 1]), (16, 128, 4, [0, 16]), (17, 64, 1, [0, 17]), (32, 768, 12, [0, 32]), (31, 384, 12, [0, 31]),
    (32, 768, 24, [0, 21]), (32, 384, 6, [5, 19]), (32, 512, 8, [17, 18]), (9, 64, 2, [0, 9]), (32, 1024, 16, [0, 32]), (19, 832, 13, [0, 17]), (17, 1024, 32, [0, 17]), (64, 384, 12, [0, 64]), (33, 384, 6, [0, 33]),
    (50, 128, 2, [3, 47]), (16, 128, 2, [0, 5])])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_attention_inside(M, h, heads, cu, dt):
    if dt == torch.float16 and h == 32 * heads:
        heads //= 2  # (heads of 32: bf16 only)
    U = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11
    g = torch.Generator(device="cuda").manual_seed(M + h)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    wide = torch.full((M, 3 * h + 8), float("nan"), device="cuda", dtype=dt)  # (rows further apart than they are long)
    qkv = wide[:, :3 * h]
    qkv[cu[0]:cu[1]] = (1.5 * r(cu[1] - cu[0], 3 * h)).to(dt)  # (and NaN elsewhere)
    resid, w, b = r(M, h).to(dt), (r(h, h) * h ** -0.5).to(dt), r(h).to(dt)
    st = torch.full((64, 64, 2), float("nan"), device="cuda")
    c = torch.tensor(cu, dtype=torch.int32, device="cuda")
    got = K.gemm_ln(qkv, w, b, K.EPI_RESID, resid=resid, st_out=st, attn=(heads, c))[cu[0]:cu[1]]
    o, m = attend(qkv, heads, cu)
    o, m, resid = (t[cu[0]:cu[1]] for t in (o, m, resid))
    ref = o @ w.double().T + b.double() + resid.double()
    # weights and output are rounded once each (2 U / 2 of m); as independent errors through the product, 6 deviations;
    # the result's own rounding and the fp32 sums
    tol = U * ref.abs() + 6 * ((U * m).square() @ w.double().square().T).sqrt() + 8 * h * 2.0 ** -24 * (o.abs() @ w.double().abs().T).max()
    assert ((got.double() - ref).abs() <= tol + 1e-6).all(), float(((got.double() - ref).abs() / (tol + 1e-6)).max())
    y = got.double().view(-1, h // 16, 16)
    assert torch.allclose(st[cu[0]:cu[1], :h // 16, 0].double(), y.mean(-1), rtol=0, atol=2.0 ** -22 * float(y.abs().max()))


def test_what_attention_refuses():
    t = lambda *s: torch.ones(s, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    st, i32 = torch.zeros((64, 64, 2), device="cuda"), lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")
    run = lambda M, h, heads, cu: K.gemm_ln(t(M, 3 * h), t(h, h), t(h), K.EPI_RESID, resid=t(M, h), st_out=st, attn=(heads, cu))  # noqa: E731
    run(8, 128, 2, i32([0, 8]))
    for M, h, heads, cu in [(33, 448, 7, i32([0, 33])), (65, 128, 2, i32([0, 65])), (8, 1088, 17, i32([0, 8])), (8, 128, 1, i32([0, 8])),
                            (8, 128, 2, i32([0, 4, 8])), (8, 128, 2, i32([0, 8]).long()), (8, 128, 2, i32([0, 8]).cpu())]:
        with pytest.raises(ValueError):
            run(M, h, heads, cu)
