"""The encoder's kernels at the edges of their rows and tiles, against 64-bit results."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu

from docagents_amd.ops import kernels as K  # noqa: E402

DEV = "cuda"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("M,D", [(1, 8), (3, 384), (5, 512), (1023, 520), (1027, 768), (9001, 1024), (2, 1032), (1030, 2048),
                                 (7, 2056), (1025, 4096)])
def test_layernorm_rows(M, D, dtype):
    """A wave per row up to 2048 columns (lanes past the end, waves that walk several rows), a workgroup beyond; with
    a residual and without a bias; the row-quantised copy."""
    torch.manual_seed(M + D)
    f16 = dtype == torch.float16
    x, r, g, b = ((torch.randn(*s, device=DEV) * 2 + 0.5).to(dtype) for s in ((M, D), (M, D), (D,), (D,)))
    ln = K.layernorm_f16 if f16 else K.layernorm
    # half a unit in the last place of the result's type, and fp32 sums of D terms before it
    ulp = 2.0 ** -11 if f16 else 2.0 ** -8
    for resid, bias in ((None, b), (r, b)) if f16 else ((None, b), (r, b), (r, None)):
        want = torch.nn.functional.layer_norm(x.double() + (0 if resid is None else resid.double()), (D,), g.double(),
                                              None if bias is None else bias.double(), 1e-5)
        got = ln(x, g, bias, 1e-5, resid=resid)
        assert bool(((got.double() - want).abs() <= ulp * want.abs() + 1e-5 * (1 + want.abs())).all())
    if not f16 and D % 16 == 0:
        y, yq, ys = K.layernorm(x, g, b, 1e-5, fp8_out=True)
        rq, rs = K.quant_fp8(y)
        assert torch.equal(y, K.layernorm(x, g, b, 1e-5))
        # both quantise a row; this copy before the rounding to bf16, that one after it
        assert torch.allclose(ys, rs, rtol=2.0 ** -8)
        err = (yq.float() * ys[:, None] - y.float()).abs()
        assert bool((err <= 2.0 ** -4 * y.float().abs() * (1 + 2.0 ** -3) + ys[:, None] * 2.0 ** -9).all())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,D", [(1, 384), (33, 768), (1029, 1024), (5, 1536), (6, 2304)])
def test_bert_embed_rows(T, D, dtype):
    torch.manual_seed(T)
    word, pos, typ, g, b = ((torch.randn(*s, device=DEV)).to(dtype) for s in ((97, D), (40, D), (2, D), (D,), (D,)))
    ids, ps, ty = (torch.randint(0, n, (T,), device=DEV, dtype=torch.int32) for n in (97, 40, 2))
    f = K.bert_embed_ln_f16 if dtype == torch.float16 else K.bert_embed_ln
    ulp = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8
    for types in (None, ty):
        e = word.double()[ids.long()] + pos.double()[ps.long()] + typ.double()[0 if types is None else types.long()]
        want = torch.nn.functional.layer_norm(e, (D,), g.double(), b.double(), 1e-12)
        got = f(ids, ps, types, word, pos, typ, g, b, 1e-12)
        assert bool(((got.double() - want).abs() <= ulp * want.abs() + 1e-5 * (1 + want.abs())).all())


@pytest.mark.parametrize("dtype,M,Kd", [(torch.bfloat16, 16, 256), (torch.bfloat16, 300, 128), (torch.float16, 300, 128)])
def test_gelu_epilogue(dtype, M, Kd):
    """The activation alone (an identity product): over its curve, its tails, infinities and NaN."""
    w = torch.eye(Kd, device=DEV).to(dtype)
    x = torch.linspace(-9, 9, M * Kd, device=DEV).view(M, Kd).to(dtype)
    zero = torch.zeros(Kd, dtype=dtype, device=DEV)
    f = K.gemm_f16 if dtype == torch.float16 else K.gemm
    got = f(x, w, bias=zero, epi=K.EPI_GELU)
    want = torch.nn.functional.gelu(x.double())
    # half a unit in the last place of the result's type; 2e-6 relative and 2.4e-7 absolute before the rounding
    ulp, tiny = (2.0 ** -11, 2.0 ** -25) if dtype == torch.float16 else (2.0 ** -8, 0.0)
    assert bool(((got.double() - want).abs() <= (ulp + 2e-6) * want.abs() + 2.4e-7 + tiny).all())
    big = 6e4 if dtype == torch.float16 else 3e38
    bias = zero.clone()
    bias[:5] = torch.tensor([math.inf, -math.inf, math.nan, big, -big])
    got = f(torch.zeros_like(x), w, bias=bias, epi=K.EPI_GELU)[0]
    assert got[0] == math.inf and bool(got[2].isnan()) and got[3] == bias[3] and got[4] == 0 and bool((got[5:] == 0).all())
