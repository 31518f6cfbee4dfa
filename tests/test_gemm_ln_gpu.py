"""Encoder products of up to 64 rows with the LayerNorms inside, against 64-bit arithmetic at the edges of their ranges."""
import pytest
import torch

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K

# (rows, hidden, ffn): each row tile's edges; one unit of K a wave, fewer units than waves that store, two groups of units
@pytest.mark.parametrize("M,h,f", [(1, 768, 3072), (16, 128, 256), (17, 384, 1536), (32, 1024, 4096), (33, 768, 3072),
                                   (64, 64, 64), (64, 1024, 4096), (20, 960, 64 * 33)])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_gemm_ln(M, h, f, dt):
    U = 2.0 ** -8 if dt == torch.bfloat16 else 2.0 ** -11  # a rounding of the type
    g = torch.Generator(device="cuda").manual_seed(M + h)
    r = lambda *s: torch.randn(*s, device="cuda", generator=g)  # noqa: E731
    a, resid = r(M, h).to(dt), (3 * r(M, h) + 40).to(dt)  # a mean far from zero: no cancellation allowed
    wo, w1, w2, wq = (r(h, h) * h ** -0.5).to(dt), (r(f, h) * h ** -0.5).to(dt), (r(h, f) * f ** -0.5).to(dt), \
        (r(3 * h, h) * h ** -0.5).to(dt)
    bo, b1, bq, lg, lb = (r(n).to(dt) for n in (h, f, 3 * h, h, h))
    st, st2 = torch.full((2, 64, 64, 2), float("nan"), device="cuda")  # (what a part does not write is not read)
    d = lambda t: t.double()  # noqa: E731

    def close(got, ref, a_, w_, slack=0.0):
        # one rounding of the result, fp32 sums (with a margin), and what the operands' own roundings allow
        tol = U * ref.abs() + 8 * w_.shape[1] * 2.0 ** -24 * (d(a_).abs() @ d(w_).abs().T).max() + slack
        assert ((d(got) - ref).abs() <= tol).all(), float(((d(got) - ref).abs() / tol).max())

    y = K.gemm_ln(a, wo, bo, K.EPI_RESID, resid=resid, st_out=st)
    close(y, d(a) @ d(wo).T + d(bo) + d(resid), a, wo)
    n = torch.nn.functional.layer_norm(d(y), (h,), d(lg), d(lb), 1e-12)
    norm = (st, lg, lb, 1e-12)
    nb = n.to(dt)  # differs from the kernel's by an ulp where fp32 rounds the other way: an operand's rounding each
    def flips(w):
        return (U * nb.double().abs()).square() @ d(w).square().T  # (their sum's variance, if all of them did)
    z = K.gemm_ln(y, wq, bq, norm=norm)
    close(z, d(nb) @ d(wq).T + d(bq), nb, wq, flips(wq).sqrt())
    u = d(nb) @ d(w1).T + d(b1)
    x = K.gemm_ln(y, w1, b1, K.EPI_GELU, norm=norm)
    close(x, torch.nn.functional.gelu(u), nb, w1, 1.2 * flips(w1).sqrt())
    x2 = K.gemm_ln(x, w2, bo, K.EPI_RESID, norm=norm, resid=y, st_out=st2)
    close(x2, d(x) @ d(w2).T + d(bo) + d(nb), x, w2, U * n.abs())
    # the statistics: each part's own, of the stored values
    parts = d(x2).view(M, h // 16, 16)
    mean = parts.mean(-1)
    assert torch.allclose(d(st2[:M, :h // 16, 0]), mean, rtol=0, atol=2.0 ** -22 * float(parts.abs().max()))
    dev = (parts - mean[..., None]).square().sum(-1)
    assert torch.allclose(d(st2[:M, :h // 16, 1]), dev, rtol=1e-5, atol=1e-5 * float(dev.max()))


def test_what_the_product_refuses():
    """Operands that the kernel would read at other places than the caller's."""
    M, h = 8, 128
    t = lambda *s: torch.ones(s, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    a, w, b, v = t(M, h), t(h, h), t(h), t(h)
    st, st2 = torch.zeros((2, 64, 64, 2), device="cuda")
    K.gemm_ln(a, w, b, norm=(st, v, v, 1e-5))
    for bias, norm in [(t(2 * h)[::2], None), (b, (st, t(2 * h)[::2], v, 1e-5)), (b, (st, v, t(h // 2), 1e-5)),
                       (b, (st, v.float(), v, 1e-5)), (b, (st.cpu(), v, v, 1e-5)), (b, (st[:32], v, v, 1e-5))]:
        with pytest.raises(ValueError):
            K.gemm_ln(a, w, bias, norm=norm)
        with pytest.raises(ValueError):
            K.gemm_ln(a, w, bias, K.EPI_RESID, norm=norm, resid=a, st_out=st2)
    with pytest.raises(ValueError):
        K.gemm_ln(a, w, b, K.EPI_RESID, resid=a, st_out=st2[:, :32])


@pytest.mark.parametrize("h,f,one", [(1024, 4096, False), (1024, 2048, True), (768, 3072, True)])
def test_which_short_texts_take_it(h, f, one, monkeypatch):
    """Up to 64 tokens do, but one token of a wide encoder has matrix-vector products; both agree."""
    from docagents_amd.models.bert import BertEncoder
    from docagents_amd.models.configs import EncoderConfig
    enc = BertEncoder(EncoderConfig("e", vocab=100, hidden=h, layers=2, heads=h // 64, ffn=f), "cuda")
    calls, real = [], K.gemm_ln
    monkeypatch.setattr(K, "gemm_ln", lambda *a, **kw: calls.append(1) or real(*a, **kw))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    for T, few in ((1, one), (2, True), (64, True), (65, False)):
        calls.clear()
        args = i32([7] * T), i32(list(range(T))), i32([0, T]), T
        got = enc.forward(*args).double()
        assert len(calls) == (8 if few else 0)
        if T == 1:
            with monkeypatch.context() as m:
                m.setattr(BertEncoder, "_one_row", lambda self, rows: one)  # the other way
                if one:
                    m.setattr(K, "gemm_ln_fit", lambda *a: False)
                want = enc.forward(*args).double()
            # bf16 roundings of two layers: each of about a dozen adds 2^-9 of values of about 1
            assert float((got - want).norm() / want.norm()) < 12 * 2.0 ** -9
