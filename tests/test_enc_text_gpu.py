"""A short text's encoder layers in one launch, against 64-bit arithmetic and the launches one by one."""
import threading

import pytest
import torch
import torch.nn.functional as F

from docagents_amd.models.bert import BertEncoder
from docagents_amd.models.configs import EncoderConfig

pytestmark = pytest.mark.gpu

if torch.cuda.is_available():
    from docagents_amd.ops import kernels as K


def make(h, f, heads, layers, dt, seed=0):
    g = torch.Generator(device="cuda").manual_seed(h + f + layers + seed)
    r = lambda *s, a=1.0: (torch.randn(*s, device="cuda", generator=g) * a).to(dt)  # noqa: E731
    out = []
    for _ in range(layers):
        out.append({"wqkv": r(3 * h, h, a=1.5 * h ** -0.5), "bqkv": r(3 * h, a=0.2), "wo": r(h, h, a=h ** -0.5), "bo": r(h, a=0.2),
                    "w1": r(f, h, a=h ** -0.5), "b1": r(f, a=0.2), "w2": r(h, f, a=f ** -0.5), "b2": r(h, a=0.2),
                    **{f"ln{i}_{n}": (r(h, a=0.1).float() + (n == "g")).to(dt) for i in (1, 2) for n in "gb"}})
    return out, r


def in64(x, layers, cu, heads, eps):
    """(the last sum in 64 bits)"""
    x, (a, b), h = x.double(), cu, x.shape[1]
    d = lambda t: t.double()  # noqa: E731
    for i, L in enumerate(layers):
        q, k, v = (t.reshape(-1, heads, h // heads).transpose(0, 1) for t in (x[a:b] @ d(L["wqkv"]).T + d(L["bqkv"])).split(h, 1))
        p = ((q @ k.transpose(1, 2).contiguous()) * (h // heads) ** -0.5).softmax(-1)
        o = torch.zeros_like(x)
        o[a:b] = (p @ v).transpose(0, 1).reshape(-1, h)
        y = F.layer_norm(x + o @ d(L["wo"]).T + d(L["bo"]), (h,), d(L["ln1_g"]), d(L["ln1_b"]), eps)
        s = y + F.gelu(y @ d(L["w1"]).T + d(L["b1"])) @ d(L["w2"]).T + d(L["b2"])
        x = F.layer_norm(s, (h,), d(L["ln2_g"]), d(L["ln2_b"]), eps)
    return s


def apart(x, layers, cu, heads, eps):
    """(the launches one by one)"""
    st1, st2 = torch.empty((2, 64, 64, 2), dtype=torch.float32, device="cuda")
    norm, h, attn = None, x.shape[1], K.flash_attn_f16 if x.dtype == torch.float16 else K.flash_attn_varlen
    for L in layers:
        qkv, inside = K.gemm_ln(x, L["wqkv"], L["bqkv"], norm=norm), K.attn_ln_fit(x.shape[0], h, heads, 1, x.dtype == torch.float16)
        a = qkv if inside else attn(qkv[:, :h], qkv[:, h:2 * h], qkv[:, 2 * h:], cu, x.shape[0], heads, heads, h // heads, causal=False)
        y = K.gemm_ln(a, L["wo"], L["bo"], K.EPI_RESID, norm=norm, resid=x, st_out=st1, attn=(heads, cu) if inside else None)
        norm = (st1, L["ln1_g"], L["ln1_b"], eps)
        x = K.gemm_ln(K.gemm_ln(y, L["w1"], L["b1"], K.EPI_GELU, norm=norm), L["w2"], L["b2"], K.EPI_RESID, norm=norm, resid=y, st_out=st2)
        norm = (st2, L["ln2_g"], L["ln2_b"], eps)
    return x


# one row; the edges of the row blocks; rows outside the text; units of K fewer than waves, as many, and 2 to 4 a wave; the most layers
@pytest.mark.parametrize("M,h,f,heads,layers,cu", [
    (1, 64, 64, 1, 4, [0, 1]), (16, 384, 1536, 12, 6, [0, 16]), (17, 384, 1536, 6, 5, [0, 17]), (32, 768, 3072, 12, 12, [0, 21]),
    (16, 768, 3072, 12, 12, [0, 7]), (31, 1024, 4096, 16, 4, [3, 29]), (32, 1024, 4096, 32, 24, [0, 32]), (9, 832, 1088, 13, 4, [0, 9]),
    (32, 128, 2112, 2, 32, [17, 18]), (2, 512, 4032, 8, 4, [0, 2]), (33, 384, 1536, 12, 6, [0, 33]), (64, 1024, 4096, 16, 6, [0, 64]),
    (48, 768, 3072, 24, 5, [0, 48]), (49, 832, 1088, 13, 4, [0, 49]), (64, 768, 3072, 12, 6, [0, 41]), (63, 64, 4096, 1, 4, [20, 50])])
@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
def test_layers(M, h, f, heads, layers, cu, dt):
    if dt == torch.float16 and h == 32 * heads:
        heads //= 2  # (heads of 32: bf16 only)
    L, r = make(h, f, heads, layers, dt)
    c = torch.tensor(cu, dtype=torch.int32, device="cuda")
    assert K.enc_text_fits(M, h, f, layers, heads, 1, dt == torch.float16)
    for seed in range(3):  # (new activations in the same buffers: nothing of the launch before)
        x = r(M, h)
        got, one = (fn(x, L, c, heads, 1e-12)[cu[0]:cu[1]].double() for fn in (K.enc_text, apart))
        ref = in64(x, L, cu, heads, 1e-12)[cu[0]:cu[1]]
        e, e1 = (float((t - ref).norm() / ref.norm()) for t in (got, one))
        # with attention inside the products, one by one: the same sums in the same order, and in bf16 the same bits (in fp16 the
        # compiler rounds some norms within the fma, and which ones differs from kernel to kernel). Where it is a launch of its
        # own the sums are in another order: the same roundings in the same places, errors of one size. A layer rounds about eight
        # times, by 2^-9 (2^-12) of values of about one each, which add as independent ones over the layers
        u = 2.0 ** -9 if dt == torch.bfloat16 else 2.0 ** -12
        assert torch.equal(got, one) or dt == torch.float16 or not K.attn_ln_fit(M, h, heads, 1)
        assert e < 1.25 * e1 + u and e < 4 * (8 * layers) ** 0.5 * u, (e, e1)
        for _ in range(10):
            again = K.enc_text(x, L, c, heads, 1e-12)
            assert torch.equal(again[cu[0]:cu[1]].double(), got) and not bool(again[cu[1]:].any())  # (rows behind the text: zeros)


@pytest.mark.parametrize("T", [16, 32, 64])
def test_replays(T):
    """Captured: each replay has its own input's result, with eager launches of the same stream between them."""
    L, r = make(768, 3072, 12, 12, torch.bfloat16)
    cu, x = torch.tensor([0, T], dtype=torch.int32, device="cuda"), r(T, 768)
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        K.enc_text(x, L, cu, 12, 1e-12)
        s.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            out = K.enc_text(x, L, cu, 12, 1e-12)
        for _ in range(6):
            x.copy_(r(T, 768))
            want = K.enc_text(x, L, cu, 12, 1e-12)
            g.replay()
            assert torch.equal(out, want)
            assert torch.equal(K.enc_text(x, L, cu, 12, 1e-12), want)


def test_which_texts_take_it(monkeypatch):
    """One text of up to 64 rows from ENC_TEXT_MIN_LAYERS layers on; others as before."""
    calls, real = [], K.enc_text
    monkeypatch.setattr(K, "enc_text", lambda *a: calls.append(1) or real(*a))
    i32 = lambda v: torch.tensor(v, dtype=torch.int32, device="cuda")  # noqa: E731
    for layers in (K.ENC_TEXT_MIN_LAYERS - 1, K.ENC_TEXT_MIN_LAYERS):
        enc = BertEncoder(EncoderConfig("e", vocab=100, hidden=128, layers=layers, heads=2, ffn=256), "cuda")
        for T, cu in ((64, [0, 64]), (65, [0, 65]), (32, [0, 16, 32])):
            calls.clear()
            enc.forward(i32([7] * T), i32(list(range(T))), i32(cu), T)
            assert len(calls) == (layers >= K.ENC_TEXT_MIN_LAYERS and T == 64 and len(cu) == 2)


@pytest.mark.parametrize("h,f,heads,pooling,dtype", [(128, 256, 4, "cls", "bf16"), (768, 3072, 12, "mean", "bf16"), (1024, 4096, 16, "cls", "fp16"),
                                                     (576, 1088, 9, "mean", "fp16")])
def test_whole_text(h, f, heads, pooling, dtype):
    """A question in three launches (embeddings; layers; norm and pooling) against the launches one by one; a result stays as it is when
    the next question runs, on whichever stream."""
    enc = BertEncoder(EncoderConfig("e", vocab=500, hidden=h, layers=5, heads=heads, ffn=f, pooling=pooling), "cuda", dtype=dtype)
    g = torch.Generator().manual_seed(h)
    for L in enc.w["layers"]:
        for k in ("wqkv", "wo", "w1", "w2"):
            L[k].mul_(3)  # (layers that matter beside the stream)
    enc.prepare_graphs()
    assert set(enc._g) == {128}
    other, had = torch.cuda.Stream(), []
    for n in (1, 2, 15, 16, 17, 21, 31, 32, 33, 7, 48, 64, 65, 3):
        seq = torch.randint(5, 500, (n,), generator=g).tolist()
        with torch.cuda.stream(other if n % 2 else torch.cuda.default_stream()):
            v = enc.encode_one(seq)
        torch.cuda.synchronize()
        ids, pos, cu = (torch.tensor(t, dtype=torch.int32, device="cuda") for t in (seq, list(range(n)), [0, n]))
        with pytest.MonkeyPatch.context() as m:
            m.setattr(K, "enc_text_fits", lambda *a: False)
            m.setattr(BertEncoder, "_one_row", lambda self, rows: False)
            want = enc._pool(enc.forward(ids, pos, cu, n), cu)
        assert v.shape == want.shape and v.dtype == torch.float32
        assert torch.equal(v, want) or dtype == "fp16" or not K.attn_ln_fit(n, h, heads, 1)
        # roundings of the type, about 8 a layer, add as independent ones in both
        u = 2.0 ** -9 if dtype == "bf16" else 2.0 ** -12
        assert float((v - want).norm()) < 2 * (8 * 5) ** 0.5 * u and abs(float(v.norm()) - 1) < 1e-5
        had.append((v, v.clone()))
    assert all(torch.equal(a, b) for a, b in had)


def test_what_it_refuses():
    """Shapes beyond the kernel's go the other way; wrong operands raise as the products one by one do."""
    for M, h, f, layers, heads, texts, f16 in [(65, 768, 3072, 12, 12, 1, False), (0, 768, 3072, 12, 12, 1, False), (8, 1088, 3072, 12, 17, 1, False),
                                               (8, 768, 4160, 12, 12, 1, False), (8, 768, 3072, 33, 12, 1, False), (8, 768, 3072, 12, 12, 2, False),
                                               (8, 768, 3072, 12, 24, 1, True), (8, 768, 3072, 12, 8, 1, False), (8, 720, 3072, 12, 12, 1, False)]:
        assert not K.enc_text_fits(M, h, f, layers, heads, texts, f16)
    L, r = make(128, 256, 2, 4, torch.bfloat16)
    cu, x = torch.tensor([0, 8], dtype=torch.int32, device="cuda"), r(8, 128)
    K.enc_text(x, L, cu, 2, 1e-12)
    for bad in ({"wo": L[0]["wo"].half()}, {"wo": L[0]["wo"].cpu()}, {"w1": L[0]["w1"][:, ::2]}, {"bqkv": L[0]["bo"]}):
        with pytest.raises(ValueError):
            K.enc_text(x, [{**L[0], **bad}, *L[1:]], cu, 2, 1e-12)
    for args in ((x.t().contiguous().t(), cu), (x, cu.long()), (x, cu.cpu()), (r(65, 128), cu)):
        with pytest.raises(ValueError):
            K.enc_text(args[0], L, args[1], 2, 1e-12)


def test_beside_one_another():
    """Texts on several streams at once, beside products that fill the chip: each takes its tasks in order on whatever room it gets."""
    L, r = make(768, 3072, 12, 6, torch.bfloat16)
    xs, cu = [r(n, 768) for n in (16, 32, 48, 64)], [torch.tensor([0, n], dtype=torch.int32, device="cuda") for n in (16, 32, 48, 64)]
    want = [K.enc_text(x, L, c, 12, 1e-12) for x, c in zip(xs, cu)]
    a, b = r(4096, 4096), r(8192, 4096)
    streams = [torch.cuda.Stream() for _ in range(5)]
    torch.cuda.synchronize()
    got = [[] for _ in xs]
    for _ in range(8):
        with torch.cuda.stream(streams[4]):
            K.gemm(a, b)
        for i, (x, c) in enumerate(zip(xs, cu)):
            with torch.cuda.stream(streams[i]):
                got[i].append(K.enc_text(x, L, c, 12, 1e-12))
    torch.cuda.synchronize()
    assert all(torch.equal(g, w) for gs, w in zip(got, want) for g in gs)


def test_a_wait_that_runs_out_is_told(monkeypatch):
    """A wait that ends before its words are there (here after one reading) leaves NaNs, and the next check or launch raises; later
    texts are as ever. Waits that do not end early say nothing, nor do NaNs that the input makes."""
    enc = BertEncoder(EncoderConfig("e", vocab=100, hidden=768, layers=12, heads=12, ffn=3072), "cuda")
    enc.prepare_graphs()
    seq = list(range(5, 26))
    want = enc.encode_one(seq)
    torch.cuda.synchronize()
    enc.check()
    for call in (enc.encode_one, lambda s: enc.encode_packed([s])):
        with monkeypatch.context() as m:
            m.setattr(K, "TEXT_POLLS", 1)
            v = call(seq)
            torch.cuda.synchronize()
        assert bool(v.isnan().any())
        with pytest.raises(K.KernelError):
            enc.check()
        enc.check()
        assert torch.equal(enc.encode_one(seq), want)
    with monkeypatch.context() as m:
        m.setattr(K, "TEXT_POLLS", 1)
        enc.encode_one(seq)
        torch.cuda.synchronize()
    with pytest.raises(K.KernelError):  # (who did not ask hears of it at the next text)
        enc.encode_one(seq)
    assert torch.equal(enc.encode_one(seq), want)


def test_each_thread_is_told():
    """Two threads with texts of one encoder: who asks first does not keep it from the other."""
    waits, ask = K.TextWaits(), [threading.Event() for _ in range(2)]
    told = [[], []]

    def thread(i):
        waits.check()
        ask[i].set()
        ran_out.wait(10)
        for _ in range(2):
            try:
                waits.check()
            except K.KernelError:
                told[i].append(1)
    ran_out, threads = threading.Event(), [threading.Thread(target=thread, args=(i,)) for i in range(2)]
    for t in threads:
        t.start()
    for a in ask:
        assert a.wait(10)
    waits._word[0] = 1
    ran_out.set()
    for t in threads:
        t.join()
    assert told == [[1], [1]]


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("where", ["x", "bqkv", "bo", "b1", "b2", "ln1_b"])
def test_words_of_set_bits(where, dt):
    """NaNs of all bits set, as words that are not there yet have them, are values like others: no wait waits for them."""
    L, r = make(128, 256, 2, 4, dt)
    x, cu, waits = r(17, 128), torch.tensor([0, 17], dtype=torch.int32, device="cuda"), K.TextWaits()
    t = x[3] if where == "x" else L[1][where]
    t.view(torch.int16)[:] = -1
    a, b = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    a.record()
    got = K.enc_text(x, L, cu, 2, 1e-12, waits)
    b.record()
    torch.cuda.synchronize()
    waits.check()
    assert a.elapsed_time(b) < 1000 and bool(got[3].isnan().all())


def shifted(t):
    """The same values two bytes behind a 16-B address."""
    out = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)[1:].view(t.shape).copy_(t)
    assert out.data_ptr() % 16 == 2
    return out


@pytest.mark.parametrize("dt", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("name", ["bqkv", "bo", "b1", "b2", "ln1_g", "ln1_b", "ln2_g", "ln2_b"])
def test_vectors_at_any_address(name, dt):
    """Vectors of the layers may lie anywhere, as the products one by one take them."""
    L, r = make(320, 640, 5, 4, dt)
    cu, x = torch.tensor([0, 19], dtype=torch.int32, device="cuda"), r(19, 320)
    assert torch.equal(K.enc_text(x, [{**one, name: shifted(one[name])} for one in L], cu, 5, 1e-12), K.enc_text(x, L, cu, 5, 1e-12))


@pytest.mark.parametrize("dtype", ["bf16", "fp16"])
@pytest.mark.parametrize("pooling", ["cls", "mean"])
def test_embeddings_at_any_address(dtype, pooling):
    """So may the embeddings' tables, their norm and the last one."""
    enc = BertEncoder(EncoderConfig("e", vocab=50, hidden=320, layers=4, heads=5, ffn=640, pooling=pooling), "cuda", dtype=dtype)
    w = {k: shifted(v) if k != "layers" else v[:-1] + [{**v[-1], **{n: shifted(v[-1][n]) for n in ("ln2_g", "ln2_b")}}] for k, v in enc.w.items()}
    seq = [3, 49, 7, 7, 20]
    tokens = torch.tensor([*seq, *range(5), 0, 5], dtype=torch.int32, device="cuda")
    a, b = (K.enc_text_pooled(K.TextPlan(t, 5, 1e-12), tokens, enc._pool_mode) for t in (w, enc.w))
    assert torch.equal(a, b) and torch.equal(a, enc.encode_one(seq))
