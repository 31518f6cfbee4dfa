"""The work that users of this framework have it do, as cases that can be timed and checked: embeddings of questions
and of chunks, vector search, prompt prefill and decode steps, at the sizes of the framework's own configurations,
benchmark and tests.

A case is a dict of plain values. ``prepare`` makes what a program holds before the call (weights, caches, an index,
captured decode graphs, token ids), ``run`` is one pass through the public entry points, ``exact`` the same results
in 64 bits without the framework's kernels.
"""
from __future__ import annotations

import math
import random

import numpy as np
import torch
import torch.nn.functional as F

from docagents_amd.engine.generator import Generator
from docagents_amd.index import make_index
from docagents_amd.models import make_decoder
from docagents_amd.models.bert import BertEncoder
from docagents_amd.models.configs import (ChannelDelta, GatedRecurrence, HybridConfig, LatentAttention, SigmoidAttention,
                                          decoder_config, encoder_config)
from docagents_amd.models.hybrid import tensor_shapes
from docagents_amd.models.llama import DecodeState
from docagents_amd.ops.reference import interleave_gate_up

DEV = "cuda"
EXACT_TOKENS = 24_000  # of a decoder of mixed layers: its recurrences are walked token by token
STATES = ("rec", "ssm", "delta")  # the recurrent states of mixed layers


def listed() -> list[dict]:
    return [
        # a question on its way to the index: latency of one short text
        {"name": "embed_question", "kind": "embed", "arch": "bge-base", "dtype": "bf16", "texts": 1, "min": 21, "max": 21},
        # ingest: a batch of 400-word chunks with a short last one per document, the fp16 embedder
        {"name": "embed_chunks", "kind": "embed", "arch": "bge-large", "dtype": "fp16", "texts": 80, "min": 61, "max": 512},
        # one question over the documents its user named
        {"name": "search_documents", "kind": "search", "index": "flat", "rows": 100_000, "dim": 768, "queries": 1, "k": 5,
         "docs": 8},
        # a batch of questions over a whole shard (10 M chunks on 8 GPUs)
        {"name": "search_all", "kind": "search", "index": "flat", "rows": 1_250_000, "dim": 1024, "queries": 128, "k": 5,
         "docs": 0},
        # questions against the inverted lists
        {"name": "search_lists", "kind": "search", "index": "ivfflat", "rows": 400_000, "dim": 768, "queries": 24, "k": 5,
         "docs": 0, "lists": 512, "probes": 8},
        # prompts of retrieved context behind the system prompt that all of them share
        {"name": "prefill_answers", "kind": "prefill", "arch": "phi3-mini", "dtype": "bf16", "prompts": 3, "min": 1811,
         "max": 2679, "head": 256},
        # decoding one answer: latency
        {"name": "decode_one", "kind": "decode", "arch": "phi3-mini", "dtype": "bf16", "rows": 1, "min": 2935, "max": 2935},
        # decoding a full batch, grouped-query attention
        {"name": "decode_batch", "kind": "decode", "arch": "llama3-8b", "dtype": "bf16", "rows": 64, "min": 900,
         "max": 3100},
        # the decoders of mixed layers: recurrence, scan and sigmoid attention
        {"name": "prefill_recurrent", "kind": "prefill", "arch": "binupel-9b", "dtype": "bf16", "prompts": 2, "min": 1365,
         "max": 2048, "head": 0},
        {"name": "decode_recurrent", "kind": "decode", "arch": "binupel-9b", "dtype": "bf16", "rows": 16, "min": 300,
         "max": 1500},
        # delta rule and latent attention
        {"name": "prefill_delta", "kind": "prefill", "arch": "zamitar-8b", "dtype": "bf16", "prompts": 5, "min": 333,
         "max": 2048, "head": 0},
        {"name": "decode_delta", "kind": "decode", "arch": "zamitar-8b", "dtype": "bf16", "rows": 64, "min": 64, "max": 500},
    ]


def _log(rng: random.Random, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng: random.Random) -> dict:
    kind = rng.choice(["embed", "embed", "search", "search", "prefill", "prefill", "prefill", "decode", "decode", "decode"])
    if kind == "embed":
        arch = rng.choice(["bge-small", "bge-base", "bge-large", "e5-base", "e5-large"])
        hi = _log(rng, 5, 512)
        dtype = rng.choice(["bf16", "bf16", "fp8"] if arch == "bge-small" else ["bf16", "bf16", "fp16", "fp8"])
        return {"kind": kind, "arch": arch, "dtype": dtype,
                "texts": _log(rng, 1, 80), "min": rng.randint(max(3, hi // 8), hi), "max": hi}
    if kind == "search":
        ivf = rng.random() < 0.4
        c = {"kind": kind, "index": "ivfflat" if ivf else "flat", "rows": _log(rng, 20_000, 1_000_000),
             "dim": rng.choice([384, 768, 1024]), "queries": _log(rng, 1, 128), "k": rng.randint(1, 20),
             "docs": rng.choice([0, 0, _log(rng, 1, 64)])}
        return {**c, "lists": 8 * rng.randint(13, 64), "probes": _log(rng, 1, 24)} if ivf else c
    arch = rng.choice(["phi3-mini", "llama3-8b", "binupel-9b", "zamitar-8b"])
    mixed = arch in ("binupel-9b", "zamitar-8b")
    if kind == "prefill":
        # (the fp32 precision of mixed layers is for checking: short prompts)
        dtype = "fp32" if mixed and rng.random() < 0.15 else "bf16"
        n = rng.randint(1, 4)
        hi = _log(rng, 24, 256 if dtype == "fp32" else min(2048, 6000 // n))
        return {"kind": kind, "arch": arch, "dtype": dtype, "prompts": n, "min": rng.randint(max(9, hi // 4), hi),
                "max": hi, "head": 0 if mixed else rng.choice([0, 64, 320])}
    rows = _log(rng, 1, 40 if arch == "phi3-mini" else 64)  # (a phi3-mini slot takes 1.6 GB)
    hi = _log(rng, 64, 400 if mixed else 3000)
    return {"kind": kind, "arch": arch, "dtype": "bf16", "rows": rows, "min": rng.randint(max(9, hi // 4), hi), "max": hi}


# ---------------------------------------------------------------------------------------- inputs
def _lens(case: dict) -> list[int]:
    """The case's sequence lengths: its longest, and others spread over its range."""
    n, lo, hi = case.get("texts") or case.get("prompts") or case["rows"], case["min"], case["max"]
    r = random.Random(n * 1_000_003 + lo * 1009 + hi)
    return [hi] + [r.randint(lo, hi) for _ in range(n - 1)]


def _gen(seed: int, part: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(seed * 64 + part)


def _normal(shape, gen, std=0.02, mean=0.0, dtype=torch.bfloat16):
    return torch.empty(shape, dtype=torch.float32, device=DEV).normal_(mean, std, generator=gen).to(dtype)


def _tokens(case: dict, seed: int, vocab: int, extra: int = 0) -> list[list[int]]:
    r = np.random.RandomState(seed % (1 << 31))
    return [r.randint(5, vocab, n + extra).tolist() for n in _lens(case)]


def _encoder_weights(cfg, seed: int) -> dict[str, torch.Tensor]:
    g, h, f = _gen(seed, 1), cfg.hidden, cfg.ffn
    sd = {"embeddings.word_embeddings.weight": _normal((cfg.vocab, h), g),
          "embeddings.position_embeddings.weight": _normal((cfg.max_pos, h), g),
          "embeddings.token_type_embeddings.weight": _normal((cfg.type_vocab, h), g)}

    def norm(name):
        sd[name + ".weight"], sd[name + ".bias"] = _normal(h, g, 0.05, 1.0), _normal(h, g)
    norm("embeddings.LayerNorm")
    for i in range(cfg.layers):
        p = f"encoder.layer.{i}."
        for name, n, k in (("attention.self.query", h, h), ("attention.self.key", h, h), ("attention.self.value", h, h),
                           ("attention.output.dense", h, h), ("intermediate.dense", f, h), ("output.dense", h, f)):
            # (a layer adds a part of the stream, as in a trained encoder)
            out = name.endswith("output.dense")
            sd[p + name + ".weight"], sd[p + name + ".bias"] = _normal((n, k), g, 0.006 if out else 0.02), _normal(n, g)
        norm(p + "attention.output.LayerNorm")
        norm(p + "output.LayerNorm")
    return sd


def _decoder_layer(cfg, seed: int, i: int) -> dict[str, torch.Tensor]:
    g, h, D = _gen(seed, 2), cfg.hidden, cfg.head_dim
    g.manual_seed(seed * 997 + 13 * i + 5)
    out = 0.02 / (2 * cfg.layers) ** 0.5
    return {"wqkv": _normal(((cfg.heads + 2 * cfg.kv_heads) * D, h), g), "wo": _normal((h, cfg.heads * D), g, out),
            "gate": _normal((cfg.ffn, h), g), "up": _normal((cfg.ffn, h), g), "w_down": _normal((h, cfg.ffn), g, out)}


def _decoder_ends(cfg, seed: int) -> dict[str, torch.Tensor]:
    g = _gen(seed, 3)  # embeddings that outweigh what a single layer adds, as in a trained decoder's stream
    return {"embed": _normal((cfg.vocab, cfg.hidden), g, 1.0), "lm_head": _normal((cfg.vocab, cfg.hidden), g)}


def _decoder_weights(cfg, seed: int) -> dict:
    one = torch.ones(cfg.hidden, dtype=torch.bfloat16, device=DEV)
    layers = []
    for i in range(cfg.layers):
        L = _decoder_layer(cfg, seed, i)
        L["w_gu"] = interleave_gate_up(L.pop("gate"), L.pop("up"))
        layers.append({**L, "ln_attn": one, "ln_mlp": one.clone()})
    return {**_decoder_ends(cfg, seed), "norm": one.clone(), "layers": layers}


def _mixed_weights(cfg, seed: int) -> dict[str, torch.Tensor]:
    """A checkpoint's tensors: matrices that keep variances, decays and step sizes in their working ranges."""
    g, out = _gen(seed, 4), {}
    uniform = {"shift": (0.0, 0.6), "lam": (-5.0, -1.0), "A_log": (0.0, math.log(16.0)), "dt.b": (-5.0, -2.0),
               "dt_bias": (-5.0, -2.0)}
    normal = {"ls1": (0.3, 0.05), "ls2": (0.3, 0.05), "pb": (-3.0, 0.5), "D": (1.0, 0.1), "norm1": (1.0, 0.1),
              "norm2": (1.0, 0.1)}
    for name, shape in tensor_shapes(cfg).items():
        p = name.split(".")
        key = ".".join(p[-2:]) if p[-1] == "b" and p[-2] == "dt" else p[-1]
        t = torch.empty(shape, dtype=torch.float32, device=DEV)
        if key in uniform:
            t.uniform_(*uniform[key], generator=g)
        elif key == "norm":
            t.normal_(1.0, 0.1, generator=g)
        elif key in normal:
            t.normal_(*normal[key], generator=g)
        elif len(shape) > 1 and (key != "b" or p[-2] == "mix"):
            small = 0.25 if key in ("o", "down") else 1.0  # a layer adds a part of the stream, as in a trained decoder
            t.normal_(0.0, small * shape[-1] ** -0.5, generator=g)
        else:
            t.normal_(0.0, 0.1, generator=g)
        out[name] = t.to(torch.bfloat16)
    return out


def _vectors(case: dict, seed: int):
    """Rows around topics, as a corpus's embeddings are, and questions around the same topics: unit norm."""
    g, n, d = _gen(seed, 6), case["rows"], case["dim"]
    topics = F.normalize(_normal((max(64, n // 800), d), g, 1.0, dtype=torch.float32), dim=-1)

    def around(m, spread):
        x = _normal((m, d), g, spread * d ** -0.5, dtype=torch.float32)
        at = torch.randint(topics.shape[0], (m,), generator=g, device=DEV)
        return F.normalize(x.add_(topics.index_select(0, at)), dim=-1).to(torch.bfloat16)
    X = torch.cat([around(min(1 << 18, n - a), 1.0) for a in range(0, n, 1 << 18)])
    return X, around(case["queries"], 0.8)


def _documents(case: dict) -> list[int]:
    """Rows of each document: 1 to 96 chunks."""
    r, left, out = random.Random(case["rows"]), case["rows"], []
    while left:
        out.append(min(left, r.randint(1, 96)))
        left -= out[-1]
    return out


def _filters(case: dict, docs: int, seed: int):
    if not case["docs"]:
        return None
    r = random.Random(seed)
    return [r.sample(range(docs), min(docs, case["docs"])) for _ in range(case["queries"])]


# ---------------------------------------------------------------------------------------- prepare and run
def prepare(case: dict, seed: int) -> dict:
    return _PREPARE[case["kind"]](case, seed)


def run(state: dict):
    return state["run"](state)


def _prepare_embed(case, seed):
    cfg = encoder_config(case["arch"])
    enc = BertEncoder.from_hf_state_dict(cfg, _encoder_weights(cfg, seed), DEV, dtype=case["dtype"])
    seqs = _tokens(case, seed, cfg.vocab)
    if len(seqs) <= 64:
        enc.prepare_graphs()
    return {"enc": enc, "seqs": seqs, "run": _run_embed}


def _run_embed(s):
    enc, seqs = s["enc"], s["seqs"]
    if len(seqs) == 1:
        return enc.encode_one(seqs[0])
    v = enc.encode_batch(seqs) if len(seqs) <= 64 else None  # None: texts too long for a captured batch
    return enc.encode_packed(seqs) if v is None else v


def _prepare_search(case, seed):
    X, q = _vectors(case, seed)
    docs = _documents(case)
    ix = make_index(case["index"], case["dim"], torch.device(DEV), lists=case.get("lists", 100), probes=case.get("probes", 1))
    ix.add_bulk([f"d{i}" for i in range(len(docs))], docs, np.arange(case["rows"]) + 7, X)
    if case["index"] == "ivfflat":
        ix.train()
    f = _filters(case, len(docs), seed)
    return {"index": ix, "q": q, "k": case["k"], "filters": f and [[f"d{i}" for i in one] for one in f], "run": _run_search}


def _run_search(s):
    return s["index"].search_ids(s["q"], s["k"], -1.0, s["filters"])


def _decoder(case, seed):
    cfg = decoder_config(case["arch"])
    mixed = isinstance(cfg, HybridConfig)
    w = _mixed_weights(cfg, seed) if mixed else _decoder_weights(cfg, seed)
    return cfg, mixed, make_decoder(cfg, DEV, weights=w, dtype=case["dtype"])


def _batch(seqs, slots, pos0):
    lens = [len(s) for s in seqs]
    cu = np.concatenate([[0], np.cumsum(lens)])

    def to(a, dt=torch.int32):
        return torch.from_numpy(np.asarray(a)).to(dt).to(DEV)
    return dict(ids=to(np.concatenate(seqs)), pos=to(np.concatenate([np.arange(n) + pos0 for n in lens])),
                slot_tok=to(np.repeat(slots, lens)), cu=to(cu), max_seqlen=max(lens),
                last_idx=to(cu[1:] - 1, torch.int64), lens=lens)


def _prepare_prefill(case, seed):
    cfg, mixed, model = _decoder(case, seed)
    P, seqs = case["head"], _tokens(case, seed, cfg.vocab)
    n, most = len(seqs), -(-(P + case["max"]) // 64) * 64
    cache = model.alloc_cache(n + (1 if P else 0), most)
    slots = cache.acquire(n, [len(s) for s in seqs]) if mixed else cache.acquire(n)
    prefix = None
    if P:
        prefix = (cache.acquire(1)[0], P)
        model.prefill(**_batch([_head(seed, P)], [prefix[0]], 0))
    return {"model": model, "batch": _batch(seqs, slots, P), "prefix": prefix, "mixed": mixed, "run": _run_prefill}


def _head(seed, P):
    return np.random.RandomState(seed % 65536 + 1).randint(5, 30000, P).tolist()


def _run_prefill(s):
    logits = s["model"].prefill(**s["batch"], prefix=s["prefix"], local_logits=True)
    cache = s["model"].cache
    return {"logits": logits, "state": _states(cache) if s["mixed"] else cache.buf}


def _states(cache):
    return [L[k] for L in cache.layers for k in STATES if k in L]


def _prepare_decode(case, seed):
    cfg, mixed, model = _decoder(case, seed)
    rows, lens = case["rows"], _lens(case)
    tokens = [s[-1] for s in _tokens(case, seed, cfg.vocab, 1)]
    # a serving cache: slots of the whole context, or pages for what is in it
    most = min(4096, cfg.max_pos) if not mixed else case["max"] + 64
    cache = model.alloc_cache(rows + 1, most)
    gen = Generator(model, max_batch=rows, max_seq=most)  # reserves the workspaces (and the spare slot)
    slots = cache.acquire(rows, [n + 1 for n in lens])
    st = DecodeState(model, rows, 64, 0.2, 0)

    def to(a):
        return torch.tensor(a, dtype=torch.int32, device=DEV)
    start = (to(tokens), to(lens), to([n + 1 for n in lens]))
    st.slot.copy_(to(slots))
    st.active.fill_(1)

    def begin():
        for t, v in zip((st.tokens, st.pos, st.lens), start):
            t.copy_(v)
    begin()
    st.start.copy_(st.pos)
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            model.decode_step(st)
            begin()
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        model.decode_step(st)
    begin()
    if mixed:
        seqs = [s[:-1] for s in _tokens(case, seed, cfg.vocab, 1)]
        for a in range(0, rows, 16):
            model.prefill(**_batch(seqs[a:a + 16], slots[a:a + 16], 0))
        kv = None
    else:
        for i in range(cfg.layers):
            _context(cfg, case, seed, i, cache.buf[i])
        kv = (st.slot.long(), st.pos.long())
    return {"gen": gen, "model": model, "st": st, "graph": graph, "begin": begin, "kv": kv, "run": _run_decode}


def _context(cfg, case, seed, i, buf):
    """Keys and values of the contexts of layer i, [2, slots, kv heads, positions, D]."""
    return buf.normal_(0.0, 1.0, generator=_gen(seed, 7).manual_seed(seed * 991 + i))


def _run_decode(s):
    s["begin"]()
    s["graph"].replay()
    model, st = s["model"], s["st"]
    if s["kv"] is None:
        return {"logits": st.logits[:, :model.cfg.vocab], "state": _states(model.cache)}
    slot, pos = s["kv"]
    return {"logits": st.logits, "new": model.cache.buf[:, :, slot, :, pos]}


_PREPARE = {"embed": _prepare_embed, "search": _prepare_search, "prefill": _prepare_prefill, "decode": _prepare_decode}


# ---------------------------------------------------------------------------------------- work and tolerance
def work(case: dict) -> dict:
    if case["kind"] == "search":
        n, d, q = case["rows"], case["dim"], case["queries"]
        docs = _documents(case)
        if case["index"] == "ivfflat":  # lists of even length
            per = n * min(1.0, case["probes"] / case["lists"])
            read = min(n, per * q)
        else:
            per = min(n, case["docs"] * n / len(docs)) if case["docs"] else n
            read = min(n, per * q)
        return {"bytes": 2 * d * (read + q) + 12 * q * case["k"], "flops": 2 * d * per * q}
    lens = _lens(case)
    if case["kind"] == "embed":
        cfg = encoder_config(case["arch"])
        mat = cfg.layers * (4 * cfg.hidden ** 2 + 2 * cfg.hidden * cfg.ffn)
        size = 1 if case["dtype"] == "fp8" else 2
        return {"bytes": size * mat + sum(lens) * 2 * cfg.hidden + 4 * len(lens) * cfg.hidden,
                "flops": sum(2 * mat * n + 4 * cfg.layers * cfg.hidden * n * n for n in lens)}
    cfg = decoder_config(case["arch"])
    size = 4 if case["dtype"] == "fp32" else 2
    mixed = isinstance(cfg, HybridConfig)
    tables = cfg.vocab * cfg.hidden * (1 if mixed and cfg.block == "parallel" else 2)
    body, head = cfg.param_count() - tables, cfg.vocab * cfg.hidden
    # recurrent state: read and written once a sequence
    fixed = sum(_state_bytes(cfg.spec[r.layer].mixer) for r in cfg.runs) if mixed else 0
    kv = cfg.kv_bytes_per_token(size)
    n = len(lens)
    out = size * n * cfg.vocab
    if case["kind"] == "decode":
        return {"bytes": size * (body + head) + sum(lens) * kv + n * (2 * fixed + kv) + out,
                "flops": n * 2 * (body + head) + sum(_attention_flops(cfg, k, 1) for k in lens)}
    P = case["head"]
    return {"bytes": size * (body + head) + (sum(lens) + P) * kv + n * fixed + out,
            "flops": sum(2 * body * k + 2 * head + _attention_flops(cfg, P + k / 2, k) for k in lens)}


def _state_bytes(m) -> int:
    if isinstance(m, GatedRecurrence):
        return 4 * m.width
    if isinstance(m, ChannelDelta):
        return 4 * m.heads * m.dim * m.vdim
    return 4 * m.inner * m.state if hasattr(m, "inner") else 0


def _attention_flops(cfg, keys: float, queries: float) -> float:
    """Products with a context's keys and values, and of recurrent layers with their state."""
    if not isinstance(cfg, HybridConfig):
        return 4.0 * cfg.layers * cfg.heads * cfg.head_dim * keys * queries
    tot = 0.0
    for r in cfg.runs:
        m = cfg.spec[r.layer].mixer
        if isinstance(m, SigmoidAttention):
            tot += 4.0 * m.heads * m.dim * keys * queries
        elif isinstance(m, LatentAttention):
            tot += 2.0 * m.heads * (m.dim + m.rot_dim + m.vdim) * keys * queries
        elif isinstance(m, ChannelDelta):
            tot += 6.0 * m.heads * m.dim * m.vdim * queries
        elif not isinstance(m, GatedRecurrence):
            tot += 6.0 * m.inner * m.state * queries
    return tot


def tolerance(case: dict):
    if case["kind"] == "search":
        return {"rel": 1e-5, "differ": 0.005}  # 32-bit sums; neighbours a rounding apart may change places
    if case.get("dtype") == "fp32":
        return {"rel": 1e-4, "max": 0.01}
    if case["kind"] == "embed":
        return {"rel": {"fp16": 0.006, "bf16": 0.03, "fp8": 0.03}[case["dtype"]], "max": 0.3}
    return {"rel": 0.03, "max": 0.6}  # bf16 through 32 layers


# ---------------------------------------------------------------------------------------- in 64 bits
@torch.no_grad()
def exact(case: dict, seed: int):
    return _EXACT[case["kind"]](case, seed)


def _lin(x, w, b=None):
    y = x @ w.double().T
    return y if b is None else y + b.double()


def _split(x, lens):
    return x.split(list(lens), 0)


def _exact_embed(case, seed):
    cfg, eps = encoder_config(case["arch"]), encoder_config(case["arch"]).eps
    w, seqs = _encoder_weights(cfg, seed), _tokens(case, seed, cfg.vocab)
    lens, H, D = [len(s) for s in seqs], cfg.heads, cfg.head_dim
    ids = torch.tensor([t for s in seqs for t in s], device=DEV)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens])

    def norm(x, name):
        return F.layer_norm(x, (cfg.hidden,), w[name + ".weight"].double(), w[name + ".bias"].double(), eps)

    def lin(x, name):
        return _lin(x, w[name + ".weight"], w[name + ".bias"])
    e = "embeddings."
    x = w[e + "word_embeddings.weight"].double()[ids] + w[e + "position_embeddings.weight"].double()[pos]
    x = norm(x + w[e + "token_type_embeddings.weight"].double()[0], e + "LayerNorm")
    for i in range(cfg.layers):
        p = f"encoder.layer.{i}."
        q, k, v = (lin(x, p + f"attention.self.{n}").view(-1, H, D) for n in ("query", "key", "value"))
        a = []
        for q1, k1, v1 in zip(*(_split(t, lens) for t in (q, k, v))):
            s = torch.softmax(q1.transpose(0, 1) @ k1.permute(1, 2, 0) * D ** -0.5, -1)
            a.append((s @ v1.transpose(0, 1)).transpose(0, 1).reshape(-1, H * D))
        x = norm(x + lin(torch.cat(a), p + "attention.output.dense"), p + "attention.output.LayerNorm")
        f = F.gelu(lin(x, p + "intermediate.dense"))
        x = norm(x + lin(f, p + "output.dense"), p + "output.LayerNorm")
    rows = [t[0] if cfg.pooling == "cls" else t.mean(0) for t in _split(x, lens)]
    return F.normalize(torch.stack(rows), dim=-1)


def _exact_search(case, seed):
    if case["index"] == "ivfflat":
        return None  # the lists are the index's own
    X, q = _vectors(case, seed)
    docs = _documents(case)
    f = _filters(case, len(docs), seed)
    top, at = [], []
    owner = torch.repeat_interleave(torch.arange(len(docs), device=DEV), torch.tensor(docs, device=DEV))
    for i in range(case["queries"]):
        s = torch.cat([x.double() @ q[i].double() for x in X.split(1 << 18)])
        if f is not None:
            s = s.masked_fill(~torch.isin(owner, torch.tensor(f[i], device=DEV)), -math.inf)
        v, j = s.topk(case["k"])
        top.append(v)
        at.append(torch.where(v > -math.inf, j + 7, -1))
    return torch.stack(top), torch.stack(at)


def _rope(x, pos, theta):
    """Pairs (2i, 2i + 1) of the columns of x [T, heads, D] turned by pos * theta^(-2i / D)."""
    D = x.shape[-1]
    a = pos.double()[:, None] * theta ** (-torch.arange(0, D, 2, device=DEV, dtype=torch.float64) / D)
    c, s = a.cos()[:, None], a.sin()[:, None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).flatten(-2)


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _llama_layers(cfg, seed, x, pos, attend):
    """The stream after all layers; attend(layer, q, k, v) is told each layer's rotated queries and keys."""
    H, G, D = cfg.heads, cfg.kv_heads, cfg.head_dim
    for i in range(cfg.layers):
        L = _decoder_layer(cfg, seed, i)
        q, k, v = _lin(_rms(x, cfg.eps), L["wqkv"]).view(-1, H + 2 * G, D).split([H, G, G], 1)
        a = attend(i, _rope(q, pos, cfg.rope_theta), _rope(k, pos, cfg.rope_theta), v)
        x = x + _lin(a, L["wo"])
        h = _rms(x, cfg.eps)
        x = x + _lin(F.silu(_lin(h, L["gate"])) * _lin(h, L["up"]), L["w_down"])
    return x


def _softmax_attention(q, k, v, causal_from=None):
    """q [T, H, D] over k, v [S, G, D]; row i sees keys up to causal_from + i (None: all)."""
    T, H, D = q.shape
    S, G, _ = k.shape
    q = q.view(T, G, H // G, D).permute(1, 2, 0, 3).reshape(G, -1, D)
    s = (q @ k.permute(1, 2, 0) * D ** -0.5).view(G, H // G, T, S)
    if causal_from is not None:
        s.masked_fill_(torch.arange(S, device=DEV)[None] > torch.arange(T, device=DEV)[:, None] + causal_from, -math.inf)
    a = torch.softmax(s, -1).view(G, -1, S) @ v.transpose(0, 1)
    return a.view(G, H // G, T, D).permute(2, 0, 1, 3).reshape(T, H * D)


def _exact_prefill(case, seed):
    cfg = decoder_config(case["arch"])
    seqs = _tokens(case, seed, cfg.vocab)
    if isinstance(cfg, HybridConfig):
        return _exact_mixed(cfg, seed, seqs, len(seqs))
    P, n = case["head"], len(seqs)
    if P:
        seqs = [_head(seed, P)] + seqs  # the head first: the others see its keys
    lens = [len(s) for s in seqs]
    first = [0] + [P] * n if P else [0] * n
    slots = [n, *range(n)] if P else list(range(n))
    most = -(-(P + case["max"]) // 64) * 64
    buf = torch.zeros((cfg.layers, 2, len(seqs), cfg.kv_heads, most, cfg.head_dim), dtype=torch.float64, device=DEV)
    ids = torch.tensor([t for s in seqs for t in s], device=DEV)
    pos = torch.cat([torch.arange(m, device=DEV) + p for m, p in zip(lens, first)])
    ends = _decoder_ends(cfg, seed)

    def attend(i, q, k, v):
        out, head = [], None
        for q1, k1, v1, p, s in zip(*(_split(t, lens) for t in (q, k, v)), first, slots):
            buf[i, 0, s, :, p:p + len(k1)] = k1.transpose(0, 1)
            buf[i, 1, s, :, p:p + len(k1)] = v1.transpose(0, 1)
            if p:
                k1, v1 = torch.cat([head[0], k1]), torch.cat([head[1], v1])
            elif P:
                head = (k1, v1)
            out.append(_softmax_attention(q1, k1, v1, p))
        return torch.cat(out)
    x = _llama_layers(cfg, seed, ends["embed"].double()[ids], pos, attend)
    last = (torch.tensor(lens, device=DEV).cumsum(0) - 1)[len(lens) - n:]
    return {"logits": _lin(_rms(x[last], cfg.eps), ends["lm_head"]), "state": buf}


def _exact_decode(case, seed):
    cfg = decoder_config(case["arch"])
    rows, lens = case["rows"], _lens(case)
    seqs = _tokens(case, seed, cfg.vocab, 1)
    if isinstance(cfg, HybridConfig):
        return _exact_mixed(cfg, seed, seqs, rows + 1)
    ends = _decoder_ends(cfg, seed)
    ids, pos = torch.tensor([s[-1] for s in seqs], device=DEV), torch.tensor(lens, device=DEV)
    kv = torch.empty((2, rows + 1, cfg.kv_heads, min(4096, cfg.max_pos), cfg.head_dim), dtype=torch.bfloat16, device=DEV)
    new = torch.empty((rows, cfg.layers, 2, cfg.kv_heads, cfg.head_dim), dtype=torch.float64, device=DEV)

    def attend(i, q, k, v):
        _context(cfg, case, seed, i, kv)
        new[:, i, 0], new[:, i, 1] = k, v
        # the spare slot is taken first: row b sits in slot b + 1
        c = [[torch.cat([kv[j, b + 1, :, :n].double().transpose(0, 1), t[b:b + 1]]) for j, t in enumerate((k, v))]
             for b, n in enumerate(lens)]
        return torch.cat([_softmax_attention(q[b:b + 1], *c[b]) for b in range(rows)])
    x = _llama_layers(cfg, seed, ends["embed"].double()[ids], pos, attend)
    return {"logits": _lin(_rms(x, cfg.eps), ends["lm_head"]), "new": new}


# decoders of mixed layers, whole sequences, longest first: a step of a recurrence runs the sequences that are left
def _conv(x, kernel, lens):
    k = kernel.double()
    taps = k.shape[1]
    return torch.cat([F.conv1d(F.pad(s.T[None], (taps - 1, 0)), k[:, None], groups=k.shape[0])[0].T for s in _split(x, lens)])


class _Steps:
    """Packed rows <-> rows by step: at(t) are the rows of step t of the sequences longer than t."""

    def __init__(self, lens):
        self.lens, self.most = lens, max(lens)
        first = np.cumsum([0] + lens[:-1])
        self.rows = [torch.tensor([f + t for f, n in zip(first, lens) if n > t], device=DEV) for t in range(self.most)]


def _delta(w, p, h, m, eps, steps):
    H, G, K, V = m.heads, m.kv_heads, m.dim, m.vdim
    q, k, v = (F.silu(_conv(_lin(h, w[p + n]), w[p + n + ".conv"], steps.lens)) for n in "qkv")

    def unit(x):
        x = x.view(-1, G, K)
        return (x / torch.sqrt((x * x).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 1)
    q, k, v = unit(q) * K ** -0.5, unit(k), v.view(-1, H, V)
    beta = torch.sigmoid(_lin(h, w[p + "b"]))[..., None]
    z = _lin(_lin(h, w[p + "a1"]), w[p + "a2"], w[p + "dt_bias"]).view(-1, H, K)
    g = torch.exp(-torch.exp(w[p + "A_log"].double())[:, None] * F.softplus(z, threshold=40))
    S = torch.zeros(len(steps.lens), H, V, K, dtype=torch.float64, device=DEV)
    out = torch.empty_like(v)
    for r in steps.rows:
        s = S[:len(r)]
        k1 = k[r]
        s.mul_(g[r][:, :, None])
        u = beta[r] * (v[r] - (s @ k1[..., None])[..., 0])
        s.view(-1, V, K).baddbmm_(u.reshape(-1, V, 1), k1.reshape(-1, 1, K))
        out[r] = (s @ q[r][..., None])[..., 0]
    gate = _lin(_lin(h, w[p + "g1"]), w[p + "g2"]).view(-1, H, V)
    o = _rms(out, eps) * w[p + "norm"].double() * torch.sigmoid(gate)
    return _lin(o.reshape(len(h), -1), w[p + "o"]), S


def _latent(w, p, h, m, eps, steps):
    H, D, R, L, V = m.heads, m.dim, m.rot_dim, m.kv_rank, m.vdim
    pos = torch.cat([torch.arange(n, device=DEV) for n in steps.lens])
    a = pos.double()[:, None] * m.rot_base ** (-2 * torch.arange(R // 2, device=DEV, dtype=torch.float64) / R)

    def turn(x):
        c, s = a.cos()[:, None], a.sin()[:, None]
        u, v = x[..., :R // 2], x[..., R // 2:]
        return torch.cat([u * c - v * s, v * c + u * s], -1)
    q = _lin(_rms(_lin(h, w[p + "dq"]), eps) * w[p + "dq.norm"].double(), w[p + "uq"]).view(-1, H, D + R)
    q = torch.cat([q[..., :D], turn(q[..., D:])], -1)
    dkv = _lin(h, w[p + "dkv"])
    c = _rms(dkv[:, :L], eps) * w[p + "dkv.norm"].double()
    k = torch.cat([_lin(c, w[p + "uk"]).view(-1, H, D), turn(dkv[:, None, L:]).expand(-1, H, R)], -1)
    v, sink, out = _lin(c, w[p + "uv"]).view(-1, H, V), w[p + "sink"].double(), []
    for q1, k1, v1 in zip(*(_split(t, steps.lens) for t in (q, k, v))):
        s = q1.transpose(0, 1) @ k1.permute(1, 2, 0) * m.scale
        s.masked_fill_(torch.ones(s.shape[1:], dtype=torch.bool, device=DEV).triu(1), -math.inf)
        s = torch.cat([s, sink[:, None, None].expand(-1, s.shape[1], 1)], -1)
        out.append((torch.softmax(s, -1)[..., :-1] @ v1.transpose(0, 1)).transpose(0, 1).reshape(-1, H * V))
    return _lin(torch.cat(out) * torch.sigmoid(_lin(h, w[p + "g"])), w[p + "o"]), None


def _recurrence(w, p, h, m, eps, steps):
    y = F.gelu(_lin(h, w[p + "y"], w[p + "y.b"]), approximate="tanh")
    u = _conv(_lin(h, w[p + "x"], w[p + "x.b"]), w[p + "conv"], steps.lens) + w[p + "conv.b"].double()
    ub = u.view(len(u), m.blocks, -1).transpose(0, 1)
    r, i = (torch.sigmoid(ub @ w[p + n].double().transpose(1, 2) + w[p + n + ".b"].double()[:, None]).transpose(0, 1)
            .reshape(u.shape) for n in ("ra", "ri"))
    a = torch.exp(-8 * r * F.softplus(w[p + "lam"].double()))
    drive = torch.sqrt(1 - a * a) * i * u
    S, out = torch.zeros(len(steps.lens), u.shape[1], dtype=torch.float64, device=DEV), torch.empty_like(u)
    for r1 in steps.rows:
        s = S[:len(r1)]
        out[r1] = s.mul_(a[r1]).add_(drive[r1])
    return _lin(out * y, w[p + "o"]), S


def _scan(w, p, h, m, eps, steps):
    n, R, N = m.inner, m.dt_rank, m.state
    xz = _lin(h, w[p + "in"])
    x = F.silu(_conv(xz[:, :n], w[p + "conv"], steps.lens) + w[p + "conv.b"].double())
    low = _lin(x, w[p + "x"])
    dt = F.softplus(_lin(low[:, :R], w[p + "dt"], w[p + "dt.b"]), threshold=40)
    A, D = -torch.exp(w[p + "A_log"].double()), w[p + "D"].double()
    S, out = torch.zeros(len(steps.lens), n, N, dtype=torch.float64, device=DEV), torch.empty_like(x)
    for r in steps.rows:
        s, d = S[:len(r)], dt[r]
        s.mul_(torch.exp(d[..., None] * A)).add_((d * x[r])[..., None] * low[r, None, R:R + N])
        out[r] = (s @ low[r, R + N:, None])[..., 0] + D * x[r]
    return _lin(out * F.silu(xz[:, n:]), w[p + "o"]), S


def _sigmoid(w, p, h, m, eps, steps):
    H, G, D = m.heads, m.kv_heads, m.dim
    q = _rms(_lin(h, w[p + "q"]).view(-1, H, D), eps) * w[p + "q.norm"].double()
    v = _lin(h, w[p + "k"]).view(-1, G, D)
    k = _rms(v, eps) * w[p + "k.norm"].double()
    if m.q_temp:
        pos = torch.cat([torch.arange(n, device=DEV) for n in steps.lens]).double()
        q = q * (1 + m.q_temp[0] * torch.log(torch.floor((pos + 1) / m.q_temp[1]) + 1))[:, None, None]
    out = []
    for q1, k1, v1 in zip(*(_split(t, steps.lens) for t in (q, k, v))):
        T = len(q1)
        s = q1.view(T, G, -1, D).permute(1, 2, 0, 3).reshape(G, -1, D) @ k1.permute(1, 2, 0) * m.scale
        s = torch.sigmoid(s.view(H, T, T) + w[p + "pb"].double()[:, None, None]).tril_()
        a = s.view(G, -1, T) @ v1.transpose(0, 1)
        out.append(a.view(H, T, D).transpose(0, 1))
    o = torch.cat(out) * torch.sigmoid(_lin(h, w[p + "g"]))[..., None]
    return _lin(o.reshape(len(h), -1), w[p + "o"]), None


_MIXERS = {ChannelDelta: _delta, LatentAttention: _latent, GatedRecurrence: _recurrence, SigmoidAttention: _sigmoid}


def _exact_mixed(cfg, seed, seqs, slots):
    if sum(map(len, seqs)) > EXACT_TOKENS:
        return None
    w, eps = _mixed_weights(cfg, seed), cfg.eps
    order = sorted(range(len(seqs)), key=lambda i: -len(seqs[i]))
    steps = _Steps([len(seqs[i]) for i in order])
    x = w["embed"][torch.tensor([t for i in order for t in seqs[i]], device=DEV)].double() * cfg.embed_scale
    back = torch.tensor(np.argsort(order), device=DEV)
    states, parallel = [], cfg.block == "parallel"

    def normed(t, name):
        t = F.layer_norm(t, (cfg.hidden,), eps=eps) if parallel else _rms(t, eps)
        return t * w[name].double()
    for r in cfg.runs:
        m, name = cfg.spec[r.layer].mixer, f"l{r.weights}."
        mix = _MIXERS.get(type(m), _scan)
        if parallel:
            h = normed(x, name + "norm1")
        else:
            prev = torch.cat([F.pad(s[:-1], (0, 0, 1, 0)) for s in _split(x, steps.lens)])
            h = x + (prev - x) * w[name + "shift"].double()
        y, S = mix(w, name + "mix.", h, m, eps, steps)
        if S is not None:
            full = torch.zeros(slots, *S.shape[1:], dtype=torch.float64, device=DEV)
            full[slots - len(seqs):] = S[back]  # a spare slot is taken first
            states.append(full)
        f = name + "mlp."
        if parallel:
            ff = F.silu(_lin(h, w[f + "gate"], w[f + "gate.b"])) * _lin(h, w[f + "up"], w[f + "up.b"])
            x = x + y * w[name + "ls1"].double() + _lin(ff, w[f + "down"], w[f + "down.b"]) * w[name + "ls2"].double()
        else:
            x = normed(cfg.alpha * x + y, name + "norm1")
            ff = torch.relu(_lin(x, w[f + "gate"])) * _lin(x, w[f + "up"])
            x = normed(cfg.alpha * x + _lin(ff, w[f + "down"]), name + "norm2")
    last = (torch.tensor(steps.lens, device=DEV).cumsum(0) - 1)[back]
    logits = _lin(normed(x[last], "final.norm"), w["embed" if parallel else "head"])
    return {"logits": logits, "state": states}


_EXACT = {"embed": _exact_embed, "search": _exact_search, "prefill": _exact_prefill, "decode": _exact_decode}
