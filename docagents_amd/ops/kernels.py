"""ctypes bindings for the gfx950 kernel library (``_da_*.so``, see ``build``).

Every wrapper validates shapes / dtypes / contiguity / device on the host BEFORE launching (a
mis-shaped launch of a hand-written kernel can fault the GPU), launches on PyTorch's current HIP
stream, and raises on any launch error. There is deliberately no silent fallback: on a GPU box,
if the library is missing the import fails loudly (``KernelLibraryMissing``). The fp32 PyTorch
oracles for tests live in ``docagents_amd.ops.reference``.
"""
from __future__ import annotations

import contextlib
import ctypes
import functools
import math
import os
import threading
from pathlib import Path

import numpy as np
import torch

_LOCK = threading.Lock()
# What the rules below choose for a shape, looked up instead of worked out for each product of each layer (2 us each, which
# an encoder's layers that are launched one by one wait for)
_rule = functools.lru_cache(maxsize=4096)
# DA_KERNELS_DEBUG=1: the -DDA_DEBUG build (device asserts: bounds / shape preconditions inside the
# kernels; python -m docagents_amd.ops.build --debug) instead of the -O3 library
_DEBUG = os.environ.get("DA_KERNELS_DEBUG", "0") == "1"
_LIB_OVERRIDE: Path | None = None  # one library with every launcher, instead of the parts (A/B runs)

EPI_NONE, EPI_BIAS, EPI_GELU, EPI_SWIGLU, EPI_RESID = 0, 1, 2, 3, 4
EPI_ROPE = 6  # gemm8p only: QKV + RoPE + KV-cache write
EPI_REGLU = 7  # EPI_SWIGLU with relu in place of silu
GATED = (EPI_SWIGLU, EPI_REGLU)

c_longlong = ctypes.c_longlong
c_void_p, c_int, c_float, c_uint, c_size_t = (ctypes.c_void_p, ctypes.c_int, ctypes.c_float,
                                             ctypes.c_uint, ctypes.c_size_t)

_SIGS = {
    "da_gemm_bf16": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int,
                     c_int, c_int, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_float, c_void_p, c_void_p, c_void_p],
    "da_gemm_rope": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int] + [c_void_p] * 5
                    + [c_int] * 5 + [c_void_p],
    "da_gemm_fp8": [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int,
                    c_int, c_int, c_int, c_int, c_void_p],
    "da_quant_fp8_rows": [c_void_p, c_int, c_int, c_int, c_void_p, c_int, c_void_p, c_void_p],
    "da_layernorm_q": [c_void_p] * 7 + [c_int, c_int, c_float, c_void_p],
    "da_bert_embed_ln_q": [c_void_p] * 11 + [c_int, c_int, c_float, c_void_p],
    "da_gemm_resid_rmsnorm": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int,
                              c_int, c_int, c_int, c_void_p, c_void_p, c_float, c_void_p, c_int, c_void_p],
    "da_rmsnorm": [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_float, c_void_p],
    "da_swiglu_interleaved": [c_void_p, c_int, c_void_p, c_int, c_int, c_int, c_void_p],
    "da_layernorm": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_float, c_void_p],
    "da_bert_embed_ln": [c_void_p] * 9 + [c_int, c_int, c_float, c_void_p],
    "da_embed": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_void_p],
    "da_pool_l2norm": [c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p],
    "da_rope_cache": [c_void_p] * 6 + [c_int] * 6 + [c_void_p],
    "da_sample": [c_void_p, c_int, c_int, c_int, c_float, c_uint, c_uint] + [c_void_p] * 9
                 + [c_int] * 6 + [c_void_p],
    "da_flash_attn_v2": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_int, c_int,
                         c_int, c_int, c_int, c_int, c_float, c_void_p, c_int, c_void_p, c_void_p, c_longlong,
                         c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p],
    "da_malloc_uncached": [c_longlong, ctypes.POINTER(c_void_p)],
    "da_gemm_dk": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                   c_int, c_void_p, c_int, c_int, c_float, c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p],
    "da_gemm_dk_rope": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_int, c_int, c_float]
                       + [c_void_p] * 5 + [c_int] * 5 + [c_void_p],
    "da_gemm_dk_ws": [c_int] * 3,
    "da_enc_text_ws": [c_int] * 6,
    "da_enc_text_pooled": [c_void_p] * 4 + [c_int] + [c_void_p] * 4 + [c_int] * 4 + [c_float, c_float, c_int, c_void_p, c_int, c_void_p, c_int, c_void_p],
    "da_host_address": [c_void_p, ctypes.POINTER(c_void_p)],
    "da_enc_text": [c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p] + [c_int] * 4 + [c_float, c_float, c_int, c_void_p, c_int, c_void_p],
    "da_gemm_dk_parts": [c_int],
    "da_gemm_dk_rows": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p] + [c_int] * 7 + [c_void_p],
    "da_enc_rows": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p] + [c_int] * 5
                  + [c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_int, c_void_p],
    "da_enc_attn_rows": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p] + [c_int] * 5 + [c_void_p, c_float]
                       + [c_void_p, c_void_p, c_void_p, c_float, c_void_p, c_int, c_void_p],
    "da_encoder_layer": [c_void_p, c_int, c_int, c_int, c_void_p],
    "da_gemm_tail_ws": [c_int] * 5,
    "da_gemm_fp8_tile": [c_int] * 2,
    "da_gemm8p_ksteps": [c_int] * 5,
    "da_gemm_capture_id": [c_void_p],
    "da_gemm_dk_splitk": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                          c_int, c_void_p, c_int, c_int, c_float, c_void_p, c_void_p, c_int, c_void_p],
    "da_decode_attn": [c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_int,
                       c_int, c_int, c_int, c_float, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p,
                       c_int, c_void_p],
    "da_topk_dense": [c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_void_p, c_int, c_float, c_int,
                      c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p],
    "da_topk_dense_stream": [c_void_p, c_int, c_int, c_void_p, c_void_p, c_int, c_void_p, c_int, c_float, c_int,
                             c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p],
    "da_topk_ranges": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int,
                       c_float, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_void_p, c_int,
                       c_void_p, c_void_p],
    "da_topk_merge": [c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p, c_int, c_void_p],
    "da_gather_ids": [c_void_p, c_int, c_void_p, c_int, c_void_p, c_void_p],
    "da_kmeans_accum": [c_void_p, c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p],
    "da_sample_partial": [c_void_p, c_int, c_int, c_int, c_int, c_float, c_uint, c_uint, c_void_p, c_void_p, c_void_p],
    "da_sample_chunked": [c_void_p, c_int, c_int, c_int, c_float, c_uint, c_uint] + [c_void_p] * 10
                         + [c_int] * 6 + [c_void_p],
    "da_sample_finalize": [c_void_p, c_int, c_int] + [c_void_p] * 8 + [c_int] * 5 + [c_void_p],
    "da_stream_create_cumask": [c_uint, ctypes.POINTER(c_uint), ctypes.POINTER(c_void_p)],
    "da_stream_get_cumask": [c_void_p, c_uint, ctypes.POINTER(c_uint)],
    "da_stream_destroy": [c_void_p],
    "da_device_cu_count": [c_int, ctypes.POINTER(c_int)],
    "da_placement_probe": [c_void_p, c_int, c_longlong, c_void_p],
    "da_spin": [c_int, c_void_p, c_void_p],
    "da_gemm8p_persist": [c_int],
    "da_gemm4w_variant": [c_int],
    "da_gemm_f16": [c_void_p, c_int, c_void_p, c_void_p, c_int, c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_int,
                    c_int, c_int, c_void_p, c_void_p, c_void_p, c_void_p],
    "da_flash_attn_f16": [c_void_p, c_void_p, c_void_p, c_int, c_int, c_int, c_void_p, c_int, c_int, c_int, c_int,
                          c_int, c_int, c_float, c_void_p, c_int, c_void_p],
    "da_layernorm_f16": [c_void_p, c_void_p, c_void_p, c_void_p, c_void_p, c_int, c_int, c_float, c_void_p],
    "da_bert_embed_ln_f16": [c_void_p] * 9 + [c_int, c_int, c_float, c_void_p],
    "da_pool_l2norm_f16": [c_void_p, c_void_p, c_int, c_int, c_int, c_int, c_void_p, c_void_p, c_void_p],
    "da_topk_dense_ws": [c_int] * 4,
    "da_topk_stream_ws": [c_int] * 4,
}
# the library part (build.py) of each launcher that is not in "kernels"; da_gemm* are in "gemm"
_PART_OF = {n: "token" for n in (
    "da_quant_fp8_rows", "da_rmsnorm", "da_swiglu_interleaved", "da_layernorm", "da_layernorm_q", "da_layernorm_f16",
    "da_bert_embed_ln", "da_bert_embed_ln_q", "da_bert_embed_ln_f16", "da_embed", "da_pool_l2norm", "da_pool_l2norm_f16",
    "da_rope_cache", "da_sample", "da_sample_partial", "da_sample_chunked", "da_sample_finalize")}


class KernelLibraryMissing(RuntimeError):
    pass


class KernelError(RuntimeError):
    pass


class _Kernels:
    """The launchers of every part; a part is built (if its sources are newer) and loaded at the first
    use of one of its launchers."""

    def __getattr__(self, name: str):
        if not name.startswith("da_"):
            raise AttributeError(name)
        load_part(_part_of(name))
        return self.__dict__.get(name) or getattr(_LOADED[_part_of(name)], name)


_LIB = _Kernels()
_LOADED: dict[str, ctypes.CDLL] = {}


def _part_of(name: str) -> str:
    return _PART_OF.get(name) or ("gemm" if name.startswith("da_gemm") else "kernels")


def load_part(part: str) -> None:
    with _LOCK:
        if part in _LOADED:
            return
        from .build import build, lib_path
        path = _LIB_OVERRIDE or lib_path(part, _DEBUG)
        if _LIB_OVERRIDE is None and os.environ.get("DA_BUILD_ON_IMPORT", "1") == "1":
            try:
                build(debug=_DEBUG, parts=(part,))
            except Exception as e:  # noqa: BLE001 - fall through to the explicit check below
                if not path.exists():
                    raise KernelLibraryMissing(f"cannot build {path}: {e}") from e
        if not path.exists():
            raise KernelLibraryMissing(f"{path} not built; run python -m docagents_amd.ops.build")
        import torch.cuda  # noqa: F401 - make sure torch's HIP runtime is loaded first
        L = ctypes.CDLL(str(path))
        for name, argt in _SIGS.items():
            if _part_of(name) == part:
                fn = getattr(L, name)
                fn.argtypes = argt
                fn.restype = c_size_t if name.endswith(("_ws", "_capture_id")) else c_int
                _LIB.__dict__[name] = fn
        _LOADED[part] = L


def lib(parts=()) -> _Kernels:
    """The kernel launchers; ``parts`` are loaded now, any other at the first use of its launchers."""
    for p in parts:
        if p not in _LOADED:
            load_part(p)
    return _LIB


@functools.lru_cache(maxsize=None)
def _address(name: str) -> int:
    """A launcher's address, for native code that calls it (its library stays loaded)."""
    return ctypes.cast(getattr(lib(), name), c_void_p).value


def available() -> bool:
    from .build import PARTS, lib_path
    return torch.cuda.is_available() and all(lib_path(p, _DEBUG).exists() for p in PARTS)


def _ptr(t):
    return None if t is None else ctypes.c_void_p(t.data_ptr())


def _raw_stream() -> int:
    """The calling thread's current stream on its current device. (torch.cuda.current_stream() builds a stream object around the
    same number: 2.8 us of the 8 that a launch took the host; this takes 0.2.)"""
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _stream():
    return ctypes.c_void_p(_raw_stream())


def _at(t):
    """``_ptr`` as a number (which the launchers' argument types take as well, 0.2 us sooner)."""
    return None if t is None else t.data_ptr()


def _check(rc: int, name: str):
    if rc != 0:
        raise KernelError(f"{name} failed with hipError {rc}")


def _req(cond: bool, msg: str):
    if not cond:
        raise ValueError(msg)


def _bf16_cuda(t, name):
    _req(t.is_cuda, f"{name} must be on GPU")
    _req(t.dtype == torch.bfloat16, f"{name} must be bf16, got {t.dtype}")


def _i32(t, name):
    _req(t.is_cuda and t.dtype == torch.int32 and t.is_contiguous(), f"{name} must be contiguous int32 on GPU")


# ----------------------------------------------------------------------------------- GEMM
_WS = {}
_ROLE = threading.local()


@contextlib.contextmanager
def workspace_role(name: str):
    """Kernels launched inside this context use the split-K / decode workspace of ``name``
    instead of the default one. Two phases that run CONCURRENTLY on different streams (the
    serving pipeline's prefill lane next to a replaying decode graph) must not share scratch:
    the decode graph captured the default workspace's pointer."""
    prev = getattr(_ROLE, "name", "main")
    _ROLE.name = name
    try:
        yield
    finally:
        _ROLE.name = prev


def workspace_buffer(device):
    """The current role's workspace tensor on ``device`` (None before its first use): callers that
    capture graphs check it is the same object after their captures (a grown workspace frees the
    buffer earlier captures point at)."""
    device = torch.device(device)
    key = (device.index if device.index is not None else torch.cuda.current_device(), getattr(_ROLE, "name", "main"))
    return _WS.get(key)


def _workspace(nbytes: int, device) -> torch.Tensor:
    key = (device.index if device.index is not None else torch.cuda.current_device(), getattr(_ROLE, "name", "main"))
    buf = _WS.get(key)
    if buf is None or buf.numel() < nbytes:
        buf = torch.empty(max(nbytes, 1 << 20), dtype=torch.uint8, device=device)
        _WS[key] = buf
    return buf


# The prefill products' shared last round (csrc/gemm8p.hip, TAIL) needs fp32 partials, up to 64 MB, and its tiles' counters,
# 8 KB that are zero between launches. The partials are the call's own: the caching allocator hands a stream the same block
# for each product and has it back in between. The counters stay, so that no launch has to clear them: a set per stream
# (streams run products beside each other) for the TAIL_STREAMS latest streams, and in a capture one per capture and
# stream, cleared by a node in front of its first such product.
TAIL_STREAMS = 32
N_COUNTERS = 256 * 8  # of a set
TAIL_MIN_K = 1024  # no round of a shorter product is shared (csrc/gemm8p.hip, tail_slices)
_TAIL: dict = {}  # (device, stream) -> counters, oldest first
_TAIL_CAPTURED: dict = {}  # (device, stream) -> (capture, counters): kept until the stream's next capture


@_rule
def _tail_bytes(M: int, N: int, K: int, epi: int, tile: int) -> int:
    return lib().da_gemm_tail_ws(M, N, K, epi, tile)


def _gemm_tail(device, stream: int, M: int, N: int, K: int, epi: int, tile: int = 0):
    """(partials, counters) of a product on the current stream ``stream`` whose last round is shared, (None, None) of
    others; the caller holds them until it is launched. A set of counters that makes room for another stream's goes back to
    the allocator, which keeps it for the stream that used it: in order."""
    nbytes = _tail_bytes(M, N, K, epi, tile) if K >= TAIL_MIN_K else 0
    if not nbytes:
        return None, None
    return torch.empty(nbytes // 4, dtype=torch.float32, device=device), _counters(device, stream)


def _counters(device, stream: int):
    """The ``N_COUNTERS`` counters, 0 between launches, of the current stream ``stream``."""
    key = (device.index, stream)
    if torch.cuda.is_current_stream_capturing():
        capture = lib().da_gemm_capture_id(stream)
        had, cnt = _TAIL_CAPTURED.get(key, (0, None))
        if had != capture:
            cnt = torch.zeros(N_COUNTERS, dtype=torch.int32, device=device)
            _TAIL_CAPTURED[key] = capture, cnt
        return cnt
    cnt = _TAIL.get(key)
    if cnt is None:
        cnt = torch.zeros(N_COUNTERS, dtype=torch.int32, device=device)
        with _LOCK:
            cnt = _TAIL.setdefault(key, cnt)
            while len(_TAIL) > TAIL_STREAMS:
                del _TAIL[next(iter(_TAIL))]
    return cnt


def _call_scratch(nbytes: int, like) -> torch.Tensor:
    """Scratch as the call's own, where ``like`` is, from the caching allocator (a capture's: from its graph's pool). The workspace of a role is
    one stream's, and one that grows drops the buffer that captured decode steps still write to: what may outgrow what a
    generator reserved (the scores or group maxima of a search, up to 67 MB) must not come from there."""
    return like.new_empty(-(-nbytes // like.element_size()))  # (0.7 us less than torch.empty with a type and a device)


def _call_partials(splits: int, M: int, N: int, like):
    """A product's K-split partials as the call's own: None if whole."""
    return _call_scratch(splits * M * N * 4, like) if splits > 1 else None


@_rule
def _row_choice(M: int, N: int, K: int, epi: int, lda: int, f16: bool = False):
    """(tile, splits) of a product of more than 64 rows (fp16: of any). A tile of ``_DK_TILES`` is da_gemm_dk_rows'."""
    if max(K, lda) < 1 << 22:
        tile = _dk_rows_tile(M, N, K, epi, f16)
        if tile:
            return tile, 1
        if _row_tiles_ok(M, N):
            return _row_tile(M, N, K, epi, f16)
    if f16 or M >= 640:
        return 0, 1
    return 11, _auto_splits(M, N, K)  # rows too long for the streaming tiles' offsets: the register-staged 64x128 tile


def _has_tail(M: int, tile: int, f16: bool = False) -> bool:
    """Whether a product runs on the kernels whose last round may be shared (gemm8p's rows and tiles)."""
    return tile in (7, 10) or (tile == 4 and not f16) or (tile == 0 and M >= (256 if f16 else 640))


def gemv_fusable(M: int, N: int, K: int, epi: int = EPI_NONE) -> bool:
    """True when gemm() runs the batch-1 GEMV (which can also fuse the input RMSNorm)."""
    return M == 1 and K % 512 == 0 and N % 4 == 0 and (epi not in GATED or N % 32 == 0)


def gemm(a: torch.Tensor, w: torch.Tensor, bias=None, epi: int = EPI_NONE, resid=None, out=None,
         tile: int = 0, splits: int = 0, rms=None) -> torch.Tensor:
    """out[M, N'] = epi(a[M, K] @ w[N, K]^T). N' = N/2 for EPI_SWIGLU (w rows interleaved by 16).
    rms = (gamma, eps): ``a`` is the raw residual stream and RMSNorm(a) * gamma is fused into the
    GEMV (M == 1 only, see gemv_fusable); gamma None = unit gain (folded into ``w``)."""
    _bf16_cuda(a, "a"); _bf16_cuda(w, "w")
    _req(a.dim() == 2 and w.dim() == 2, "gemm expects 2-D operands")
    M, K = a.shape
    N, K2 = w.shape
    _req(K == K2, f"K mismatch {K} vs {K2}")
    _req(K % 64 == 0, f"K={K} must be a multiple of 64")
    _req(N % 8 == 0, f"N={N} must be a multiple of 8")
    _req(a.stride(1) == 1 and a.stride(0) % 8 == 0 and a.stride(0) >= K, "a must be row-major, 16-B aligned rows")
    _req(w.is_contiguous(), "w must be contiguous")
    _req(a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0, "operands must be 16-B aligned")
    nout = N // 2 if epi in GATED else N
    if epi in GATED:
        _req(N % 32 == 0, "SwiGLU needs N % 32 == 0")
    if out is None:
        out = torch.empty((M, nout), dtype=torch.bfloat16, device=a.device)
    _bf16_cuda(out, "out")
    _req(out.shape == (M, nout) and out.stride(1) == 1 and out.stride(0) % 8 == 0, "bad out")
    if bias is not None:
        _bf16_cuda(bias, "bias"); _req(bias.numel() == N and bias.is_contiguous(), "bias must be [N]")
        _req(epi in (EPI_BIAS, EPI_GELU, EPI_RESID, *GATED), "bias only with BIAS/GELU/RESID/gated epilogues")
    ldr = 0
    if epi == EPI_RESID:
        _req(resid is not None, "EPI_RESID needs resid")
        _bf16_cuda(resid, "resid")
        _req(resid.shape == (M, N) and resid.stride(1) == 1 and resid.stride(0) % 8 == 0, "bad resid")
        ldr = resid.stride(0)
    if M == 0:
        return out
    if (tile == 12 or (tile == 0 and splits <= 0)) and rms is None and dk_fusable(M, N, K, epi):
        return gemm_dk(a, w, epi=epi, bias=bias, resid=resid, out=out)
    ws = None
    if tile == 0 and splits <= 0 and rms is None and M > 64:
        tile, splits = _row_choice(M, N, K, epi, a.stride(0))
        ws = _call_partials(splits, M, N, a)
    if tile in _DK_TILES:
        _req(rms is None and splits <= 1, "gemm_dk rows: whole, without a norm")
        return _gemm_dk_rows(a, w, bias, epi, resid, out, tile)
    if tile == 0 and splits <= 0 and gemv_fusable(M, N, K, epi):
        tile, splits = 6, 1  # batch-1 decode: weight-streaming GEMV, one launch, no split-K workspace
    gamma, eps = (None, 0.0) if rms is None else rms  # rms = (gain or None for unit gain, eps > 0)
    if rms is not None:
        _req(tile == 6, "fused RMSNorm needs the M == 1 GEMV path")
        _req(eps > 0, "fused RMSNorm needs eps > 0")
        if gamma is not None:
            _bf16_cuda(gamma, "gamma"); _req(gamma.numel() == K, "gamma must be [K]")
    if splits <= 0:
        if tile == 0 and M < 640:
            tile = _decode_tile(M)
        splits = _auto_splits(M, N, K) if tile in (0, 2, 3) or (tile == 9 and M <= 128) else 1
    if splits > 1 and ws is None:
        ws = _workspace(splits * M * N * 4, a.device)
    stream = _raw_stream()
    tail = _gemm_tail(a.device, stream, M, N, K, epi, tile) if _has_tail(M, tile) else (None, None)
    rc = lib().da_gemm_bf16(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), _ptr(bias), _ptr(resid), ldr,
                            M, N, K, epi, tile, splits, _ptr(ws), _ptr(gamma), float(eps), *map(_ptr, tail), c_void_p(stream))
    _check(rc, "gemm")
    return out


# Decode GEMMs with 2..64 rows: gemm_dk (csrc/gemm_dk.hip: K-steps dealt out to the 4 waves of a
# workgroup and summed through LDS; one launch, also where workgroups share K). False: the 64x128 /
# 32x128 tiles + split-K + reduce (bench/ab_arms.py DA_DECODE_DK=0).
DECODE_DK = True
# 33..64 rows keep the gemm_dk layer structure (norms deferred into the consumer); what ``_dk_whole`` does
# not take, and residuals with row sums, run on the streaming tiles (da_gemm_dk_splitk: reduce + residual
# + row sums of squares; the consumer's reduce or epilogue applies the row scale): a dk tile reads the
# activations once per 16-64 weight rows
DK_MAX_M = 64
DK_SPLITK_ABOVE = 32


def dk_fusable(M: int, N: int, K: int, epi: int = EPI_NONE) -> bool:
    """True when gemm() runs a decode-sized product on gemm_dk."""
    return (DECODE_DK and 2 <= M <= DK_MAX_M and K % 256 == 0 and N % 16 == 0
            and epi in (EPI_NONE, EPI_BIAS, EPI_RESID, *GATED) and (epi not in GATED or N % 32 == 0))


def dk_wide(M: int, N: int, K: int, lda: int) -> bool:
    """Products of up to 32 rows and more than 8192 columns, which the streaming tiles of csrc/gemm.hip cover the CUs with too."""
    return 1 <= M <= DK_SPLITK_ABOVE and N > 8192 and max(K, lda) <= 8192


def _dk_streams(M: int, N: int, K: int, lda: int) -> bool:
    """Products of more than 16384 columns on the streaming tiles of 128. More than 16 rows: the waves share a stage of A (28672 x 4096,
    32 rows: 40.6 us, 41.2 on gemm_dk; 16384 x 3072, 32 rows: 19.7 and 19.0). Of fewer where one tile a CU covers the columns in a round
    that is less than 7/8 full (gemm_dk's second workgroup of a CU then has nothing beside it), or where most of two rounds is, and
    short products of many. us, streaming / gemm_dk: 17920 x 5120 37 / 41, 17600 x 6144 44 / 49, 25344 x 6912 56 / 59, 50016 x
    4096 64 / 69, 50304 x 2048 35.3 / 36.8, 65472 x 512 14.2 / 15.2, 150688 x 768 37.3 / 40.3; not 28672 x 4096 (37.3 / 37.0), 30976 x 256
    (7.5 / 7.1), 32064 x 3072 (32.3 / 31.2), 41504 x 3584 (57.8 / 48.0), 70464 x 1280 (38.4 / 34.0) or 128256 x 4096 (153 / 149). Of 303
    such products it takes the slower way by more than 3 % at three, by 4.4 % at most (58688 x 2048 39.0 / 37.4)."""
    if N <= 16384 or not dk_wide(M, N, K, lda):
        return False
    if M > 16 or N < 28672:
        return M > 16 or 32 * K > N
    return N > 49152 and (N <= 61440 or K <= (1024 if N > 81920 else 512))


def _dk_whole(M: int, N: int, K: int, epi: int = EPI_NONE, norm: bool = False) -> bool:
    """33..64 rows that one gemm_dk launch runs faster than streaming tiles (with split-K and a reduce up to 8192 columns): up to
    16384 columns while K is short, as a workgroup reads all of A. us at 48 / 64 rows, tiles -> gemm_dk: 6144 x 4096
    17.1 / 18.5 -> 15.2 / 16.7, 8192 x 4096 20.2 / 21.7 -> 16.2 / 17.7, 9216 x 3072 21.4 / 21.6 -> 16.4 / 18.1, 12608 x 4096
    25.1 / 26.7 -> 22.6 / 24.8; 3072 x 8192 17.5 / 19.0 -> 19.5 / 21.9. Not 1024 columns and fewer of many rows and a K that eight
    splits and more share (few workgroups walk all of it): 64 x 128 x 4096 9.2 -> 11.6, 58 x 768 x 4096 10.5 -> 12.0, 56 x 288 x 3584
    10.0 -> 11.1; but 36 x 288 x 3840 10.1 -> 10.0, 57 x 256 x 3328 (four splits) 12.7 -> 10.7. The norm's row sums cost the reduce more."""
    if N <= 1024 and epi not in GATED and M * K > (235_000 if norm else 160_000) and _dk_splits(N, K) >= 8:
        return False
    return N <= 16384 and K <= 4096


@_rule
def _dk_split(M: int, N: int, K: int, epi: int):
    """(16-column groups of a tile, workgroups that share its K, bytes of their sums) of 2..32 rows on gemm_dk, zeros: K whole
    (both measured: csrc/gemm_dk.hip). Columns in whole 64s, not gated. From 17 rows on up to 8192 columns where K is at least 2.5 N and
    3072; of fewer rows, whose workgroups read little of A, up to 2048 columns where K is at least 4 N (up to 8 rows 16 N) and 4096."""
    if epi not in (EPI_NONE, EPI_BIAS, EPI_RESID) or N % 64 or not 1 < M <= 32:
        return 0, 0, 0
    if not (2 * K >= 5 * N and K >= 3072 and N <= 8192 if M > 16 else K >= (4 if M > 8 else 16) * N and K >= 4096 and N <= 2048):
        return 0, 0, 0
    fn = 1 if N < 1024 else 2 if N < 3072 else 4
    splits = min(256 // (N // (16 * fn)), 6 if fn == 4 else 4)
    return fn, splits, int(lib().da_gemm_dk_ws(N, fn, splits))


def _dk_splitk(M: int, N: int) -> bool:
    return DK_SPLITK_ABOVE < M <= 64 and N % 512 == 0


@_rule
def _dk_splits(N: int, K: int, reduce: bool = False) -> int:
    """Split-K of the 33..64-row route (64x128 tiles): the largest of 2, 3, 4, 6, 8, 12, 16 that keeps
    the grid within one round of 256 workgroups and >= 4 K-steps of 64 per split. 3 is the point of this
    list: the Phi-3 QKV projection (72 tiles) 18.7 us at 3 splits vs 21.8 at 2 and 25.7 at 4
    (bench/splitk_m64.py, profiles/r3/splitk_m64.txt). None above N = 8192 (to K = 8192): the streaming
    tile (64 wide to N = 16384) reaches HBM's rate on the CUs that it fills without, and the reduce launch
    goes (64 rows, N = 17920, K = 5120: 49 us vs 59 at 2; 28672 x 4096: 48 vs 60; 12672 x 4096: 29 vs 33;
    9216 x 3072: 21.2 vs 23.1 at 3; below the line 8192 x 4096: 25.0 vs 22.8 at 4); with a longer K two
    128-wide splits move half of A and are faster (12288 x 8192: 45.1 vs 47.2 at 2, x 14336: 86.6 vs 71.7).
    reduce: at least 2 (row sums of squares are written there)."""
    tiles, ks = (N + 127) // 128, K // 64
    best = 2 if reduce else 1
    if not reduce and N > 8192 and K <= 8192:
        return 1
    for s in (2, 3, 4, 6, 8, 12, 16):
        if ks % s == 0 and ks // s >= 4 and tiles * s <= 256:
            best = s
    return best if ks % best == 0 else 2


def dk_parts(N: int, M: int = 0) -> int:
    """Row-norm partial sums an EPI_RESID gemm_dk of width N and M rows writes (the consumer's part
    count): one per dk output tile, or one per 512 columns on the 33..64-row split-K route."""
    if _dk_splitk(M, N):
        return N // 512
    return int(lib().da_gemm_dk_parts(N))


def gemm_dk(a, w, epi: int = EPI_NONE, bias=None, resid=None, out=None, norm_in=None, ssq_out=None):
    """Decode-sized product (1 <= M <= 64), in one launch but for what streams in splits:
    out = epi(rownorm(a) @ w^T). norm_in = (ssq, parts, eps): ``a`` is the raw residual stream and
    each row's sums are scaled by rsqrt(sum of ssq[:parts, row] / K + eps) (RMSNorm gains folded into w). ssq_out (EPI_RESID only): fp32
    [dk_parts(N), 64] receives the per-part sums of squares of the new rows, for the next consumer."""
    _bf16_cuda(a, "a"); _bf16_cuda(w, "w")
    M, K = a.shape
    N = w.shape[0]
    _req(1 <= M <= 64 and K % 256 == 0 and N % 16 == 0 and w.shape[1] == K, f"gemm_dk shape M={M} N={N} K={K}")
    _req(a.stride(1) == 1 and a.stride(0) % 8 == 0 and w.is_contiguous(), "gemm_dk layout")
    _req(a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0, "operands must be 16-B aligned")
    nout = N // 2 if epi in GATED else N
    if out is None:
        out = torch.empty((M, nout), dtype=torch.bfloat16, device=a.device)
    _req(out.shape == (M, nout) and out.stride(1) == 1 and out.stride(0) % 8 == 0, "bad out")
    ldr = 0
    if epi == EPI_RESID:
        _req(resid is not None and resid.shape == (M, N) and resid.stride(1) == 1 and resid.stride(0) % 8 == 0,
             "bad resid")
        ldr = resid.stride(0)
    ssq, parts, eps = (None, 0, 0.0) if norm_in is None else norm_in
    if ssq is not None:
        _req(ssq.dtype == torch.float32 and ssq.is_contiguous() and ssq.numel() >= parts * 64, "bad ssq_in")
    if ssq_out is not None:
        _req(epi == EPI_RESID and ssq_out.dtype == torch.float32 and ssq_out.is_contiguous()
             and ssq_out.numel() >= dk_parts(N, M) * 64, "bad ssq_out")
    if _dk_streams(M, N, K, a.stride(0)) and ssq_out is None:
        _check(lib().da_gemm_dk_splitk(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), _ptr(bias), _ptr(resid),
                                       ldr, M, N, K, epi, _ptr(ssq), parts, K, float(eps), None, None, 1, _stream()), "gemm_dk_wide")
        return out
    far = max(K, a.stride(0)) >= 1 << 22  # rows too long for 32-bit offsets within a tile: the reduce carries the epilogue
    if (_dk_splitk(M, N) and ssq_out is not None) or (ssq_out is None and (far or (M > DK_SPLITK_ABOVE and not _dk_whole(M, N, K, epi, ssq is not None)))):
        splits = _dk_splits(N, K, ssq_out is not None or far)
        ws = _workspace(splits * M * N * 4, a.device) if splits > 1 else None
        _check(lib().da_gemm_dk_splitk(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), _ptr(bias), _ptr(resid),
                                       ldr, M, N, K, epi, _ptr(ssq), parts, K, float(eps), _ptr(ssq_out), _ptr(ws),
                                       splits, _stream()), "gemm_dk_splitk")
        return out
    stream, ws, cnt = _raw_stream(), None, None
    fn, splits, nbytes = _dk_split(M, N, K, epi) if ssq is None else (0, 0, 0)
    if splits:
        ws, cnt = _call_scratch(nbytes, a), _counters(a.device, stream)
    _check(lib().da_gemm_dk(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), _ptr(bias), _ptr(resid), ldr,
                            M, N, K, epi, _ptr(ssq), parts, K, float(eps), _ptr(ssq_out), fn, splits, _ptr(ws), _ptr(cnt),
                            c_void_p(stream)), "gemm_dk")
    return out


def dk_rope_fits(M: int, N: int, K: int, lda: int) -> bool:
    """Whether ``gemm_dk_rope`` takes a QKV projection that gemm_dk runs as one plain launch."""
    return (dk_fusable(M, N, K) and max(K, lda) < 1 << 22 and not _dk_streams(M, N, K, lda) and not _dk_split(M, N, K, EPI_NONE)[1]
            and (M <= DK_SPLITK_ABOVE or _dk_whole(M, N, K, EPI_NONE, True)))


def gemm_dk_rope(a, w, pos, cos_sin, H: int, Hkv: int, D: int, slot, k_cache, v_cache, norm_in=None, out=None, kv_out: bool = True):
    """gemm_dk of a QKV projection with the q / k heads rotated and k / v written to the cache, in one launch (``dk_rope_fits``): the
    same values as the product and ``rope_cache`` behind it. norm_in as gemm_dk's, kv_out as gemm_rope's."""
    _bf16_cuda(a, "a"); _bf16_cuda(w, "w"); _i32(pos, "pos"); _i32(slot, "slot")
    M, K = a.shape
    N = w.shape[0]
    _req(dk_rope_fits(M, N, K, a.stride(0)) and w.shape[1] == K and N == (H + 2 * Hkv) * D and D % 8 == 0, f"gemm_dk_rope shape M={M} N={N} K={K}")
    _req(a.stride(1) == 1 and a.stride(0) % 8 == 0 and w.is_contiguous(), "gemm_dk_rope layout")
    _req(a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0, "operands must be 16-B aligned")
    _req(pos.numel() >= M and slot.numel() >= M, "pos / slot length")
    _req(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous() and cos_sin.shape[-1] == 2 and cos_sin.shape[1] == D // 2, "cos_sin")
    _req(k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape == v_cache.shape
         and k_cache.dim() == 4 and k_cache.shape[1] == Hkv and k_cache.shape[3] == D, "caches")
    if out is None:
        out = torch.empty((M, N), dtype=torch.bfloat16, device=a.device)
    _bf16_cuda(out, "out")
    _req(out.shape == (M, N) and out.stride(1) == 1 and out.stride(0) % 8 == 0 and out.data_ptr() % 16 == 0, "bad out")
    ssq, parts, eps = (None, 0, 0.0) if norm_in is None else norm_in
    if ssq is not None:
        _req(ssq.dtype == torch.float32 and ssq.is_contiguous() and ssq.numel() >= parts * 64, "bad ssq_in")
    _check(lib().da_gemm_dk_rope(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), M, N, K, _ptr(ssq), parts, K, float(eps),
                                 _ptr(pos), _ptr(slot), _ptr(cos_sin), _ptr(k_cache), _ptr(v_cache), H, Hkv, D, k_cache.shape[2],
                                 int(kv_out), _stream()), "gemm_dk_rope")
    return out


def gemm_ln_fit(M: int, hidden: int, ffn: int) -> bool:
    """Whether an encoder layer's products take ``gemm_ln`` (csrc/encoder_rows.hip)."""
    return 1 <= M <= 64 and hidden % 64 == 0 and ffn % 64 == 0 and hidden <= 1024


def attn_ln_fit(M: int, hidden: int, heads: int, texts: int, f16: bool = False) -> bool:
    """Whether ``gemm_ln`` takes attention inside (``attn``) where an encoder's products take it: one short text of an encoder that ``enc_text``
    refuses (fewer than ENC_TEXT_MIN_LAYERS layers, where it is the faster way, more than 32, a feed-forward of more than 4096 columns)."""
    return M <= (32 if hidden > 384 else 64) and hidden <= 1024 and hidden in ((64 * heads,) if f16 else (32 * heads, 64 * heads)) and texts == 1


def gemm_ln(a, w, bias, epi: int = EPI_BIAS, norm=None, resid=None, st_out=None, attn=None):
    """bf16 or fp16 products of up to 64 rows between LayerNorms. norm = (st, g, b, eps): the rows of ``a`` (EPI_BIAS, EPI_GELU) or
    of ``resid`` (EPI_RESID) are sums whose LayerNorm is taken here, by the statistics st (fp32 [64, 64, 2]) that the
    EPI_RESID product which made them wrote as its ``st_out``. attn = (heads, cu_seqlens) (EPI_RESID, ``attn_ln_fit``):
    ``a`` holds q, k and v, and the product is that of their attention's output."""
    f16 = a.dtype == torch.float16
    is_cuda = _f16_cuda if f16 else _bf16_cuda
    is_cuda(a, "a"); is_cuda(w, "w"); is_cuda(bias, "bias")
    M, K = a.shape
    if attn is not None:
        heads, cu = attn
        _i32(cu, "cu_seqlens")
        _req(K % 3 == 0 and attn_ln_fit(M, K // 3, heads, cu.numel() - 1, f16) and epi == EPI_RESID, "gemm_ln attention")
        K //= 3
    N = w.shape[0]
    _req(gemm_ln_fit(M, K if epi != EPI_RESID else N, N if epi != EPI_RESID else K) and w.shape[1] == K
         and bias.shape == (N,) and bias.is_contiguous(), f"gemm_ln shape M={M} N={N} K={K}")
    _req(a.stride(1) == 1 and a.stride(0) % 8 == 0 and a.data_ptr() % 16 == 0 and w.is_contiguous()
         and w.data_ptr() % 16 == 0, "gemm_ln layout")
    _req(epi == EPI_BIAS or (epi == EPI_GELU and norm is not None) or (epi == EPI_RESID and st_out is not None),
         "gemm_ln epilogue")
    st, g, b, eps = norm or (None, None, None, 0.0)
    for t in (st, st_out):
        _req(t is None or (t.is_cuda and t.dtype == torch.float32 and t.shape == (64, 64, 2) and t.is_contiguous()),
             "bad statistics")
    if norm is not None:
        for t in (g, b):
            is_cuda(t, "norm")
            _req(t.shape == (N if epi == EPI_RESID else K,) and t.is_contiguous(), "norm must be [columns]")
    if epi == EPI_RESID:
        is_cuda(resid, "resid")
        _req(resid.shape == (M, N) and resid.stride(1) == 1 and resid.stride(0) % 8 == 0, "bad resid")
    out = torch.empty((M, N), dtype=a.dtype, device=a.device)
    if attn is not None:
        D = K // heads
        _check(lib().da_enc_attn_rows(_ptr(a), a.stride(0), _ptr(w), _ptr(out), N, _ptr(bias), _ptr(resid), resid.stride(0), M, N, K,
                                     D, _ptr(cu), math.log2(math.e) / math.sqrt(D), _ptr(st), _ptr(g), _ptr(b),
                                     float(eps), _ptr(st_out), f16, _stream()), "gemm_ln")
        return out
    _check(lib().da_enc_rows(_ptr(a), a.stride(0), _ptr(w), _ptr(out), N, _ptr(bias), _ptr(resid),
                            0 if resid is None else resid.stride(0), M, N, K, epi, _ptr(st), _ptr(g), _ptr(b), float(eps),
                            _ptr(st_out), f16, _stream()), "gemm_ln")
    return out


ENC_TEXT_MIN_LAYERS = 4  # (two: 42 us for 48 of launches one by one; 4: 69 for 94)


def enc_text_fits(M: int, hidden: int, ffn: int, layers: int, heads: int, texts: int, f16: bool = False) -> bool:
    """Whether ``enc_text`` takes the layers of an encoder."""
    return (1 <= M <= 64 and ENC_TEXT_MIN_LAYERS <= layers <= 32 and hidden % 64 == 0 and hidden <= 1024 and ffn % 64 == 0 and 64 <= ffn <= 4096
            and hidden in ((64 * heads,) if f16 else (32 * heads, 64 * heads)) and texts == 1)


TEXT_POLLS = 1 << 22  # readings of a wait in csrc/encoder_text.hip, of 1 us and more each


class TextWaits:
    """Where an encoder's ``enc_text`` launches say that a wait ran out (no order of their workgroups does that; the result is NaNs then): a
    pinned word of the host, which a reader sees once it has waited for the launch."""

    def __init__(self):
        self._word = torch.zeros(1, dtype=torch.int32, pin_memory=True)
        self._value, at = c_int.from_address(self._word.data_ptr()), c_void_p()
        _check(lib().da_host_address(self._word.data_ptr(), ctypes.byref(at)), "host_address")
        self.at, self.launches = at.value, 0
        self._lock, self._ran_out, self._told = threading.Lock(), 0, threading.local()

    def begin(self) -> None:
        """Before a launch."""
        self.check()
        with self._lock:
            self.launches += 1

    def check(self) -> None:
        """KernelError if a wait ran out in a launch that has run since this thread's last check (whose launch it was is not known: each thread
        that uses the encoder is told once)."""
        told = getattr(self._told, "n", None)
        if told is None:
            told = self._told.n = self._ran_out
        if self._value.value:
            with self._lock:
                self._ran_out += bool(self._value.value)
                self._value.value = 0
        if self._ran_out != told:
            self._told.n = self._ran_out
            raise KernelError("enc_text: a wait ran out, the text's embedding is NaNs")


def _text_layers(layers, h: int, f: int, is_cuda):
    """The layers' pointers (csrc/encoder_text.hip, TextLayer), and how many."""
    shapes = {"wqkv": (3 * h, h), "bqkv": (3 * h,), "wo": (h, h), "bo": (h,), "ln1_g": (h,), "ln1_b": (h,), "w1": (f, h), "b1": (f,),
              "w2": (h, f), "b2": (h,), "ln2_g": (h,), "ln2_b": (h,)}
    table = []
    for L in layers:
        for name, shape in shapes.items():
            t = L[name]
            is_cuda(t, name)
            _req(t.shape == shape and t.is_contiguous() and (t.dim() == 1 or t.data_ptr() % 16 == 0), f"enc_text {name}")
            table.append(t.data_ptr())
    return (c_void_p * len(table))(*table), len(layers)


def enc_text(x, layers, cu, heads: int, eps: float, waits: TextWaits | None = None):
    """All layers of one text of up to 64 rows in one launch (csrc/encoder_text.hip): x [M, h] -> the last layer's sum before
    its norm (rows behind the text: zeros). layers: dicts of wqkv, bqkv, wo, bo, ln1_g, ln1_b, w1, b1, w2, b2, ln2_g, ln2_b.
    waits: told of a wait that runs out, and asked first about the launches before."""
    if waits is not None:
        waits.begin()
    f16 = x.dtype == torch.float16
    is_cuda = _f16_cuda if f16 else _bf16_cuda
    is_cuda(x, "x"); _i32(cu, "cu_seqlens")
    M, h = x.shape
    f, D = layers[0]["w1"].shape[0], h // heads
    _req(enc_text_fits(M, h, f, len(layers), heads, cu.numel() - 1, f16) and x.is_contiguous() and x.data_ptr() % 16 == 0, "enc_text shape")
    table, n = _text_layers(layers, h, f, is_cuda)
    ws = torch.empty(int(lib().da_enc_text_ws(M, h, f, n, D, f16)), dtype=torch.uint8, device=x.device)
    out = torch.empty_like(x)
    _check(lib().da_enc_text(_ptr(x), table, n, _ptr(out), _ptr(ws), _ptr(cu), M, h, f, D, float(eps), math.log2(math.e) / math.sqrt(D), f16,
                             waits and waits.at, TEXT_POLLS, _stream()), "enc_text")
    return out


class TextPlan:
    """An encoder's weights (word, pos, type, emb_ln_g, emb_ln_b, layers) as ``enc_text_pooled`` takes them: the tensors, checked once. waits as ``enc_text``'s."""

    def __init__(self, w: dict, heads: int, eps: float, waits: TextWaits | None = None):
        self.waits, self.f16 = waits, w["word"].dtype == torch.float16
        is_cuda = _f16_cuda if self.f16 else _bf16_cuda
        self.emb, self.weights = [w[k] for k in ("word", "pos", "type", "emb_ln_g", "emb_ln_b")], w["layers"]
        self.h, self.f, self.D, self.eps = w["word"].shape[1], self.weights[0]["w1"].shape[0], w["word"].shape[1] // heads, float(eps)
        for t in self.emb:
            is_cuda(t, "embeddings")
            _req(t.shape[-1] == self.h and t.is_contiguous(), "TextPlan embeddings")
        _req(enc_text_fits(1, self.h, self.f, len(self.weights), heads, 1, self.f16), "TextPlan shape")
        self.weights = [dict(L) for L in self.weights]  # (kept as they are)
        self.table, self.n = _text_layers(self.weights, self.h, self.f, is_cuda)
        self.emb_table = (c_void_p * 5)(*(t.data_ptr() for t in self.emb))


def enc_text_pooled(plan: TextPlan, tokens, mode: int) -> torch.Tensor:
    """The whole encoder of one text of n <= 64 tokens, in three launches: the unit vector of its pooled rows (mode as pool_l2norm's),
    fp32 [1, h]. tokens int32 [2 n + 2]: ids, positions, 0 and n."""
    if plan.waits is not None:
        plan.waits.begin()
    _i32(tokens, "tokens")
    n, h = tokens.numel() // 2 - 1, plan.h
    _req(1 <= n <= 64 and tokens.numel() == 2 * n + 2 and tokens.device == plan.emb[0].device, "enc_text_pooled tokens")
    size, row = int(lib().da_enc_text_ws(n, h, plan.f, plan.n, plan.D, plan.f16)), n * h * 2
    ws = torch.empty(size + 2 * row, dtype=torch.uint8, device=tokens.device)
    out = torch.empty((1, h), dtype=torch.float32, device=tokens.device)
    at, t = ws.data_ptr(), tokens.data_ptr()
    _check(lib().da_enc_text_pooled(t, t + 4 * n, plan.emb_table, plan.table, plan.n, at + size, at + size + row, at, t + 8 * n, n, h, plan.f, plan.D,
                                    plan.eps, math.log2(math.e) / math.sqrt(plan.D), mode, out.data_ptr(), plan.f16,
                                    plan.waits and plan.waits.at, TEXT_POLLS, _raw_stream()), "enc_text_pooled")
    return out


# Every GEMM runs on the in-tree kernels: gemm8p (phase-split BMx256, csrc/gemm8p.hip) from 256
# rows, the 64x128 / 32x128 weight-streaming tiles + split-K below, the GEMV at batch 1. The
# vendor-library arms used for comparisons live in bench/ab_arms.py (same-box measurements:
# profiles/r2/ab_gemm8p_vs_hipblaslt.txt).


def gemm_rope(a, w, pos, cos_sin, H: int, Hkv: int, D: int, slot, k_cache, v_cache, out=None,
              kv_out: bool = True) -> torch.Tensor:
    """Prefill QKV projection: qkv = a @ w^T with RoPE applied to the q / k heads and the token's
    k / v written to the KV cache (cache [slots, Hkv, max_seq, D]) — one kernel (gemm8p EPI_ROPE)
    from 256 rows on, but where ``_rope_apart`` (and not ``_rope_round``); those and 65 - 255 rows run gemm + rope_cache (identical
    roundings). Fewer take that way too, where a decoder does not use ``gemm_dk_rope`` for them. kv_out=False: the
    k / v columns of the result may be left unwritten (the attention reads the cache; see
    flash_attn_varlen kv_cache) — only the q columns are defined."""
    _bf16_cuda(a, "a"); _bf16_cuda(w, "w"); _i32(pos, "pos"); _i32(slot, "slot")
    M, K = a.shape
    N = w.shape[0]
    _req(N == (H + 2 * Hkv) * D and w.shape[1] == K and D % 8 == 0, "qkv weight shape")
    _req(pos.numel() >= M and slot.numel() >= M, "pos / slot length")
    _req(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous() and cos_sin.shape[1] == D // 2, "cos_sin")
    _req(k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape == v_cache.shape
         and k_cache.dim() == 4 and k_cache.shape[1] == Hkv and k_cache.shape[3] == D, "caches")
    plain = K % 64 == 0 and K >= 128 and a.stride(1) == 1 and a.stride(0) % 8 == 0 and w.is_contiguous()
    # (what gemm and rope_cache refuse and the one kernel takes stays with that)
    apart = (a.data_ptr() % 16 == 0 and w.data_ptr() % 16 == 0 and a.stride(0) >= K and cos_sin.shape[-1] == 2
             and (out is None or out.is_contiguous()) and M >= 256 and _rope_apart(M, N, K) and not _rope_round(M, N))
    if M < 256 or not plain or apart:
        qkv = gemm(a, w, out=out)
        return rope_cache(qkv, pos, cos_sin, H, Hkv, D, slot=slot, k_cache=k_cache, v_cache=v_cache)
    if out is None:
        out = torch.empty((M, N), dtype=torch.bfloat16, device=a.device)
    _req(out.shape == (M, N) and out.stride(1) == 1 and out.stride(0) % 8 == 0, "bad out")
    _check(lib().da_gemm_rope(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), M, N, K, _ptr(pos), _ptr(slot),
                              _ptr(cos_sin), _ptr(k_cache), _ptr(v_cache), H, Hkv, D, k_cache.shape[2], int(kv_out),
                              _stream()),
           "gemm_rope")
    return out


FP8 = torch.float8_e4m3fn  # OCP e4m3 (gfx950), not the MI300 fnuz variant


def quant_fp8(x: torch.Tensor, out=None, scale=None):
    """Per-row dynamic e4m3 quantisation: returns (q [M, K] float8_e4m3fn, scale [M] fp32)."""
    _bf16_cuda(x, "x")
    _req(x.dim() == 2 and x.stride(1) == 1 and x.stride(0) % 8 == 0 and x.shape[1] % 8 == 0, "x layout")
    M, K = x.shape
    if out is None:
        out = torch.empty((M, K), dtype=FP8, device=x.device)
    if scale is None:
        scale = torch.empty(M, dtype=torch.float32, device=x.device)
    _req(out.dtype == FP8 and out.shape == (M, K) and out.stride(1) == 1 and out.stride(0) % 16 == 0, "bad out")
    _req(scale.dtype == torch.float32 and scale.numel() >= M, "bad scale")
    _check(lib().da_quant_fp8_rows(_ptr(x), x.stride(0), M, K, _ptr(out), out.stride(0), _ptr(scale), _stream()),
           "quant_fp8")
    return out, scale


def quant_weight_fp8(w: torch.Tensor):
    """Per-output-channel e4m3 weight quantisation (host-side torch; done once at load)."""
    wf = w.float()
    sw = (wf.abs().amax(dim=1) / 448.0).clamp_min(1e-30)
    return (wf / sw[:, None]).clamp(-448, 448).to(FP8).contiguous(), sw.contiguous()


class _EncoderProduct(ctypes.Structure):
    _fields_ = [(n, c_void_p) for n in ("ws", "tail_ws", "tail_cnt")] + [(n, c_int) for n in ("tile", "splits", "rows", "pad")]


_ENCODER_WEIGHTS = ("wqkv", "bqkv", "wo", "bo", "ln1_g", "ln1_b", "w1", "b1", "w2", "b2", "ln2_g", "ln2_b")


class _EncoderLayer(ctypes.Structure):
    _fields_ = ([(n, c_void_p) for n in ("gemm", "gemm_rows", "gemm_fp8", "attn", "norm")] + [("w", c_void_p * 14)]
                + [(n, c_void_p * 3) for n in ("x", "xq", "xscale")] + [("qkv", c_void_p), ("a", c_void_p), ("y", c_void_p * 2)]
                + [("f", c_void_p), ("cu", c_void_p)] + [("p", _EncoderProduct * 4)]
                + [(n, c_int) for n in ("kind", "T", "B", "max_len", "heads", "head_dim", "hidden", "ffn")]
                + [("eps", c_float), ("scale", c_float)])


def encoder_layers_fit(rows: int) -> bool:
    """Whether an encoder's layers take ``encoder_layers`` (fewer rows have products of their own, and captured graphs)."""
    return rows > 64


def _encoder_sets(rows: int, hidden: int, ffn: int) -> int:
    """Sets of buffers that an encoder's layers take in turn: two while both fit the dies' L2s (8 of 4 MB), one from there on. A kernel
    that writes over what all dies' caches have just read waits for them to give it up; where the buffers leave the L2s anyway, a
    second set only makes more of them leave. us of 12 layers, one / two: 512 rows of 384 columns, fp8 401 / 372, 1024 481 / 461, 256 of
    768 445 / 417, 24 layers of 1024, fp16, 128 995 / 963; 2000 of 384 646 / 644, 1000 of 768, bf16 738 / 734, 3000 1313 / 1456, 4000 1464 /
    1566, 12000 of 384 1580 / 1712, 8100 of 1024, fp8 5823 / 6013."""
    return 2 if rows * (8 * hidden + ffn) * 2 <= 16 << 20 else 1


def encoder_layers(x, layers, cu_seqlens, max_seqlen: int, heads: int, head_dim: int, eps: float, xq=None):
    """The layers of an encoder over x [T, hidden] (bf16, fp16; with xq = (e4m3 rows, scales) the fp8 products of
    ``gemm_fp8``) -> [T, hidden]: what gemm / gemm_f16 / gemm_fp8, the attention and the LayerNorms give one by one, with
    one native call a layer (csrc/encoder_layer.hip). ``layers``: each layer's weights by name."""
    f16, q8 = x.dtype == torch.float16, xq is not None
    (_f16_cuda if f16 else _bf16_cuda)(x, "x")
    _i32(cu_seqlens, "cu_seqlens")
    if not layers:
        return x
    T, h = x.shape
    ffn = layers[0]["w1"].shape[0]
    _req(T > 64 and x.is_contiguous() and x.data_ptr() % 16 == 0, "x [T, hidden], contiguous")
    _req(h == heads * head_dim and head_dim in ((64, 96) if f16 else (32, 64, 96, 128)), f"head dim {head_dim} unsupported")
    _req(h % (128 if q8 else 64) == 0 and ffn % 64 == 0 and (not f16 or min(h, ffn) >= 128), f"hidden {h}, feed-forward {ffn}")
    stream, L, dt = _raw_stream(), _EncoderLayer(), x.dtype
    new = lambda n: torch.empty((T, n), dtype=dt, device=x.device)  # noqa: E731
    sets = [{n: new(c) for n, c in (("qkv", 3 * h), ("a", h), ("y0", h), ("m", h), ("f", ffn), ("y1", h), ("x", h))}
            for _ in layers[:_encoder_sets(T, h, ffn)]]
    L.cu = cu_seqlens.data_ptr()
    if q8:
        _req(xq[0].dtype == FP8 and xq[0].shape == x.shape and xq[0].is_contiguous() and xq[0].data_ptr() % 16 == 0
             and xq[1].dtype == torch.float32 and xq[1].numel() >= T, "fp8 rows")
        L.gemm_fp8 = _address("da_gemm_fp8")
        for S in sets:
            for n in ("m8", "x8"):
                S[n] = (torch.empty((T, h), dtype=FP8, device=x.device), torch.empty(T, dtype=torch.float32, device=x.device))
    L.gemm, L.gemm_rows = _address("da_gemm_f16" if f16 else "da_gemm_bf16"), _address("da_gemm_dk_rows")
    L.attn = _address("da_flash_attn_f16" if f16 else "da_flash_attn_v2")
    L.norm = _address("da_layernorm_f16" if f16 else "da_layernorm_q" if q8 else "da_layernorm")
    L.kind, L.T, L.B, L.max_len = 1 if f16 else 2 if q8 else 0, T, cu_seqlens.numel() - 1, int(max_seqlen)
    L.heads, L.head_dim, L.hidden, L.ffn, L.eps, L.scale = heads, head_dim, h, ffn, float(eps), 1.0 / math.sqrt(head_dim)
    held = []  # (a product's partials and counters serve every layer: one after another on this stream)
    for p, (N, K, epi, fp8) in zip(L.p, ((3 * h, h, EPI_BIAS, q8), (h, h, EPI_RESID, False), (ffn, h, EPI_GELU, q8),
                                        (h, ffn, EPI_RESID, False))):
        if fp8:
            continue
        p.tile, p.splits = _row_choice(T, N, K, epi, K, f16)
        p.rows = p.tile in _DK_TILES
        if p.rows:
            continue
        ws = _call_partials(p.splits, T, N, x)
        tail = _gemm_tail(x.device, stream, T, N, K, epi, p.tile) if _has_tail(T, p.tile, f16) else (None, None)
        held.append((ws, tail))
        p.ws, p.tail_ws, p.tail_cnt = (None if t is None else t.data_ptr() for t in (ws, *tail))
    wide, square, up, down, row, row3, rowf = (3 * h, h), (h, h), (ffn, h), (h, ffn), (h,), (3 * h,), (ffn,)
    need = list(zip(_ENCODER_WEIGHTS, (wide, row3, square, row, row, row, up, rowf, down, row, row, row), (dt,) * 12))
    if q8:
        need[0], need[6] = ("wqkv_q", wide, FP8), ("w1_q", up, FP8)
        need += [("wqkv_s", row3, torch.float32), ("w1_s", rowf, torch.float32)]
    run, at = lib().da_encoder_layer, ctypes.byref(L)
    for n, layer in enumerate(layers):
        S = sets[n % len(sets)]
        L.qkv, L.a, L.f, L.y[:] = S["qkv"].data_ptr(), S["a"].data_ptr(), S["f"].data_ptr(), (S["y0"].data_ptr(), S["y1"].data_ptr())
        L.x[:] = [t.data_ptr() for t in (x, S["m"], S["x"])]
        if q8:
            (L.xq[:], L.xscale[:]) = zip(*(tuple(t.data_ptr() for t in p) for p in (xq, S["m8"], S["x8"])))
            xq = S["x8"]
        x = S["x"]
        for i, (name, shape, dtype) in enumerate(need):
            t = layer[name]
            p = t.data_ptr()
            if t.dtype is not dtype or t.shape != shape or not t.is_cuda or not t.is_contiguous() or (p % 16 and len(shape) == 2):
                _req(False, f"{name} must be {dtype} {list(shape)} on the GPU, contiguous and aligned")
            L.w[i] = p
        _check(run(at, EPI_BIAS, EPI_GELU, EPI_RESID, stream), "encoder_layer")
    return x


def gemm_fp8(aq, sa, wq, sw, bias=None, epi: int = EPI_NONE, resid=None, out=None) -> torch.Tensor:
    """out[M, N] = epi((aq . wq^T) * sa[:, None] * sw[None, :]) with e4m3 operands (MFMA tiles of 64, 128 or 256 squared)."""
    _req(aq.is_cuda and aq.dtype == FP8 and wq.dtype == FP8, "fp8 operands expected")
    M, K = aq.shape
    N, K2 = wq.shape
    _req(K == K2 and K % 128 == 0 and N % 8 == 0, f"fp8 gemm shape M={M} N={N} K={K}")
    _req(aq.stride(1) == 1 and aq.stride(0) % 16 == 0 and wq.is_contiguous(), "fp8 operand layout")
    _req(aq.data_ptr() % 16 == 0 and wq.data_ptr() % 16 == 0, "operands must be 16-B aligned")
    _req(sa.dtype == torch.float32 and sa.numel() >= M and sw.dtype == torch.float32 and sw.numel() == N, "scales")
    nout = N // 2 if epi == EPI_SWIGLU else N
    if out is None:
        out = torch.empty((M, nout), dtype=torch.bfloat16, device=aq.device)
    _bf16_cuda(out, "out")
    _req(out.shape == (M, nout) and out.stride(1) == 1 and out.stride(0) % 8 == 0, "bad out")
    if bias is not None:
        _bf16_cuda(bias, "bias"); _req(bias.numel() == N, "bias must be [N]")
    ldr = 0
    if epi == EPI_RESID:
        _req(resid is not None and resid.shape == (M, N) and resid.stride(1) == 1, "bad resid")
        ldr = resid.stride(0)
    if M == 0:
        return out
    _check(lib().da_gemm_fp8(_ptr(aq), aq.stride(0), _ptr(wq), _ptr(sa), _ptr(sw), _ptr(out), out.stride(0),
                             _ptr(bias), _ptr(resid), ldr, M, N, K, epi, _stream()), "gemm_fp8")
    return out


def gemm_resid_norm(a, w, resid, gamma, eps: float, out=None, h_out=None, bias=None, tile: int = 0, splits: int = 0):
    """Decode layer tail (M <= 128): out = resid + a @ w^T (+ bias) — the new residual stream — and
    h_out = RMSNorm(out) * gamma, with the norm fused into the split-K reduction. Returns h_out."""
    _bf16_cuda(a, "a"); _bf16_cuda(w, "w"); _bf16_cuda(resid, "resid"); _bf16_cuda(gamma, "gamma")
    M, K = a.shape
    N = w.shape[0]
    _req(M <= 128 and K % 64 == 0 and N % 8 == 0 and N <= 8192 and w.shape[1] == K, "gemm_resid_norm shape")
    _req(a.stride(1) == 1 and a.stride(0) % 8 == 0 and w.is_contiguous() and gamma.numel() == N, "layout")
    _req(resid.shape == (M, N) and resid.stride(1) == 1, "bad resid")
    out = resid if out is None else out
    if h_out is None:
        h_out = torch.empty((M, N), dtype=torch.bfloat16, device=a.device)
    if M == 0:
        return h_out
    tile = tile or (9 if M > 64 else _decode_tile(M))  # the fused reduce + norm: 128x64 tile above 64 rows
    if splits <= 0:
        splits = _auto_splits(M, N, K)
    ws = _workspace(splits * M * N * 4, a.device)
    _check(lib().da_gemm_resid_rmsnorm(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), _ptr(bias),
                                       _ptr(resid), resid.stride(0), M, N, K, tile, splits, _ptr(ws), _ptr(gamma),
                                       float(eps), _ptr(h_out), h_out.stride(0), _stream()), "gemm_resid_norm")
    return h_out


def _decode_tile(M: int) -> int:
    """The tile of up to 64 rows: 32x128 up to 32, else the weight-streaming tile (csrc/gemm.hip)."""
    return 3 if M <= 32 else 2


@_rule
def _auto_splits(M: int, N: int, K: int) -> int:
    """Split-K for decode-sized M. Up to 64 rows (without the exceptions below): the largest power of two
    keeping <= 256 workgroups (one per CU) and >= 4 K-steps per split. With 4 k-tiles in flight per
    workgroup (gemm.hip PF) a tile needs fewer splits to cover HBM latency, and fewer splits = fewer
    partial bytes to reduce. From a graph-replayed sweep with weights streamed cold from HBM, as in a real
    decode step (profiles/decode_gemm_prefetch_sweep_r1.jsonl: matches the best split on 17 of 20 Phi-3 /
    Llama-3-8B shapes at M = 16 / 64, within 0.7 us on the rest)."""
    if M >= 640:
        return 1
    ksteps = K // 64
    if 64 < M <= 128:  # wide N: no split; else 4 splits, fewer if K is short
        if N >= 8192:
            return 1
        s = 4
        while s > 1 and (ksteps % s or ksteps // s < 4):
            s //= 2
        return s
    if 32 < M <= 64 and N > 8192 and K <= 8192:  # (see _dk_splits)
        return 1
    tiles = math.ceil(M / 64) * math.ceil(N / 128)
    s = 1
    while tiles * s * 2 <= 256 and ksteps % (s * 2) == 0 and ksteps // (s * 2) >= 4:
        s *= 2
    return s


# Weight-streaming tiles of more than 64 rows (csrc/gemm.hip): code -> rows, columns, and what a product takes on them in us:
# the first round's fill and drain, a K-step of 64 of a round, each further round, a reduce and its partials per million
# values, and a unit's K-step on 1/256 of the chip (what all of them load). Phase-split kernel (csrc/gemm8p.hip): code ->
# rows, fill, a K-step of 256 columns, the same on 1/256 of the chip. Fitted, with no cost below zero, to 598 products of 65 -
# 1200 rows (projections, feed-forwards and encoder layers 384 - 4096 wide, weights cold): off by 5 - 7 % on average, by up to 48
# where all rows of a tile are real and K is 14336. The choice takes 1.008 times the fastest tile on average and at worst 1.2, and
# 0.81 times the rules before it (12 products longer by more than 2 %, up to 1.11 times).
_ROW_TILES = {14: (128, 128, 8.37, 0.38, 0.07, 0.0, 1.84, 0.14), 15: (128, 64, 5.96, 0.25, 0.83, 1.35, 1.96, 0.1),
              16: (64, 64, 5.82, 0.16, 1.66, 2.54, 1.26, 0.08), 17: (64, 128, 5.79, 0.26, 0.72, 1.61, 1.78, 0.13),
              18: (192, 128, 10.64, 0.47, 0.7, 0.0, 1.45, 0.16)}
_PHASE_TILES = {7: (256, 10.76, 0.67, 0.64), 10: (128, 7.11, 0.55, 0.37)}
ROW_TILES_BELOW = 1280
# From there on small results only, whole, and where the estimate, 10 % up (rows are a larger part of what tiles load), is still
# below the phase-split kernel's: of 1300 - 5000 rows, us phase-split / streaming: 1300 x 1024 x 1024 16.8 / 11.5, 2000 17.0 / 13.5;
# 1600 x 768 x 3072 25.1 / 22.3; 1600 x 1024 x 4096 29.3 / 25.2; 3500 x 384 x 1536 22.4 / 17.7; 1300 x 4096 x 4096 54.0 / 46.7.
# Not 2600 x 1024 x 1024 (18.1 / 19.2), 1600 x 4096 x 1024 (24.5 / 28.3) or 2000 x 3072 x 768 (20.3 / 22.4).
# Of 44 products that it takes, bf16 and fp16, 43 run in 0.49 - 1.00 of the time and one in 1.07 (1700 x 1024 x 4096 with a residual).
SMALL_RESULT_ROWS, SMALL_RESULT = 5120, 21 << 18
# Tiles of csrc/gemm_dk.hip for more than 64 rows, where K is shared out within a workgroup and nothing waits for a barrier: code ->
# 16-row groups, 16-column groups, workgroups of a CU at a time, and us: start and end, each further round, a K-step of 64 of a round,
# of a CU's workgroup, of a workgroup on 1/256 of the chip, a million weights. Fitted, with no cost below zero, to 1600 products of 65 -
# 1279 rows (256 - 12288 columns and K, bf16 and fp16, every epilogue, weights cold): off by 5 % on average (20 and 21: 9 and 8).
_DK_TILES = {20: (2, 1, 2, 3.227, 1.608, 0.0, 0.041, 0.032, 0.03), 21: (2, 2, 2, 3.195, 1.584, 0.0, 0.066, 0.03, 0.14),
             22: (4, 2, 1, 3.822, 2.207, 0.106, 0.0, 0.047, 0.07), 23: (4, 3, 1, 4.445, 2.823, 0.126, 0.0, 0.05, 0.132),
             24: (4, 4, 1, 5.0, 3.36, 0.149, 0.0, 0.05, 0.174), 25: (4, 6, 1, 6.87, 5.082, 0.218, 0.0, 0.039, 0.193)}


def _row_tiles_ok(M: int, N: int) -> bool:
    return M < ROW_TILES_BELOW or (M <= SMALL_RESULT_ROWS and M * N <= SMALL_RESULT)


def _stream_us(M: int, N: int, K: int):
    """(us, tile, splits) of a product on the fastest weight-streaming tile. Splits: below 8192 columns (wider products
    cover the CUs), 4 K-steps at least, two rounds of units at most, and 32 MB of partials below 256 rows, 20 MB from there."""
    ksteps, best = K // 64, None
    most = (1024 if M < 256 else 640) // (math.ceil(M / 64) * math.ceil(N / 128))
    for t, (bm, bn, fill, step, again, reduce, part, load) in _ROW_TILES.items():
        tiles = math.ceil(M / bm) * math.ceil(N / bn)
        for s in (1, 2, 4, 8):
            if s > 1 and (N >= 8192 or M >= ROW_TILES_BELOW or ksteps % s or ksteps // s < 4 or tiles * s > 520 or s > most):
                continue
            rounds, nk = math.ceil(tiles * s / 256), ksteps // s
            us = fill + rounds * nk * step + (rounds - 1) * again + tiles * s * nk * load / 256
            if s > 1:
                # (a close call stays whole; less so with full tiles of 128 rows, which whole K takes longer than estimated:
                # 128 x 3072 x 3072 18.7 / 15.7 in four splits, 112 x 5120 x 5120 28.4 / 25.9; 80 x 2048 x 2048 10.2 / 10.6)
                us = (1.03 if 96 < M <= 128 else 1.06) * (us + reduce + part * s * M * N * 1e-6)
            if best is None or us < best[0]:
                best = us, t, s
    return best


def _phase_us(M: int, N: int, K: int, epi: int, tile: int) -> float:
    """us of a product on the phase-split kernel, its last round shared where that kernel shares it."""
    rows, fill, step, load = _PHASE_TILES[tile]
    tiles = math.ceil(M / rows) * math.ceil(N / 256)
    return fill + step * lib().da_gemm8p_ksteps(M, N, K, epi, tile) / 100 + load * tiles * (K // 64) / 256


@_rule
def _row_us(M: int, N: int, K: int, epi: int = EPI_NONE, f16: bool = False):
    """(us, tile, splits) of a product of 65 rows to ROW_TILES_BELOW, and of more with a small result (``_row_tiles_ok``): the
    fastest by estimate (``_ROW_TILES``). From 640 rows on the phase-split kernel picks its own row height, and keeps what is
    within 3 %. Below, bf16 residuals are added to the fp32 sums only (that kernel rounds the product first)."""
    us, tile, splits = _stream_us(M, N, K)
    if K < 128 or (epi == EPI_RESID and M < 640 and not f16):
        return us, tile, splits
    phase = min((_phase_us(M, N, K, epi, t), t) for t in _PHASE_TILES)
    if us * (1.1 if M >= ROW_TILES_BELOW else 1) < phase[0] * (0.97 if M >= 640 else 1):
        return us, tile, splits
    return phase[0], (0 if M >= 640 else phase[1]), 1


def _row_tile(M: int, N: int, K: int, epi: int = EPI_NONE, f16: bool = False):
    """(tile, splits) of such a product."""
    return _row_us(M, N, K, epi, f16)[1:]


@_rule
def _dk_rows_tile(M: int, N: int, K: int, epi: int = EPI_NONE, f16: bool = False) -> int:
    """The tile of ``_DK_TILES`` that a product of 65 rows to ROW_TILES_BELOW runs on, 0: those of ``_row_tile`` are faster. Where the
    estimate is 3 % below theirs, 10 % from 257 rows on, 15 % where K is above 4096 (768 x 320 x 8192 is not: 15.9 / 19.0 us): 1025 of
    the 1600 products that it is fitted to, in 0.63 of their time, seven of them in 1.02 - 1.12; of 500 others 334, two in more than 1.02
    (850 x 256 x 6656 14.2 / 16.9). us, tiles of ``_row_tile`` -> these: 128 x 384 x 1536 8.9 ->
    4.3, 256 x 768 x 768 6.6 -> 4.3, 256 x 768 x 3072 12.2 -> 7.6, 256 x 1024 x 4096 13.8 -> 8.8, 128 x 4096 x 1024 8.1 -> 6.3,
    640 x 1024 x 1024 8.2 -> 6.9; 96 x 3072 x 3072 13.0 -> 9.6, 128 x 4096 x 4096 19.8 -> 15.8; not 171 x 5920 x 2688 (18.0 / 20.6),
    1022 x 1088 x 1216 (10.2 / 11.7) or 1192 x 864 x 1216 (10.9 / 12.6)."""
    if not 64 < M < ROW_TILES_BELOW:
        return 0
    best, ksteps = None, K // 64
    for t, (fm, fn, beside, start, again, step, wg, load, weights) in _DK_TILES.items():
        if epi in GATED and fn % 2:
            continue
        units = math.ceil(M / (16 * fm)) * math.ceil(N / (16 * fn))
        per_cu = math.ceil(units / 256)
        rounds = math.ceil(per_cu / beside)
        us = start + again * (rounds - 1) + ksteps * (step * rounds + wg * per_cu + load * units / 256) + weights * N * K * 1e-6
        if best is None or us < best[0]:
            best = us, t
    line = 0.85 if K > 4096 else 0.97 if M <= 256 else 0.9
    return best[1] if best[0] < line * _row_us(M, N, K, epi, f16)[0] else 0


def _gemm_dk_rows(a, w, bias, epi: int, resid, out, tile: int):
    _check(lib().da_gemm_dk_rows(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), _ptr(bias), _ptr(resid),
                                 0 if resid is None else resid.stride(0), a.shape[0], *w.shape, epi, tile,
                                 int(a.dtype == torch.float16), _stream()), "gemm_dk_rows")
    return out


@_rule
def _rope_apart(M: int, N: int, K: int) -> bool:
    """A QKV projection of 256 rows and more as a product by itself, on the tile that it has then, and rope_cache behind it (which
    reads and writes the result once more; the rotation costs the phase-split kernel 4 us): 432 x 6144 x 4096 54 -> 39 us, 300 x 9216
    x 3072 46 -> 34, 800 x 6144 x 4096 54 -> 50, where 128x256 tiles leave CUs idle, and 1024 x 9216 x 3072 95 -> 69, 1200 x 10240 x
    8192 212 -> 173, where the one kernel had two rounds of 128-row tiles and the product alone one of 256-row ones. From
    ROW_TILES_BELOW rows on where the one kernel's last round is short, which the product alone shares out: 2817 x 6144 x 4096
    158 -> 140, 3600 168 -> 160, 5400 250 -> 237, 1931 x 9216 x 3072 131 -> 127; not 2300 (128 / 131), 3600 (194 / 199) or
    4100 x 6144 x 4096 (176 / 184). The estimates are 5 us and 8 % off either way there; 1 us and 5 % in favour of apart put the line
    where it takes the slower way by more than 2 % least often: at 4 of 70 products of five projections (2235 x 9216 x 3072 115 / 123, 4142 x
    5120 x 3072 117 / 121 and 5010 x 7680 x 5120 290 / 298 stay in one kernel, 3185 x 5120 x 3072 83 / 92 does not, whose kernel is then one
    of 128-row tiles), at 10 without. The 19 that it takes run in 0.92 of the one kernel's time on average."""
    tiles = math.ceil(M / 256) * math.ceil(N / 256)
    if M >= ROW_TILES_BELOW:
        alone = min(_phase_us(M, N, K, EPI_NONE, t) for t in _PHASE_TILES)
        return tiles > 256 and alone + M * N * 1e-6 - 1 < 1.05 * (_phase_us(M, N, K, EPI_ROPE, 7) + 4)
    return _row_us(M, N, K)[0] + 4 + M * N * 1e-6 < 0.97 * (_phase_us(M, N, K, EPI_ROPE, 7 if tiles >= 256 else 10) + 4)


def _rope_round(M: int, N: int) -> bool:
    """The one kernel has a single round of 256-row tiles, of more than half of the chip: us, product and rope_cache / one kernel:
    900 x 9216 x 3072 65 / 62, 1024 69 / 65, 1200 70 / 64. (Of fewer tiles 900 x 6144 x 4096 53 / 57.)"""
    return 128 < math.ceil(M / 256) * math.ceil(N / 256) <= 256


# ------------------------------------------------------------------------------ norms etc.
def rmsnorm(x, w, eps: float, resid=None, out=None):
    _bf16_cuda(x, "x"); _bf16_cuda(w, "w")
    M, D = x.shape
    _req(x.stride(1) == 1 and x.stride(0) % 8 == 0 and D % 8 == 0, "x must be row-major, D % 8 == 0")
    _req(w.numel() == D, "w must be [D]")
    if resid is not None:
        _bf16_cuda(resid, "resid"); _req(resid.is_contiguous() and resid.shape == (M, D), "resid must be [M, D]")
    if out is None:
        out = torch.empty((M, D), dtype=torch.bfloat16, device=x.device)
    _req(out.stride(1) == 1 and out.stride(0) % 8 == 0, "bad out")
    _check(lib().da_rmsnorm(_ptr(x), x.stride(0), _ptr(resid), _ptr(w), _ptr(out), out.stride(0), M, D,
                            float(eps), _stream()), "rmsnorm")
    return out


def layernorm(x, g, b, eps: float, resid=None, out=None, fp8_out: bool = False):
    """LayerNorm; with ``fp8_out`` also returns the row-quantised e4m3 copy and its scales
    (fused: the row is quantised from registers) -> (y, yq, yscale)."""
    _bf16_cuda(x, "x")
    M, D = x.shape
    _req(x.is_contiguous() and D % 8 == 0, "x must be contiguous, D % 8 == 0")
    if resid is not None:
        _req(resid.is_contiguous() and resid.shape == x.shape, "bad resid")
    if out is None:
        out = torch.empty_like(x)
    if fp8_out:
        yq = torch.empty((M, D), dtype=FP8, device=x.device)
        ys = torch.empty(M, dtype=torch.float32, device=x.device)
        _check(lib().da_layernorm_q(_ptr(x), _ptr(resid), _ptr(g), _ptr(b), _ptr(out), _ptr(yq), _ptr(ys), M, D,
                                    float(eps), _stream()), "layernorm_q")
        return out, yq, ys
    _check(lib().da_layernorm(_ptr(x), _ptr(resid), _ptr(g), _ptr(b), _ptr(out), M, D, float(eps), _stream()),
           "layernorm")
    return out


def bert_embed_ln(ids, positions, types, word, pos, type_, g, b, eps: float, out=None, fp8_out: bool = False):
    _i32(ids, "ids"); _i32(positions, "positions")
    if types is not None:
        _i32(types, "types")
    T = ids.numel()
    D = word.shape[1]
    _req(positions.numel() == T, "positions length")
    if out is None:
        out = torch.empty((T, D), dtype=torch.bfloat16, device=ids.device)
    if fp8_out:
        yq = torch.empty((T, D), dtype=FP8, device=ids.device)
        ys = torch.empty(T, dtype=torch.float32, device=ids.device)
        _check(lib().da_bert_embed_ln_q(_ptr(ids), _ptr(positions), _ptr(types), _ptr(word), _ptr(pos), _ptr(type_),
                                        _ptr(g), _ptr(b), _ptr(out), _ptr(yq), _ptr(ys), T, D, float(eps), _stream()),
               "bert_embed_ln_q")
        return out, yq, ys
    _check(lib().da_bert_embed_ln(_ptr(ids), _ptr(positions), _ptr(types), _ptr(word), _ptr(pos), _ptr(type_),
                                  _ptr(g), _ptr(b), _ptr(out), T, D, float(eps), _stream()), "bert_embed_ln")
    return out


def embed(ids, table, out=None):
    _i32(ids, "ids"); _bf16_cuda(table, "table")
    T, D = ids.numel(), table.shape[1]
    if out is None:
        out = torch.empty((T, D), dtype=torch.bfloat16, device=ids.device)
    _check(lib().da_embed(_ptr(ids), _ptr(table), _ptr(out), T, D, _stream()), "embed")
    return out


def pool_l2norm(h, cu_seqlens, mode: int = 0, out32=None, out16=None):
    _bf16_cuda(h, "h"); _i32(cu_seqlens, "cu_seqlens")
    B = cu_seqlens.numel() - 1
    D = h.shape[1]
    _req(h.is_contiguous(), "h contiguous")
    if out32 is None and out16 is None:
        out32 = torch.empty((B, D), dtype=torch.float32, device=h.device)
    _check(lib().da_pool_l2norm(_ptr(h), _ptr(cu_seqlens), B, D, mode, h.shape[0], _ptr(out32), _ptr(out16), _stream()),
           "pool_l2norm")
    return out32 if out32 is not None else out16


def rope_cache(qkv, pos, cos_sin, H, Hkv, D, slot=None, k_cache=None, v_cache=None, rotate_q=True):
    """In-place RoPE on q and k heads of qkv [T, (H+2Hkv)*D]; optionally writes k/v into the cache."""
    _bf16_cuda(qkv, "qkv"); _i32(pos, "pos")
    T = qkv.shape[0]
    _req(qkv.is_contiguous() and qkv.shape[1] == (H + 2 * Hkv) * D, "qkv shape")
    _req(cos_sin.dtype == torch.float32 and cos_sin.is_contiguous() and cos_sin.shape[-1] == 2
         and cos_sin.shape[1] == D // 2, "cos_sin must be fp32 [max_pos, D/2, 2]")
    max_seq = 0
    if k_cache is not None:
        _i32(slot, "slot")
        _req(k_cache.is_contiguous() and v_cache.is_contiguous() and k_cache.shape == v_cache.shape, "caches")
        _req(k_cache.dim() == 4 and k_cache.shape[1] == Hkv and k_cache.shape[3] == D, "cache [S, Hkv, max_seq, D]")
        max_seq = k_cache.shape[2]
    _check(lib().da_rope_cache(_ptr(qkv), _ptr(pos), _ptr(slot), _ptr(cos_sin), _ptr(k_cache), _ptr(v_cache),
                               T, H, Hkv, D, max_seq, 1 if rotate_q else 0, _stream()), "rope_cache")
    return qkv


def flash_kv_cache_ok(D: int, causal: bool) -> bool:
    """True when flash_attn_varlen can read the sequences' own keys from the KV cache (kv_cache=)."""
    return causal and D == 96


def flash_attn_varlen(q, k, v, cu_seqlens, max_seqlen: int, H: int, Hkv: int, D: int, causal: bool,
                      scale: float | None = None, out=None, prefix=None, kv_cache=None):
    """q/k/v: 2-D [T, *] views with head h at columns h*D (strided views into a packed qkv are fine).
    prefix = (k_pre, v_pre, P): shared-prefix keys of every sequence, one KV-cache slot's
    [Hkv, max_seq, D] K and V (RoPE applied); query i of a sequence is key P + i.
    kv_cache = (k_cache, v_cache, slot, pos) (flash_kv_cache_ok only): the own keys of the sequence
    starting at token t are k_cache[slot[t], :, pos[t] + j] (slot / pos int32 per token, as the QKV
    projection wrote them); k / v are then ignored (None allowed)."""
    kc = vc = ks = kpos = None
    if kv_cache is not None:
        kc, vc, ks, kpos = kv_cache
        _req(flash_kv_cache_ok(D, causal), "kv_cache: causal D = 96 only")
        _bf16_cuda(kc, "k_cache"); _bf16_cuda(vc, "v_cache"); _i32(ks, "slot"); _i32(kpos, "pos")
        _req(kc.is_contiguous() and vc.is_contiguous() and kc.shape == vc.shape and kc.dim() == 4
             and kc.shape[1] == Hkv and kc.shape[3] == D, "caches [slots, Hkv, max_seq, D]")
        _req(ks.numel() >= q.shape[0] and kpos.numel() >= q.shape[0], "slot / pos per token")
        k = v = q  # unused by the kernel in this mode
    for t, n in ((q, "q"), (k, "k"), (v, "v")):
        _bf16_cuda(t, n)
        _req(t.dim() == 2 and t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0, f"{n} layout")
    _i32(cu_seqlens, "cu_seqlens")
    _req(D in (32, 64, 96, 128), f"head dim {D} unsupported")
    _req(H % Hkv == 0, "H % Hkv")
    T = q.shape[0]
    if out is None:
        out = torch.empty((T, H * D), dtype=torch.bfloat16, device=q.device)
    scale = scale if scale is not None else 1.0 / math.sqrt(D)
    B = cu_seqlens.numel() - 1
    kp = vp = None
    hstride, P = 0, 0
    if prefix is not None:
        kp, vp, P = prefix
        P = int(P)
        _bf16_cuda(kp, "k_pre"); _bf16_cuda(vp, "v_pre")
        _req(kp.dim() == 3 and kp.shape == vp.shape and kp.shape[0] == Hkv and kp.shape[2] == D
             and kp.is_contiguous() and vp.is_contiguous() and 0 <= P <= kp.shape[1], "prefix K/V [Hkv, max_seq, D]")
        hstride = kp.shape[1] * D
    if kc is not None:
        _req(prefix is None or kp.shape[1] == kc.shape[2], "prefix and caches differ in max_seq")
        hstride = kc.shape[2] * D
    _check(lib().da_flash_attn_v2(_ptr(q), _ptr(k), _ptr(v), q.stride(0), k.stride(0), v.stride(0),
                                  _ptr(cu_seqlens), B, int(max_seqlen), H, Hkv, D, int(causal), float(scale),
                                  _ptr(out), out.stride(0), _ptr(kp), _ptr(vp), hstride, P, _ptr(ks), _ptr(kpos),
                                  _ptr(kc), _ptr(vc), _stream()),
           "flash_attn_varlen")
    return out


# Split-KV partials merged inside the decode kernel by the last split of each (row, kv head)
# (False: separate combine launch; tests cover both). The ticket counters stay zero between
# launches; buffers are only ever added, never freed, so a captured graph's pointer stays valid.
_FUSED_COMBINE = True
_UC: dict = {}


class _RawBuf:
    """A device allocation outside PyTorch's allocator (uncached memory), as a ``_ptr``-able object."""

    def __init__(self, ptr: int, nbytes: int):
        self.ptr, self.nbytes = ptr, nbytes

    def data_ptr(self) -> int:
        return self.ptr


def _uncached(tag: str, nbytes: int, device) -> _RawBuf:
    """Zeroed uncached (L2-bypassing) device memory for cross-workgroup hand-offs (decode split
    partials + tickets). Grows by adding buffers, never frees: captured graphs keep their pointers."""
    key = (tag, device.index if device.index is not None else torch.cuda.current_device(),
           getattr(_ROLE, "name", "main"))
    bufs = _UC.setdefault(key, [])
    if not bufs or bufs[-1].nbytes < nbytes:
        n = max(nbytes, 1 << 20)
        p = ctypes.c_void_p()
        with torch.cuda.device(device):
            _check(lib().da_malloc_uncached(n, ctypes.byref(p)), "hipExtMallocWithFlags(uncached)")
        bufs.append(_RawBuf(p.value, n))
    return bufs[-1]


def _decode_split(B: int, Hkv: int, max_len: int, chunk: int):
    """(chunk, nsplit) of a decode-attention launch (static for a captured graph: from max_len)."""
    if chunk <= 0:
        # measured on MI355X (profiles/decode_attn_chunks_r1.txt): per-workgroup overhead dominates
        # small chunks; aim for ~768 workgroups, 512..4096 keys each
        want = max_len * B * Hkv / 768
        chunk = 512
        while chunk < want and chunk < 4096:
            chunk *= 2
    return chunk, max(1, math.ceil(max_len / chunk))


BY_LEN_KEYS = 256


@_rule
def _gqa_split(B: int, Hkv: int, max_len: int):
    """(chunk, nsplit, by_len) of a grouped-query launch (head dims 64 and 128) whose caller names no chunk. by_len: a row's
    keys over as many of the nsplit splits as hold ``chunk`` of them each; else over all of them. Measured over 16 query
    heads on 2 KV heads x 64, 32 on 4 and on 8 x 128, 1 - 64 rows in caches of 1024 - 16384 keys, all rows of a length or
    mixed:
      * 192 - 256 (row, head) pairs in up to 2048 keys: whole rows, a workgroup per CU (8 heads, 24 - 32 rows of 100 - 750
        of 1024: 24 - 28 -> 18 - 19 us; of 250 - 1500 of 2048: 37 - 42 -> 31 - 32; one full row among short ones loses
        up to 1.5x). In 4096 keys the gain is 3 - 13 % and the loss 1.65x: not there.
      * the even splits are of 512 keys and more than one round of workgroups, or the cache is up to 1024 or from 8192
        keys long: by the row's length (8 heads, 8 rows of 1024 in 4096: 21.9 -> 14.5; 4 rows of 2000 in 8192: 26.5 ->
        15.1, of 4000 30.5 -> 26.5; 12 rows of 500 in 2048: 21.2 -> 13.6, full 33.5 -> 32.3; half the rows full and half
        short loses up to 1.17x). Even splits of 1024 keys gain 4 % by it and lose up to 1.5x.
      * else even: a launch that leaves CUs idle is the faster the more splits it has (one row of 1024 in 4096: 10.9 us
        even, 12.1 by length)."""
    if 192 <= B * Hkv <= 256 and max_len <= 2048:
        return math.ceil(max_len / 64) * 64, 1, False
    chunk, nsplit = _decode_split(B, Hkv, max_len, 0)
    if chunk == 512 and nsplit > 1 and (B * Hkv * nsplit > 256 or not 1024 < max_len < 8192):
        return BY_LEN_KEYS, nsplit, True
    return chunk, nsplit, False


def _mha_split(B: int, H: int, max_len: int):
    """(chunk, nsplit, by_len) of a launch with a KV head to each query head whose caller names no chunk: a row's keys over as
    many of the even splits as hold 256 of them each, or 128 where the launch has up to 32 (row, head) pairs and would leave
    CUs idle. us even / by length of 64 / 128 / 256, 32 heads x 96 in caches of 4096: one row of 60 7.4 / 5.5 / 5.5 / 5.5, of 500
    8.0 / 8.1 / 7.5 / 8.3, of 2935 11.7 / 11.7 / 11.6 / 11.6; 4 rows of 64 - 146 8.7 / 9.3 / 7.8 / 6.5, of 200 - 500 9.8 / 10.6 /
    10.5 / 9.0, of 900 - 3100 26.5 / 26.2 / 26.0 / 25.1; 8 rows 9.3 / 10.0 / 9.9 / 6.9, 12.2 / 13.3 / 13.2 / 13.1, 38.9 / 40.0 /
    40.2 / 40.4."""
    chunk, nsplit = _decode_split(B, H, max_len, 0)
    if nsplit == 1:
        return chunk, 1, False
    return (BY_LEN_KEYS if B * H > 32 else BY_LEN_KEYS // 2), nsplit, True


# Same-XCD split exchange of the batch-1..small-batch MHA decode attention (attention.hip, VAR bit 3):
# all splits of a (row, kv head) pair on one XCD, their partials and ticket in cached memory (L2
# round trips instead of uncached ones). It relies on the launch's workgroup -> XCD round-robin, so
# it is used only after the placement probe confirmed that on this device, and never once a
# CU-masked stream exists in the process (a masked queue need not dispatch round-robin over XCDs;
# ops/streams.py sets MASKED_STREAMS). DA_DECODE_XC=0 turns it off.
DECODE_XC = os.environ.get("DA_DECODE_XC", "1") != "0"
MASKED_STREAMS = False
_XC_PROBE: dict = {}


def decode_xc_ok(device) -> bool:
    """True when every workgroup w of a launch runs on XCD w % 8 here (placement probe, once per
    device; not during a graph capture, where the answer stays unknown = False)."""
    if not DECODE_XC or MASKED_STREAMS:
        return False
    idx = device.index if device.index is not None else torch.cuda.current_device()
    if idx in _XC_PROBE:
        return _XC_PROBE[idx]
    if torch.cuda.is_current_stream_capturing():
        return False
    n = 1024
    out = torch.zeros(n * 4, dtype=torch.int32, device=device)
    _check(lib().da_placement_probe(_ptr(out), n, 0, _stream()), "placement_probe")
    xcc = out.view(n, 4)[:, 0].cpu().numpy()
    ok = bool(len(set(xcc.tolist())) == 8 and all(len(set(xcc[r::8].tolist())) == 1 for r in range(8)))
    _XC_PROBE[idx] = ok
    return ok


_COUNTERS: dict = {}


def _cached_counters(tag: str, n: int, device) -> torch.Tensor:
    """Zeroed int32 counters in ordinary device memory that stay allocated (captured graphs keep the
    pointer; the kernels leave them zero)."""
    key = (tag, device.index if device.index is not None else torch.cuda.current_device(),
           getattr(_ROLE, "name", "main"))  # per workspace role, like the uncached ones: concurrent lanes
    bufs = _COUNTERS.setdefault(key, [])
    if not bufs or bufs[-1].numel() < n:
        bufs.append(torch.zeros(max(n, 1024), dtype=torch.int32, device=device))
    return bufs[-1]


def _decode_checks(q, k_cache, v_cache, lens, slot, H, Hkv, D, max_len, pre, rope):
    _bf16_cuda(q, "q"); _i32(lens, "lens"); _i32(slot, "slot")
    _req(D in (64, 96, 128), "head dim")
    _req((H // Hkv) in (1, 2, 4, 8) and H % Hkv == 0, "GQA group must be 1/2/4/8")
    B = q.shape[0]
    _req(k_cache.dim() == 4 and k_cache.shape[1] == Hkv and k_cache.shape[3] == D, "cache shape")
    _req(max_len <= k_cache.shape[2], "max_len > cache capacity")
    if pre is not None:
        _i32(pre, "pre"); _req(pre.shape == (B, 2) and pre.is_contiguous(), "pre must be int32 [B, 2]")
    cs = ps = None
    if rope is not None:
        cs, ps = rope
        _req(H == Hkv and D % 8 == 0, "fused RoPE decode: MHA only")
        _i32(ps, "pos")
        _req(cs.dtype == torch.float32 and cs.is_contiguous() and cs.shape[1] == D // 2 and cs.shape[2] == 2, "cos_sin")
        _req(q.stride(1) == 1 and q.shape[1] >= (H + 2 * Hkv) * D, "fused RoPE decode needs the qkv row")
        _req(k_cache.is_contiguous() and v_cache.is_contiguous(), "caches must be contiguous")
    return cs, ps


def decode_attn(q, k_cache, v_cache, lens, slot, H, Hkv, D, max_len: int, chunk: int = 0, scale=None, out=None,
                pre=None, rope=None):
    """q [B, >=H*D] (row stride any multiple of 8); lens/slot int32 [B]; max_len = max(lens) or the
    cache capacity (host int, fixes the split count so the launch is graph-capturable).
    chunk = keys per workgroup (0 = auto: enough workgroups to fill 256 CUs, 4 waves x 64-key tiles).
    pre: optional int32 [B, 2] device tensor (P, prefix slot), P % 64 == 0: keys [0, P) of row b
    are the batch's shared prompt head, stored once in the prefix slot (read through the cache).
    rope = (cos_sin fp32 [max_pos, D/2, 2], pos int32 [B]), MHA only: q is the raw qkv row
    [B, (H + 2 Hkv) D]; the kernel applies RoPE to q and the new token's k and writes that token's
    k / v into the cache at pos (== lens - 1) — the decode step's rope_cache launch folded in."""
    cs, ps = _decode_checks(q, k_cache, v_cache, lens, slot, H, Hkv, D, max_len, pre, rope)
    B = q.shape[0]
    if chunk <= 0 and H == Hkv:
        chunk, nsplit, by_len = _mha_split(B, H, max_len)
    elif chunk <= 0 and D in (64, 128):
        chunk, nsplit, by_len = _gqa_split(B, Hkv, max_len)
    else:
        (chunk, nsplit), by_len = _decode_split(B, Hkv, max_len, chunk), False
    ws = _workspace(B * H * nsplit * (D + 2) * 4, q.device)
    if out is None:
        out = torch.empty((B, H * D), dtype=torch.bfloat16, device=q.device)
    scale = scale if scale is not None else 1.0 / math.sqrt(D)
    cnt = None
    xc = 0
    if _FUSED_COMBINE and nsplit > 1:
        if H == Hkv and B * Hkv <= 32 and (B * Hkv) % 8 == 0 and decode_xc_ok(q.device):
            xc = 1  # same-XCD exchange: ws (the role workspace) and counters in cached memory
            cnt = _cached_counters("decode_cnt_xc", B * Hkv, q.device)
        else:
            cnt = _uncached("decode_cnt", B * Hkv * 4, q.device)
            ws = _uncached("decode_ws", B * H * nsplit * (D + 2) * 4, q.device)
    _check(lib().da_decode_attn(_ptr(q), q.stride(0), _ptr(k_cache), _ptr(v_cache), _ptr(lens), _ptr(slot), _ptr(pre), B, H,
                                Hkv, D, k_cache.shape[2], chunk, nsplit, float(scale), _ptr(ws), _ptr(out), out.stride(0),
                                _ptr(cnt), _ptr(cs), _ptr(ps), xc | 2 * by_len, _stream()), "decode_attn")
    return out


# rows up to which sample() cuts the vocabulary over many workgroups (0: always one per row); at
# batch 64 one workgroup per row leaves 192 CUs idle too
SAMPLE_CHUNKED_MAX_B = 64
_SAMPLE_WS: dict = {}


def _sample_ws(nfloats: int, device) -> torch.Tensor:
    """Per-(device, workspace role) fp32 scratch of the chunked sampler. Grows by adding buffers and
    never frees one: a captured decode graph keeps pointing at the buffer it was captured with."""
    key = (device.index if device.index is not None else torch.cuda.current_device(), getattr(_ROLE, "name", "main"))
    bufs = _SAMPLE_WS.setdefault(key, [])
    if not bufs or bufs[-1].numel() < nfloats:
        bufs.append(torch.empty(max(nfloats, 16384), dtype=torch.float32, device=device))
    return bufs[-1]


def sample(logits, temperature: float, seed: int, step: int = 0, out_tok=None, out_lp=None, conf=None,
           active=None, ctr=None, pos=None, lens=None, hist=None, start=None, eos=()):
    """Fused temperature sampler over bf16 or fp32 logits (see rope_sample.hip). Returns (tokens, logprobs)."""
    f32 = int(logits.dtype == torch.float32)
    if f32:
        _req(logits.is_cuda, "logits must be on GPU")
    else:
        _bf16_cuda(logits, "logits")
    B, V = logits.shape
    _req(logits.stride(1) == 1 and logits.stride(0) % 8 == 0, "logits layout")
    dev = logits.device
    if out_tok is None:
        out_tok = torch.empty(B, dtype=torch.int32, device=dev)
    if out_lp is None:
        out_lp = torch.empty(B, dtype=torch.float32, device=dev)
    if conf is not None:
        _req(conf.dtype == torch.float32 and conf.shape == (B, 2), "conf must be fp32 [B, 2]")
    for t, n in ((active, "active"), (ctr, "ctr"), (pos, "pos"), (lens, "lens"), (start, "start")):
        if t is not None:
            _i32(t, n); _req(t.numel() >= B, f"{n} too short")
    hist_ld = 0
    if hist is not None:
        _i32(hist, "hist"); _req(hist.dim() == 2 and hist.shape[0] >= B, "hist [B, n]")
        _req(pos is not None and start is not None, "hist needs pos and start")
        hist_ld = hist.shape[1]
    e = list(eos)[:4] + [-1] * (4 - min(4, len(eos)))
    if B <= SAMPLE_CHUNKED_MAX_B and V >= 4096:
        # few rows: the row is split over ceil(V / 1024) workgroups + a finalize launch (same token;
        # the batch-1 sampler took ~21 us on one CU, rope_sample.hip sample_chunk_kernel)
        ws = _sample_ws(B * ((V + 1023) // 1024) * 8, dev)
        _check(lib().da_sample_chunked(_ptr(logits), B, V, logits.stride(0), float(temperature), seed & 0xffffffff,
                                       step & 0xffffffff, _ptr(ctr), _ptr(ws), _ptr(out_tok), _ptr(out_lp),
                                       _ptr(conf), _ptr(active), _ptr(pos), _ptr(lens), _ptr(hist), _ptr(start),
                                       hist_ld, e[0], e[1], e[2], e[3], f32, _stream()), "sample_chunked")
        return out_tok, out_lp
    _check(lib().da_sample(_ptr(logits), B, V, logits.stride(0), float(temperature), seed & 0xffffffff,
                           step & 0xffffffff, _ptr(ctr), _ptr(out_tok), _ptr(out_lp), _ptr(conf), _ptr(active),
                           _ptr(pos), _ptr(lens), _ptr(hist), _ptr(start), hist_ld, e[0], e[1], e[2], e[3],
                           f32, _stream()), "sample")
    return out_tok, out_lp


def sample_partial(logits, temperature: float, seed: int, v0: int, step: int = 0, ctr=None, out=None):
    """Vocab-parallel sampling, rank side: logits [B, Vl] of the vocabulary slice starting at global
    index v0 -> stats fp32 [B, 8] = (best Gumbel score, best global index as int bits, local max,
    local sum exp(x - max), logit of the best, 0, 0, 0). See rope_sample.hip."""
    _bf16_cuda(logits, "logits")
    B, V = logits.shape
    _req(logits.stride(1) == 1, "logits rows must be contiguous")
    if ctr is not None:
        _i32(ctr, "ctr"); _req(ctr.numel() >= B, "ctr too short")
    if out is None:
        out = torch.empty((B, 8), dtype=torch.float32, device=logits.device)
    _req(out.dtype == torch.float32 and out.shape == (B, 8) and out.is_contiguous(), "stats must be fp32 [B, 8]")
    _check(lib().da_sample_partial(_ptr(logits), B, V, logits.stride(0), int(v0), float(temperature),
                                   seed & 0xffffffff, step & 0xffffffff, _ptr(ctr), _ptr(out), _stream()),
           "sample_partial")
    return out


def sample_finalize(gathered, ranks: int, out_tok=None, out_lp=None, conf=None, active=None, pos=None, lens=None,
                    hist=None, start=None, eos=()):
    """Vocab-parallel sampling, merge side: gathered fp32 [B, ranks * 8] (every rank's stats, rank
    order) -> the token / logprob / bookkeeping of ``sample`` on the full row."""
    _req(gathered.is_cuda and gathered.dtype == torch.float32 and gathered.is_contiguous(), "gathered fp32")
    B = gathered.shape[0]
    _req(gathered.shape == (B, 8 * ranks), f"gathered must be [B, {8 * ranks}]")
    dev = gathered.device
    if out_tok is None:
        out_tok = torch.empty(B, dtype=torch.int32, device=dev)
    if out_lp is None:
        out_lp = torch.empty(B, dtype=torch.float32, device=dev)
    if conf is not None:
        _req(conf.dtype == torch.float32 and conf.shape == (B, 2), "conf must be fp32 [B, 2]")
    for t, n in ((active, "active"), (pos, "pos"), (lens, "lens"), (start, "start")):
        if t is not None:
            _i32(t, n); _req(t.numel() >= B, f"{n} too short")
    hist_ld = 0
    if hist is not None:
        _i32(hist, "hist"); _req(hist.dim() == 2 and hist.shape[0] >= B, "hist [B, n]")
        _req(pos is not None and start is not None, "hist needs pos and start")
        hist_ld = hist.shape[1]
    e = list(eos)[:4] + [-1] * (4 - min(4, len(eos)))
    _check(lib().da_sample_finalize(_ptr(gathered), B, ranks, _ptr(out_tok), _ptr(out_lp), _ptr(conf), _ptr(active),
                                    _ptr(pos), _ptr(lens), _ptr(hist), _ptr(start), hist_ld, e[0], e[1], e[2], e[3],
                                    _stream()), "sample_finalize")
    return out_tok, out_lp


# --------------------------------------------------------------------------- vector search
def _scan_rows(N: int) -> int:
    """Rows that a wave of the streaming scan of up to 16 queries takes at least (the launcher gives it what one round of
    workgroups needs, if that is more): 16 waves a CU over the chip (256 CUs), but at least 64 rows each, with 256 workgroups
    of 4 waves where that leaves CUs idle (one tile of 16 rows each at least: a few hundred centroids)."""
    tiles = lambda waves: math.ceil(N / waves / 16) * 16  # noqa: E731
    return max(min(tiles(256 * 4), 64), tiles(256 * 16), 16)


def _found(Q: int, K: int, ids, like):
    """A search's results (scores, rows; the rows' external ids where ``ids`` is their table) and the launcher's arguments."""
    out_s = like.new_empty((Q, K), dtype=torch.float32)
    if ids is None:
        out = like.new_empty((Q, K), dtype=torch.int32)
        return out_s, out, (out_s.data_ptr(), out.data_ptr(), None, 0)
    _req(ids.is_cuda and ids.dtype == torch.int64 and ids.is_contiguous() and ids.dim() == 1 and ids.numel() > 0,
         "ids must be int64 [N]")
    out = like.new_empty((Q, K), dtype=torch.int64)
    return out_s, out, (out_s.data_ptr(), out.data_ptr(), ids.data_ptr(), ids.numel())


def topk_dense(X, Qv, K: int, thr: float, slots=None, bitmap=None, rows_per_block: int | None = None, ids=None):
    """Exact top-K of Qv @ X^T per query with threshold and optional doc-slot bitmap [Q, W] int32: scores and rows, or
    (``ids`` int64 [N]) scores and ids[rows], as ``gather_ids`` gives them."""
    _bf16_cuda(X, "X"); _bf16_cuda(Qv, "Qv")
    N, d = X.shape
    Q = Qv.shape[0]
    _req(X.is_contiguous() and Qv.is_contiguous() and Qv.shape[1] == d, "X/Qv layout")
    _req(d % 32 == 0 and 1 <= K <= 32, "d % 32 and 1 <= K <= 32")
    W = 0
    if slots is not None:
        _i32(slots, "slots")
        _req(slots.numel() >= N, "slots length")
    if bitmap is not None:
        _req(slots is not None, "bitmap needs slots")
        _req(bitmap.dtype == torch.int32 and bitmap.is_contiguous() and bitmap.shape[0] == Q, "bitmap [Q, W] int32")
        W = bitmap.shape[1]
    if d in (384, 768, 1024) and rows_per_block is None and N > 0 and Q <= 256:
        # the streaming scan (search-sized batches over a big shard; k-means assignment, with the
        # rows as the queries, keeps the query-major tiles below)
        rpw = _scan_rows(N)
        ws = _call_scratch(int(lib().da_topk_stream_ws(N, Q, K, rpw)), X)
        out_s, out, args = _found(Q, K, ids, X)
        _check(lib().da_topk_dense_stream(X.data_ptr(), N, d, _at(slots), Qv.data_ptr(), Q, _at(bitmap), W, float(thr), K,
                                          rpw, ws.data_ptr(), *args, _raw_stream()), "topk_dense_stream")
        return out_s, out
    if rows_per_block is None:
        qt = math.ceil(Q / 16)
        nblk = max(1, min(math.ceil(N / 256), max(1, 1024 // qt)))
        rows_per_block = max(64, math.ceil(math.ceil(N / nblk) / 64) * 64)
    nblk = max(1, math.ceil(N / rows_per_block))
    ws = _call_scratch(nblk * Q * K * 8, X)
    out_s, out, args = _found(Q, K, ids, X)
    _check(lib().da_topk_dense(_ptr(X), N, d, _ptr(slots), _ptr(Qv), Q, _ptr(bitmap), W, float(thr), K,
                               rows_per_block, _ptr(ws), *args, _stream()), "topk_dense")
    return out_s, out


TABLE_MAX = 512  # numbers of a filter's row ranges that ride in a launch's arguments (the kernel's TR_TABLE)


def topk_ranges(X, Qv, ranges, range_off, K: int, thr: float, max_rows: int, slots=None, bitmap=None,
                rows_per_split: int | None = None, ids=None):
    """Top-K per query over its own row ranges. ranges int32 [R, 2], range_off int32 [Q+1] (both on the
    device or both arrays of the host, or lists of their numbers: a few ride in the launch's arguments, more go in one copy);
    max_rows = max total rows of any query (host int) — sets the split count: rows_per_split rows of a query per
    workgroup (default: ``_rows_per_split``)."""
    rows, Q, table = rows_per_split or _rows_per_split(max_rows, Qv.shape[0], K), Qv.shape[0], None
    if isinstance(ranges, list):
        _req(len(range_off) == Q + 1 and len(ranges) == 2 * range_off[-1], "range_off length")
        size = len(range_off) + len(ranges)
        if size <= TABLE_MAX:
            table = (c_int * size)(*range_off, *ranges)
        else:
            ranges, range_off = np.array(ranges, dtype=np.int32).reshape(-1, 2), np.array(range_off, dtype=np.int32)
    if isinstance(ranges, np.ndarray):
        _req(range_off.shape == (Q + 1,) and ranges.shape == (range_off[-1], 2), "range_off length")
        host = np.concatenate([range_off, ranges.reshape(-1)]).astype(np.int32, copy=False)
        if host.size > TABLE_MAX:
            from . import h2d
            t = h2d(host, X.device)
            range_off, ranges = t[:Q + 1], t[Q + 1:]
        else:
            table = (c_int * host.size).from_buffer(host)
    if table is None:
        _i32(ranges, "ranges"); _i32(range_off, "range_off")
        _req(range_off.numel() == Q + 1, "range_off length")
    else:
        ranges = range_off = None
    return _ranges(X, Qv, ranges, range_off, None, K, thr, max_rows, slots, bitmap, rows, ids, table)


def topk_lists(X, Qv, lists, list_off, K: int, thr: float, mean_rows: int, max_rows: int, slots=None, bitmap=None,
               ids=None):
    """Top-K per query over the lists it names: lists int32 [Q, probes] (on the device; negative: none), list l =
    rows list_off[l] .. list_off[l + 1] (int32). mean_rows / max_rows: rows of a query, expected / at most (host
    ints). The lists never visit the host: nothing waits for the kernel that chose them."""
    _i32(lists, "lists"); _i32(list_off, "list_off")
    _req(lists.dim() == 2 and lists.shape[0] == Qv.shape[0], "lists [Q, probes]")
    # workgroups past a query's rows end at once, but lists of very uneven length must not make too many of them
    rows = max(_rows_per_split(mean_rows, Qv.shape[0], K), math.ceil(max_rows / 512 / 64) * 64)
    return _ranges(X, Qv, list_off, None, lists, K, thr, max_rows, slots, bitmap, rows, ids)


def _rows_per_split(rows: int, Q: int, K: int) -> int:
    """Rows of a query per workgroup of the range scan: what gives about 1024 workgroups (4 per CU: a workgroup keeps
    48 KB of rows on their way), from one step of the kernel (64) to 512; half a step where there are few rows in all (us, 64 / 32: one
    query's 384 rows of 768 12.2 / 10.5, 64 queries of 144 12.8 / 11.8; 6250 rows of 24 queries 47.4 / 62.7) and twice the lists are
    still few to put together (on the device, of 384 columns: K = 10, 1500 rows, 470 candidates of half steps 20.6 / 18.1, 2200, 690 17.4 /
    18.2; K = 20, 600, 380 21.0 / 18.8, 1500, 940 19.9 / 22.8; K = 32, 300, 320 22.5 / 19.4, 600, 608 19.9 / 25.0, 6400, 6400 40 / 48)."""
    half = rows * Q <= RANGE_SMALL and math.ceil(rows / 32) * K <= RANGE_HALF
    return 32 if half else min(512, max(64, math.ceil(rows * Q / 1024 / 64) * 64))


RANGE_SMALL = 10240  # rows of all queries up to which a workgroup of the range scan takes half a step
RANGE_HALF = 512     # and candidates of a query that half steps leave
RANGE_JOIN = 256     # candidates of a query up to which its last workgroup puts them together


def _range_join(splits: int, Q: int, K: int) -> bool:
    """Whether the lists of a query's workgroups meet in the same launch: its four waves take a cut each up to 256 candidates, a
    launch's up to sixteen more of them at a time (us on the device, in the launch / after it: 60 candidates 10.5 / 10.5,
    240 15.0 / 15.2, 405 15.0 / 13.2, 960 16.7 / 15.0; one workgroup a query 5.3 / 7.1; the host 15.8 / 17.5)."""
    return splits * K <= RANGE_JOIN and Q <= N_COUNTERS


def _ranges(X, Qv, ranges, range_off, lists, K, thr, max_rows, slots, bitmap, rows_per_split, ids=None, table=None):
    _bf16_cuda(X, "X"); _bf16_cuda(Qv, "Qv")
    N, d = X.shape
    Q = Qv.shape[0]
    _req(d % 8 == 0 and d <= 4096 and 1 <= K <= 32, "d / K limits")
    W = 0
    if slots is not None:
        _i32(slots, "slots")
        _req(slots.numel() >= N, "slots length")
    if bitmap is not None:
        _req(slots is not None, "bitmap needs slots")
        _req(bitmap.dtype == torch.int32 and bitmap.shape[0] == Q, "bitmap")
        W = bitmap.shape[1]
    out_s, out, args = _found(Q, K, ids, X)
    if Q == 0:
        return out_s, out
    splits = max(1, math.ceil(max_rows / rows_per_split))
    ws = _call_scratch(splits * Q * K * 8, X)
    stream = _raw_stream()
    cnt = _counters(X.device, stream) if _range_join(splits, Q, K) else None
    _check(lib().da_topk_ranges(X.data_ptr(), d, _at(slots), Qv.data_ptr(), Q, _at(ranges), _at(range_off), _at(lists),
                                0 if lists is None else lists.shape[1], _at(bitmap), W, float(thr), K, splits, rows_per_split, ws.data_ptr(), *args,
                                table, 0 if table is None else len(table), _at(cnt), stream), "topk_ranges")
    return out_s, out


def topk_merge(cand_s, cand_i, K: int, ids=None):
    """cand [P, Q, K] -> the best K of each query, sorted."""
    _req(cand_s.dtype == torch.float32 and cand_i.dtype == torch.int32, "dtypes")
    P, Q, K2 = cand_s.shape
    _req(K2 == K, "K mismatch")
    cs, ci = cand_s.contiguous(), cand_i.contiguous()
    out_s, out, args = _found(Q, K, ids, cs)
    _check(lib().da_topk_merge(_ptr(cs), _ptr(ci), P, Q, K, *args, _stream()), "topk_merge")
    return out_s, out


def gather_ids(rows, ids):
    """ids[rows] (int64, in the shape of rows), -1 where a row is outside [0, len(ids))."""
    _req(rows.is_cuda, "rows must be on GPU")
    _req(ids.is_cuda and ids.dtype == torch.int64 and ids.is_contiguous() and ids.dim() == 1, "ids must be int64 [N]")
    if rows.dtype != torch.int32:
        rows = rows.long().clamp(-1, 2**31 - 1).int()
    rows = rows.contiguous()
    out = torch.empty(rows.shape, dtype=torch.int64, device=rows.device)
    _check(lib().da_gather_ids(_ptr(rows), rows.numel(), _ptr(ids), ids.numel(), _ptr(out), _stream()), "gather_ids")
    return out


def kmeans_accum(X, assign, sums, counts):
    _bf16_cuda(X, "X"); _i32(assign, "assign")
    N, d = X.shape
    _req(sums.dtype == torch.float32 and sums.shape[1] == d and counts.dtype == torch.float32, "sums/counts fp32")
    _check(lib().da_kmeans_accum(_ptr(X), N, d, _ptr(assign), _ptr(sums), _ptr(counts), _stream()), "kmeans_accum")


def reserve_workspace(nbytes: int, device=None) -> None:
    """Pre-size the shared split-K / decode workspace. Must be called before capturing HIP graphs
    so the captured kernels keep pointing at a live buffer."""
    dev = torch.device(device) if device is not None else torch.device("cuda", torch.cuda.current_device())
    _workspace(nbytes, dev)


def spin(us: int, device=None) -> None:
    """Hold the current stream busy for ``us`` microseconds (one wave polling the wall clock;
    bounded to 10 s). Test helper: work queued behind it on this stream is provably still pending."""
    _req(0 <= us <= 10_000_000, "spin: 0 <= us <= 1e7")
    _check(lib().da_spin(int(us), None, _stream()), "da_spin")


def gemm8p_persist(on: int = -1) -> int:
    """Persistent tile loop of the prefill GEMM (one workgroup per CU walking its XCD's tiles) on
    (1) / off (0) for later launches; -1 only queries. Returns the previous setting."""
    for rule in (_tail_bytes, _row_us, _dk_rows_tile, _row_choice, _rope_apart):  # (the rules that ask which rounds are shared)
        rule.cache_clear()
    return int(lib().da_gemm8p_persist(int(on)))


def gemm4w_variant(v: int = -1) -> int:
    """Schedule of the four-wave 256x256 kernel (tile 13, csrc/gemm4w.hip) where K / 64 is even and
    >= 4: 0 = three fragment sets, two barriers per K-tile (default), 1 = two sets, 2 = three sets,
    one barrier; -1 only queries. Returns the previous setting."""
    return int(lib().da_gemm4w_variant(int(v)))


def _f16_cuda(t, name):
    _req(t.is_cuda, f"{name} must be on GPU")
    _req(t.dtype == torch.float16, f"{name} must be fp16, got {t.dtype}")


def gemm_f16(a, w, bias=None, epi: int = EPI_NONE, resid=None, out=None) -> torch.Tensor:
    """out = epi(a @ w^T) in fp16 (fp32 accumulate); epi NONE / BIAS / GELU / RESID."""
    _f16_cuda(a, "a"); _f16_cuda(w, "w")
    M, K = a.shape
    N = w.shape[0]
    _req(w.shape[1] == K and w.is_contiguous() and a.stride(1) == 1 and a.stride(0) % 8 == 0, "gemm_f16 layout")
    _req(K % 64 == 0 and K >= 128 and N % 8 == 0, f"gemm_f16 shape N={N} K={K}")
    _req(epi in (EPI_NONE, EPI_BIAS, EPI_GELU, EPI_RESID), "gemm_f16 epilogue")
    if bias is not None:
        _f16_cuda(bias, "bias"); _req(bias.numel() == N, "bias")
    ldr = 0
    if epi == EPI_RESID:
        _f16_cuda(resid, "resid")
        _req(resid.shape == (M, N) and resid.stride(1) == 1 and resid.stride(0) % 8 == 0, "resid")
        ldr = resid.stride(0)
    if out is None:
        out = torch.empty((M, N), dtype=torch.float16, device=a.device)
    _req(out.dtype == torch.float16 and out.shape == (M, N) and out.stride(1) == 1 and out.stride(0) % 8 == 0, "out")
    tile, splits = _row_choice(M, N, K, epi, a.stride(0), True)
    if tile in _DK_TILES:
        return _gemm_dk_rows(a, w, bias, epi, resid, out, tile)
    stream = _raw_stream()
    ws = _call_partials(splits, M, N, a)
    tail = _gemm_tail(a.device, stream, M, N, K, epi, tile) if _has_tail(M, tile, True) else (None, None)
    _check(lib().da_gemm_f16(_ptr(a), a.stride(0), _ptr(w), _ptr(out), out.stride(0), _ptr(bias), _ptr(resid), ldr,
                             M, N, K, epi, tile, splits, _ptr(ws), *map(_ptr, tail), c_void_p(stream)), "gemm_f16")
    return out


def flash_attn_f16(q, k, v, cu_seqlens, max_seqlen: int, H: int, Hkv: int, D: int, causal: bool = False,
                   scale: float | None = None, out=None):
    for t, n in ((q, "q"), (k, "k"), (v, "v")):
        _f16_cuda(t, n)
        _req(t.dim() == 2 and t.stride(1) == 1 and t.stride(0) % 8 == 0 and t.data_ptr() % 16 == 0, f"{n} layout")
    _i32(cu_seqlens, "cu_seqlens")
    _req(D in (64, 96) and H % Hkv == 0, "flash_attn_f16: D 64 / 96")
    T = q.shape[0]
    if out is None:
        out = torch.empty((T, H * D), dtype=torch.float16, device=q.device)
    scale = scale if scale is not None else 1.0 / math.sqrt(D)
    _check(lib().da_flash_attn_f16(_ptr(q), _ptr(k), _ptr(v), q.stride(0), k.stride(0), v.stride(0), _ptr(cu_seqlens),
                                   cu_seqlens.numel() - 1, int(max_seqlen), H, Hkv, D, int(causal), float(scale),
                                   _ptr(out), out.stride(0), _stream()), "flash_attn_f16")
    return out


def layernorm_f16(x, g, b, eps: float, resid=None, out=None):
    _f16_cuda(x, "x")
    M, D = x.shape
    _req(x.is_contiguous() and D % 8 == 0, "x must be contiguous, D % 8 == 0")
    if resid is not None:
        _f16_cuda(resid, "resid"); _req(resid.is_contiguous() and resid.shape == x.shape, "bad resid")
    _f16_cuda(g, "g"); _f16_cuda(b, "b")
    if out is None:
        out = torch.empty_like(x)
    _check(lib().da_layernorm_f16(_ptr(x), _ptr(resid), _ptr(g), _ptr(b), _ptr(out), M, D, float(eps), _stream()),
           "layernorm_f16")
    return out


def bert_embed_ln_f16(ids, positions, types, word, pos, type_, g, b, eps: float, out=None):
    _i32(ids, "ids"); _i32(positions, "positions")
    for t, n in ((word, "word"), (pos, "pos"), (type_, "type"), (g, "g"), (b, "b")):
        _f16_cuda(t, n)
    T, D = ids.numel(), word.shape[1]
    _req(positions.numel() == T and D % 8 == 0, "positions length / D")
    if out is None:
        out = torch.empty((T, D), dtype=torch.float16, device=ids.device)
    _check(lib().da_bert_embed_ln_f16(_ptr(ids), _ptr(positions), _ptr(types), _ptr(word), _ptr(pos), _ptr(type_),
                                      _ptr(g), _ptr(b), _ptr(out), T, D, float(eps), _stream()), "bert_embed_ln_f16")
    return out


def pool_l2norm_f16(h, cu_seqlens, mode: int = 0, out32=None, out16=None):
    """fp16 hidden states -> unit-norm pooled rows, fp32 and / or bf16 (the index storage type)."""
    _f16_cuda(h, "h"); _i32(cu_seqlens, "cu_seqlens")
    B, D = cu_seqlens.numel() - 1, h.shape[1]
    _req(h.is_contiguous() and D % 8 == 0, "h contiguous")
    if out16 is not None:
        _bf16_cuda(out16, "out16")
    if out32 is None and out16 is None:
        out32 = torch.empty((B, D), dtype=torch.float32, device=h.device)
    _check(lib().da_pool_l2norm_f16(_ptr(h), _ptr(cu_seqlens), B, D, mode, h.shape[0], _ptr(out32), _ptr(out16), _stream()),
           "pool_l2norm_f16")
    return out32 if out32 is not None else out16


# the batch-of-portions ops (recurrent mixers, paged attention, 32-bit residual stream)
from .seq_kernels import (causal_conv, delta_rule, delta_step, delta_step_fits, gated_scan, gemm_any, gemm_heads,  # noqa: E402,F401
                          gemm_partials, latent_attn, latent_flash, latent_flash_fits, latent_gather, latent_prep, partials_fit, rglru_gates,
                          selective_scan, sigmoid_attn, stream_add, stream_final, stream_step)
