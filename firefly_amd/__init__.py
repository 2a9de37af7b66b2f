"""firefly_amd - MI355X (gfx950) paged KV-cache path for Firefly.

The product is the shared library ``firefly_amd/libffkv.so`` (C ABI in ``include/ffkv.h``; C++ API in
``include/firefly/``).  This module loads it and offers thin wrappers that take torch tensors, so programs, tests
and benchmarks can drive the C ABI with device memory torch allocated: the calls of a step go through ``_front.so``
(csrc/python/front.cpp, built with the library), sizes and the like through ctypes.  There is no CPU fallback: if
either is missing or fails to load, importing this package raises.
"""

from __future__ import annotations

import ctypes
import os
from pathlib import Path

try:
    from . import _front
except ImportError as e:
    raise ImportError("firefly_amd/_front.so is not built; run `python firefly_amd/build.py`") from e

_PKG = Path(__file__).resolve().parent
LIB_PATH = _PKG / "libffkv.so"

DTYPE_F32 = 0
DTYPE_F16 = 1
DTYPE_BF16 = 2
DTYPE_I8 = 3
DTYPE_FP8_E4M3 = 8

OK = 0
ERR_INVALID_ARGUMENT = -1
ERR_UNSUPPORTED = -2
ERR_WORKSPACE = -3
ERR_HIP = -4

BLOCK_SIZE = 16
NOALLOC_SCRATCH_BYTES = 32 << 20  # FFKV_NOALLOC_SCRATCH_BYTES (include/ffkv.h)


class FFKVError(RuntimeError):
    """A C ABI call returned a non-zero status."""

    def __init__(self, code: int, message: str):
        super().__init__(f"ffkv error {code}: {message}")
        self.code = code


def _load() -> ctypes.CDLL:
    if not LIB_PATH.exists():
        raise ImportError(f"{LIB_PATH} is not built; run `python firefly_amd/build.py` (no CPU fallback exists)")
    # torch wheels bundle their own HIP runtime under the same soname (libamdhip64.so.7).  Loading torch first
    # makes libffkv.so bind to that already-loaded runtime, so there is one runtime per process and torch's
    # device pointers and streams are valid here; loading ours first would put two runtimes in the process.
    try:
        import torch
    except ImportError:
        torch = None
    lib = ctypes.CDLL(str(LIB_PATH), mode=os.RTLD_NOW | ctypes.RTLD_LOCAL)
    vp, i32, f32, sz = ctypes.c_void_p, ctypes.c_int, ctypes.c_float, ctypes.c_size_t
    lib.ffkv_append.restype = i32
    lib.ffkv_append.argtypes = [vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, i32, vp]
    lib.ffkv_kv_block_bytes.restype = sz
    lib.ffkv_kv_block_bytes.argtypes = [i32, i32, i32]
    lib.ffkv_decode_workspace_bytes.restype = sz
    lib.ffkv_decode_workspace_bytes.argtypes = [i32, i32, i32, i32, i32]
    lib.ffkv_paged_decode.restype = i32
    lib.ffkv_paged_decode.argtypes = [vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, i32,
                                      i32, f32, vp, sz, vp]
    lib.ffkv_paged_decode_noalloc.restype = i32
    lib.ffkv_paged_decode_noalloc.argtypes = [vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32, i32, i32, i32,
                                              i32, i32, f32, vp]
    lib.ffkv_decode_shared_prefix_workspace_bytes.restype = sz
    lib.ffkv_decode_shared_prefix_workspace_bytes.argtypes = [i32, i32, i32, i32, i32, i32, i32]
    lib.ffkv_paged_decode_shared_prefix.restype = i32
    lib.ffkv_paged_decode_shared_prefix.argtypes = [vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32, i32,
                                                    i32, i32, i32, i32, f32, i32, vp, sz, vp]
    lib.ffkv_append_paged_decode.restype = i32
    lib.ffkv_append_paged_decode.argtypes = [vp, vp, i32, vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32,
                                             i32, i32, i32, i32, i32, f32, vp, sz, vp]
    lib.ffkv_paged_prefill.restype = i32
    lib.ffkv_paged_prefill.argtypes = [vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, i32,
                                       i32, i32, ctypes.c_float, vp]
    lib.ffkv_prefill_workspace_bytes.restype = sz
    lib.ffkv_prefill_workspace_bytes.argtypes = [i32] * 10
    lib.ffkv_paged_prefill_ws.restype = i32
    lib.ffkv_paged_prefill_ws.argtypes = [vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, i32,
                                          i32, i32, f32, vp, sz, vp]
    lib.ffkv_rope.restype = i32
    lib.ffkv_rope.argtypes = [vp, vp, i32, vp, i32, i32, i32, i32, i32, ctypes.c_float, vp]
    lib.ffkv_rope_append.restype = i32
    lib.ffkv_rope_append.argtypes = [vp, vp, vp, i32, vp, vp, i32, vp, vp, vp, vp, i32, i32, i32, i32, i32, i32, i32,
                                     i32, ctypes.c_float, vp]
    lib.ffkv_last_error.restype = ctypes.c_char_p
    lib.ffkv_last_error.argtypes = []
    lib.ffkv_version.restype = ctypes.c_char_p
    lib.ffkv_version.argtypes = []
    if torch is not None:
        _bind(lib, torch)
    return lib


def _bind(lib, torch) -> None:
    """Point the native front end (``_front``, csrc/python/front.cpp) at ``lib``'s functions."""
    names = ("append", "paged_decode", "append_paged_decode", "paged_decode_shared_prefix", "paged_decode_noalloc",
             "prefill_workspace_bytes", "paged_prefill_ws", "rope", "rope_append")
    _front.bind(tuple(ctypes.cast(getattr(lib, "ffkv_" + n), ctypes.c_void_p).value for n in names),
                list(_torch_dtypes(torch).items()), getattr(torch._C, "_cuda_getDevice", None),
                getattr(torch._C, "_cuda_getCurrentRawStream", None), lambda: torch.cuda.current_stream().cuda_stream)


def version() -> str:
    return lib.ffkv_version().decode()


def check(code: int) -> None:
    if code != OK:
        raise FFKVError(code, lib.ffkv_last_error().decode())


def _torch_dtypes(torch) -> dict:
    """torch dtype -> ffkv dtype code (uint8 storage is read as OCP fp8 e4m3)."""
    table = {
        torch.float32: DTYPE_F32,
        torch.float16: DTYPE_F16,
        torch.bfloat16: DTYPE_BF16,
        torch.int8: DTYPE_I8,
        torch.uint8: DTYPE_FP8_E4M3,
    }
    fp8 = getattr(torch, "float8_e4m3fn", None)
    if fp8 is not None:
        table[fp8] = DTYPE_FP8_E4M3
    return table


def torch_dtype_code(t) -> int:
    """ffkv dtype code of a torch tensor (uint8 storage is read as OCP fp8 e4m3)."""
    import torch

    try:
        return _torch_dtypes(torch)[t.dtype]
    except KeyError as e:
        raise TypeError(f"unsupported dtype {t.dtype}") from e


lib = _load()
os.register_at_fork(after_in_child=_front.forget_stream)


def _ptr(t) -> int | None:
    return None if t is None else t.data_ptr()


def _stream(stream) -> int | None:
    import torch

    if stream is None:
        stream = torch.cuda.current_stream()
    return stream.cuda_stream if hasattr(stream, "cuda_stream") else int(stream)


def append_kv_cache(k, v, k_cache, v_cache, block_table, context_lens=None, k_scale=None, v_scale=None,
                    num_blocks: int | None = None, stream=None) -> None:
    """Append ``k``/``v`` ``[B, S, Hkv, D]`` into pages ``[N, 16, Hkv, D]`` (``ffkv_append``)."""
    check(_front.append(k, v, k_cache, v_cache, block_table, context_lens, k_scale, v_scale, num_blocks, stream))


def paged_prefill(q, k_cache, v_cache, block_table, context_lens, out=None, k_scale=None, v_scale=None,
                  max_context_len: int = 0, scale: float = 0.0, num_blocks: int | None = None, stream=None):
    """Causal prefill attention (``ffkv_paged_prefill_ws``): ``q`` ``[B, S, Hq, D]`` over the paged cache (queries at
    ``context_lens[b] + t``), or, with ``block_table=None``, over contiguous ``k_cache``/``v_cache``
    ``[B, S, Hkv, D]``.  Returns ``out`` ``[B, S, Hq * D]``.  Calls too small to fill the GPU are split over their keys
    where the rows may be long; ``max_context_len`` (no row has more tokens, the chunk's included) says that they are
    not, behind a wide table."""
    if out is None:
        import torch

        B, S, Hq, D = q.shape
        out = torch.empty((B, S, Hq * D), dtype=q.dtype, device=q.device)
    check(_front.prefill(q, out, k_cache, v_cache, k_scale, v_scale, block_table, context_lens, max_context_len, scale,
                         num_blocks, stream, _prefill_scratch))
    return out


def _prefill_scratch(n: int, q, stream):
    """Scratch of ``n`` bytes for one call on ``stream`` (None: the current one), from torch's allocator and belonging
    to that stream, so that it can be reused once the call's work on the stream is done.  None, where the call
    runs unsplit, while the stream is being captured (a capture allocates nothing here) and where there is no memory
    for it."""
    import torch

    if stream is not None:
        if not isinstance(stream, torch.cuda.Stream):
            stream = torch.cuda.ExternalStream(int(getattr(stream, "cuda_stream", stream)), device=q.device)
        with torch.cuda.stream(stream):
            return _prefill_scratch(n, q, None)
    if torch.cuda.is_current_stream_capturing():
        return None
    try:
        return torch.empty(n, dtype=torch.uint8, device=q.device)
    except torch.OutOfMemoryError:
        return None


def apply_rope(q, k, context_lens=None, theta: float = 1e6, stream=None) -> None:
    """Rotary embedding of ``q`` ``[B, S, Hq, D]`` (or None) and ``k`` ``[B, S, Hkv, D]`` in place
    (``ffkv_rope``; the reference's ``kernels::apply_rope``)."""
    check(_front.rope(q, k, context_lens, theta, stream))


def rope_append_kv_cache(q, k, v, k_cache, v_cache, block_table, context_lens=None, theta: float = 1e6,
                         k_scale=None, v_scale=None, num_blocks: int | None = None, stream=None) -> None:
    """``apply_rope(q, k)`` then ``append_kv_cache(k, v, ...)`` in one kernel (``ffkv_rope_append``)."""
    check(_front.rope_append(q, k, v, k_cache, v_cache, block_table, context_lens, theta, k_scale, v_scale, num_blocks,
                             stream))


def kv_block_bytes(cache_dtype: int, num_kv_heads: int, head_dim: int) -> int:
    """Bytes of one pool block (16 tokens of one layer, K and V, scales included) for a cache dtype."""
    return int(lib.ffkv_kv_block_bytes(cache_dtype, num_kv_heads, head_dim))


def decode_workspace_bytes(batch: int, num_heads: int, head_dim: int, max_blocks: int,
                           max_context_len: int = 0) -> int:
    return int(lib.ffkv_decode_workspace_bytes(batch, num_heads, head_dim, max_blocks, max_context_len))


def decode_workspace(batch: int, num_heads: int, head_dim: int, max_blocks: int, max_context_len: int = 0,
                     device=None, stream=None):
    """A decode workspace (uint8 tensor, contents irrelevant) sized by ``ffkv_decode_workspace_bytes``."""
    import torch

    n = max(decode_workspace_bytes(batch, num_heads, head_dim, max_blocks, max_context_len), 256)
    return torch.empty(n, dtype=torch.uint8, device=device if device is not None else "cuda")


def shared_prefix_workspace(batch: int, num_heads: int, num_kv_heads: int, head_dim: int, max_blocks: int,
                            shared_blocks: int, max_context_len: int = 0, device=None):
    """A workspace for ``paged_attention_shared_prefix`` (``ffkv_decode_shared_prefix_workspace_bytes``)."""
    import torch

    n = max(int(lib.ffkv_decode_shared_prefix_workspace_bytes(batch, num_heads, num_kv_heads, head_dim, max_blocks,
                                                              max_context_len, shared_blocks)), 256)
    return torch.empty(n, dtype=torch.uint8, device=device if device is not None else "cuda")


def _decode_out(q, out):
    """``out``, or a new ``[B, 1, Hq * D]`` like ``q``."""
    if out is None:
        import torch

        out = torch.empty((q.shape[0], 1, q.shape[-2] * q.shape[-1]), dtype=q.dtype, device=q.device)
    return out


def paged_attention_shared_prefix(q, k_cache, v_cache, block_table, context_lens, shared_blocks: int, out=None,
                                  k_scale=None, v_scale=None, max_context_len: int = 0, scale: float = 0.0,
                                  workspace=None, num_blocks: int | None = None, stream=None):
    """Decode over rows whose first ``shared_blocks`` block-table entries are the same pages
    (``ffkv_paged_decode_shared_prefix``): the shared pages are attended once for all rows."""
    out = _decode_out(q, out)
    check(_front.decode_shared(q, out, k_cache, v_cache, k_scale, v_scale, block_table, context_lens, max_context_len,
                               scale, num_blocks, int(shared_blocks), workspace, stream))
    return out


def append_paged_attention(k_new, v_new, q, k_cache, v_cache, block_table, context_lens, out=None, k_scale=None,
                           v_scale=None, max_context_len: int = 0, scale: float = 0.0, workspace=None,
                           num_blocks: int | None = None, stream=None):
    """``append_kv_cache(k_new, v_new, ...)`` (one token per row) then ``paged_attention``, as one call
    (``ffkv_append_paged_decode``; for 16-bit caches fed in their own dtype the decode's launch appends too, and no
    other row of the call may then attend a row's new slot)."""
    out = _decode_out(q, out)
    check(_front.append_decode(q, out, k_cache, v_cache, k_scale, v_scale, block_table, context_lens, max_context_len,
                               scale, num_blocks, k_new, v_new, workspace, stream))
    return out


def paged_attention_noalloc(q, k_cache, v_cache, block_table, context_lens, out, k_scale=None, v_scale=None,
                            max_context_len: int = 0, scale: float = 0.0, num_blocks: int | None = None, stream=None):
    """PagedAttention decode that allocates no device memory (``ffkv_paged_decode_noalloc``): the split-K partials
    use the library's static per-GPU scratch.  ``out`` ``[B, 1, Hq * D]`` is the caller's."""
    check(_front.decode_noalloc(q, out, k_cache, v_cache, k_scale, v_scale, block_table, context_lens, max_context_len,
                                scale, num_blocks, stream))
    return out


def paged_attention(q, k_cache, v_cache, block_table, context_lens, out=None, k_scale=None, v_scale=None,
                    max_context_len: int = 0, scale: float = 0.0, workspace=None, num_blocks: int | None = None,
                    stream=None):
    """PagedAttention decode (``ffkv_paged_decode``).  ``q`` is ``[B, 1, Hq, D]`` (or ``[B, Hq, D]``)."""
    out = _decode_out(q, out)
    check(_front.decode(q, out, k_cache, v_cache, k_scale, v_scale, block_table, context_lens, max_context_len, scale,
                        num_blocks, workspace, stream))
    return out
