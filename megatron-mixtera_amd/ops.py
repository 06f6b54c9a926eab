"""Torch-level wrappers over the C ABI: tensors in, raw pointers + strides out.

Each function enqueues exactly one C-ABI call on torch's current stream.  The keyword signatures live here; the
checks (dtypes, devices, contiguity of the innermost dimension), the result tensor, the workspace and the call itself
are one native function each (``csrc/host/native.cpp``), because building these calls in Python took 12-20 us apiece
-- more than the kernels of a small decode step.  Nothing here computes: without the HIP library these functions raise.
"""
from __future__ import annotations

from typing import Optional, Tuple

import torch
from torch import Tensor

import threading

from . import _lib
from ._lib import (MI_DTYPE_BF16, MI_DTYPE_FP16, MI_KV_16BIT, MI_KV_BF16, MI_KV_FP8_E4M3,  # noqa: F401
                   MI_NORM_L2, MI_NORM_NONE, MI_NORM_RMS)

_NORM_KINDS = {None: MI_NORM_NONE, "none": MI_NORM_NONE, "rms": MI_NORM_RMS, "l2": MI_NORM_L2}


_native = _lib.native


def _stream(t: Tensor) -> int:
    if t.device.type != "cuda":
        raise RuntimeError(
            f"the HIP kernels need device tensors, got a tensor on {t.device}; there is no CPU path")
    return torch._C._cuda_getCurrentRawStream(t.device.index)


def _require(cond: bool, msg: str) -> None:
    if not cond:
        raise ValueError(msg)


def _cache_strides(cache: Tensor) -> Tuple[int, int, int]:
    """(chunk, token, head) element strides of a ``[N, C, Hkv, d]`` cache view."""
    _require(cache.dim() == 4 and cache.stride(3) == 1, "KV cache must be [N, C, Hkv, d] with contiguous d")
    return cache.stride(0), cache.stride(1), cache.stride(2)


# Split-K workspaces, one per (device, stream) and grown on demand (owned here, handed to the C ABI as caller
# memory).  Calls on one stream are ordered and may share a buffer; calls on different streams of a device may
# overlap, so each stream gets its own.  The native side finds them; a missing or outgrown one is made here.
_retired_workspaces: list = []   # outgrown buffers stay alive: work already enqueued may still use them
_override_local = threading.local()   # ``use_workspace`` buffers of THIS thread (innermost last)


def _override_stack() -> list:
    stack = getattr(_override_local, "stack", None)
    if stack is None:
        stack = _override_local.stack = []
    return stack


def _override() -> Optional[Tensor]:
    """The innermost ``use_workspace`` buffer of this thread."""
    stack = getattr(_override_local, "stack", None)
    return stack[-1] if stack else None


def _grow_workspace(device_index: int, stream: int, nbytes: int) -> None:
    """Give (device, stream) a workspace of at least ``nbytes``; called by the native side when it has none."""
    device = torch.device("cuda", device_index)
    native = _native()
    size = max(nbytes, 2 * _workspace_sizes.get((device_index, stream), 0))
    old = native.set_workspace(device_index, stream, torch.empty(size, dtype=torch.uint8, device=device))
    _workspace_sizes[(device_index, stream)] = size
    if old is not None:
        _retired_workspaces.append(old)
        if len(_retired_workspaces) > 8:  # enqueued work may still use them: wait for it once, then let them go
            torch.cuda.synchronize(device)
            _retired_workspaces.clear()


_workspace_sizes: dict = {}      # (device index, stream) -> bytes


class use_workspace:
    """Context manager: attention calls this thread makes inside use ``buffer`` as their scratch instead of the
    per-stream one (graph capture needs a buffer that is never re-allocated).  Other threads are not affected."""

    def __init__(self, buffer: Tensor):
        self.buffer = buffer

    def __enter__(self):
        _override_stack().append(self.buffer)
        return self.buffer

    def __exit__(self, *exc):
        _override_stack().pop()
        return False


# ---------------------------------------------------------------------------------------------
# experiment knobs: the C ABI takes them per call (MiTuning); this module keeps the set that its own calls pass
# ---------------------------------------------------------------------------------------------
_TUNING_FIELDS = tuple(name for name, _ in _lib.MiTuning._fields_ if name != "reserved")
_tuning_defaults: dict = {}          # set_tuning: every thread, until changed back
_tuning_local = threading.local()    # tuning(...): this thread, inside the with block


def set_tuning(name: str, value: int) -> None:
    """Knob ``name`` (a field of ``MiTuning`` in the header) for every later call of this module; 0 = the default.
    A sweep / test hook: the library itself keeps no such state."""
    _require(name in _TUNING_FIELDS, f"unknown knob {name!r}; the knobs are {', '.join(_TUNING_FIELDS)}")
    if int(value) == 0:
        _tuning_defaults.pop(name, None)
    else:
        _tuning_defaults[name] = int(value)


class tuning:
    """``with ops.tuning(decode_grid=7, prefill_two_phase=-1): ...`` -- knobs for the calls this thread makes
    inside the block (on top of :func:`set_tuning`)."""

    def __init__(self, **knobs: int):
        for name in knobs:
            _require(name in _TUNING_FIELDS, f"unknown knob {name!r}")
        self.knobs = {k: int(v) for k, v in knobs.items()}

    def __enter__(self):
        stack = getattr(_tuning_local, "stack", None)
        if stack is None:
            stack = _tuning_local.stack = []
        stack.append(self.knobs)
        return self

    def __exit__(self, *exc):
        _tuning_local.stack.pop()
        return False


def current_tuning() -> dict:
    """The knobs a call made now would pass (name -> non-zero value)."""
    merged = dict(_tuning_defaults)
    for layer in getattr(_tuning_local, "stack", None) or ():
        merged.update(layer)
    return {k: v for k, v in merged.items() if v != 0}


def _tuning_arg() -> Optional[_lib.MiTuning]:
    """``const MiTuning*`` for a native call: None (NULL) when every knob is at its default."""
    if not _tuning_defaults and not getattr(_tuning_local, "stack", None):
        return None
    knobs = current_tuning()
    return _lib.MiTuning(**knobs) if knobs else None


_DTYPE_CODES = {torch.bfloat16: MI_DTYPE_BF16, torch.float16: MI_DTYPE_FP16}


def _dtype_code(t: Tensor, name: str) -> int:
    _require(t.dtype in _DTYPE_CODES, f"{name} must be bf16 or fp16, got {t.dtype}")
    return _DTYPE_CODES[t.dtype]


# ---------------------------------------------------------------------------------------------
# KV append
# ---------------------------------------------------------------------------------------------
def _rows(x: Tensor, name: str) -> Tuple[Tensor, int, int]:
    """View ``[T, (1,) Hkv, d]`` as T rows of Hkv*d contiguous elements."""
    if x.dim() == 4:
        _require(x.size(1) == 1, f"{name}.size(1) must be 1")
        x = x.squeeze(1)
    _require(x.dim() == 3, f"{name} must be [T, Hkv, d]")
    _require(x.stride(2) == 1 and x.stride(1) == x.size(2), f"{name} rows must be contiguous")
    return x, x.size(1) * x.size(2), x.stride(0)


def kv_append(key: Tensor, value: Optional[Tensor], k_cache: Tensor, v_cache: Optional[Tensor],
              token_to_chunk_idx: Tensor, token_to_local_pos: Tensor) -> None:
    """``k_cache[chunk_idx[t], local[t]] = key[t]`` (and value): bit-exact scatter.  ``value`` and
    ``v_cache`` may both be ``None`` (a cache with one tensor, e.g. MLA latents ``[N, C, 1, r]``)."""
    _native().kv_append(key, value, k_cache, v_cache, token_to_chunk_idx, token_to_local_pos)


def kv_append_decode(key: Tensor, value: Tensor, k_cache: Tensor, v_cache: Tensor,
                     block_table: Tensor, kv_lens: Tensor) -> None:
    """Decode-step append with the slot derived on the GPU from block table + kv length."""
    _stream(key)  # device check first: there is no CPU path
    key, row, k_st = _rows(key, "key")
    value, row_v, v_st = _rows(value, "value")
    R = key.size(0)
    _require(row == row_v and value.size(0) == R and k_st == v_st, "key/value shapes differ")
    _require(key.dtype == k_cache.dtype == v_cache.dtype == value.dtype, "dtype mismatch between K/V and cache")
    sc, st, sh = _cache_strides(k_cache)
    _require(_cache_strides(v_cache) == (sc, st, sh), "k_cache / v_cache strides differ")
    _require(sh == k_cache.size(3) and row == k_cache.size(2) * k_cache.size(3), "cache rows must be contiguous [Hkv, d]")
    _require(block_table.dtype == torch.int32 and kv_lens.dtype == torch.int32, "block_table / kv_lens must be int32")
    _require(block_table.dim() == 2 and block_table.stride(1) == 1 and block_table.size(0) >= R, "bad block_table")
    _require(kv_lens.is_contiguous() and kv_lens.numel() >= R, "bad kv_lens")
    _lib.check(_native().abi_mi_kv_append_decode(key.data_ptr(), value.data_ptr(), k_st, k_cache.data_ptr(), v_cache.data_ptr(),
                                       sc, st, block_table.data_ptr(), block_table.stride(0), kv_lens.data_ptr(),
                                       R, k_cache.size(1), row, key.element_size(), _stream(key)),
               "mi_kv_append_decode")


# ---------------------------------------------------------------------------------------------
# fp8 KV storage
# ---------------------------------------------------------------------------------------------
def quantize_chunks_fp8(src: Tensor, dst: Tensor, scales: Tensor) -> None:
    """Quantise whole 16-bit chunks ``[N, C, Hkv, d]`` into an e4m3fn byte cache + ``[N, Hkv]`` scales."""
    _stream(src)  # device check first: there is no CPU path
    _require(src.dtype in (torch.bfloat16, torch.float16), "source chunks must be bf16 or fp16")
    _require(dst.element_size() == 1, "destination cache must hold one byte per element")
    _require(scales.dtype == torch.float32 and scales.is_contiguous(), "scales must be contiguous fp32")
    ssc, sst, ssh = _cache_strides(src)
    dsc, dst_t, dsh = _cache_strides(dst)
    N, C, H, D = src.shape
    _require(tuple(dst.shape) == (N, C, H, D) and tuple(scales.shape) == (N, H), "shape mismatch")
    _require(ssh == D and dsh == D, "heads must be contiguous")
    _lib.check(_native().abi_mi_kv_quantize_chunks_fp8(src.data_ptr(), ssc, sst, dst.data_ptr(), dsc, dst_t,
                                             scales.data_ptr(), N, C, H, D, _dtype_code(src, "src"), _stream(src)),
               "mi_kv_quantize_chunks_fp8")


def kv_append_decode_fp8(key: Tensor, value: Tensor, k_cache: Tensor, v_cache: Tensor, k_scales: Tensor,
                         v_scales: Tensor, block_table: Tensor, kv_lens: Tensor, headroom: float = 2.0) -> None:
    """Quantise and append one new 16-bit token per request into an fp8 cache."""
    _stream(key)  # device check first: there is no CPU path
    key, row, k_st = _rows(key, "key")
    value, _, v_st = _rows(value, "value")
    _require(key.dtype in (torch.bfloat16, torch.float16) and value.dtype == key.dtype and k_st == v_st,
             "K/V must share one 16-bit type and have equal strides")
    _require(k_cache.element_size() == 1 and v_cache.element_size() == 1, "fp8 caches hold one byte per element")
    sc, st, sh = _cache_strides(k_cache)
    _require(_cache_strides(v_cache) == (sc, st, sh) and sh == k_cache.size(3), "cache layout")
    _require(k_scales.dtype == torch.float32 and v_scales.dtype == torch.float32, "scales must be fp32")
    _require(k_scales.is_contiguous() and v_scales.is_contiguous(), "scales must be contiguous")
    _require(block_table.dtype == torch.int32 and kv_lens.dtype == torch.int32, "block_table / kv_lens must be int32")
    _lib.check(_native().abi_mi_kv_append_decode_fp8(key.data_ptr(), value.data_ptr(), k_st, k_cache.data_ptr(), v_cache.data_ptr(),
                                           sc, st, k_scales.data_ptr(), v_scales.data_ptr(), block_table.data_ptr(),
                                           block_table.stride(0), kv_lens.data_ptr(), key.size(0), k_cache.size(1),
                                           k_cache.size(2), k_cache.size(3), float(headroom), _dtype_code(key, "key"),
                                           _stream(key)), "mi_kv_append_decode_fp8")


def kv_append_fp8(key: Tensor, value: Tensor, k_cache: Tensor, v_cache: Tensor, k_scales: Tensor, v_scales: Tensor,
                  token_to_chunk_idx: Tensor, token_to_local_pos: Tensor, headroom: float = 2.0) -> None:
    """Quantise and append 16-bit tokens with explicit slots into an fp8 cache (prefill / mixed steps)."""
    _native().kv_append_fp8(key, value, k_cache, v_cache, k_scales, v_scales, token_to_chunk_idx, token_to_local_pos,
                            headroom)


# ---------------------------------------------------------------------------------------------
# attention
# ---------------------------------------------------------------------------------------------
def _qo_view(x: Tensor, name: str) -> Tensor:
    if x.dim() == 4:
        _require(x.size(1) == 1, f"{name} must be [T, 1, Hq, d] or [T, Hq, d]")
        x = x.squeeze(1)
    _require(x.dim() == 3 and x.stride(2) == 1, f"{name} must be [T, Hq, d] with contiguous d")
    _require(x.dtype in _DTYPE_CODES, f"{name} must be bf16 or fp16, got {x.dtype}")
    return x


def decode_workspace_bytes(R: int, Hq: int, Hkv: int, head_dim: int, chunk: int, max_kv_len: int,
                           split_tokens: int = 0) -> int:
    return _native().abi_mi_decode_workspace_bytes(R, Hq, Hkv, head_dim, chunk, max_kv_len, split_tokens, _tuning_arg())


def prefill_workspace_bytes(T: int, R: int, Hq: int, Hkv: int, head_dim: int, max_kv_len: int,
                            split_tokens: int = 0) -> int:
    """Scratch of one varlen attention call over ``T`` query rows of ``R`` requests: the decode part's
    partials and, when the tile kernel splits the keys, its partials behind them."""
    return _native().abi_mi_prefill_workspace_bytes(T, R, Hq, Hkv, head_dim, max_kv_len, split_tokens, _tuning_arg())


def paged_decode_attention(q: Tensor, k_cache: Tensor, v_cache: Tensor, kv_lens: Tensor, block_table: Tensor,
                           *, softmax_scale: Optional[float] = None, max_kv_len: Optional[int] = None,
                           split_tokens: int = 0, out: Optional[Tensor] = None,
                           workspace: Optional[Tensor] = None, k_scales: Optional[Tensor] = None,
                           v_scales: Optional[Tensor] = None) -> Tensor:
    """One query token per request against the paged cache; returns a tensor shaped like ``q``."""
    return _native().paged_decode_attention(q, k_cache, v_cache, kv_lens, block_table, softmax_scale, max_kv_len,
                                            split_tokens, out, workspace, k_scales, v_scales, _tuning_arg(), _override())


def paged_decode_attention_noalloc(q: Tensor, k_cache: Tensor, v_cache: Tensor, kv_lens: Tensor, block_table: Tensor,
                                   out: Tensor, *, softmax_scale: Optional[float] = None,
                                   max_kv_len: Optional[int] = None, split_tokens: int = 0,
                                   k_scales: Optional[Tensor] = None, v_scales: Optional[Tensor] = None) -> Tensor:
    """:func:`paged_decode_attention` through the entry point that allocates nothing: the caller brings
    ``out``, the partials live in the library's built-in device scratch (16 MiB per GPU; larger problems are
    rejected).  Calls that overlap on one GPU share that scratch and race."""
    stream = _stream(q)
    q3 = _qo_view(q, "q")
    R, Hq, D = q3.shape
    N, C, Hkv, Dk = k_cache.shape
    _require(Dk == D and tuple(v_cache.shape) == tuple(k_cache.shape), "cache shape mismatch")
    fp8 = k_cache.element_size() == 1
    _require(fp8 or k_cache.dtype == q3.dtype, "the KV cache must have the queries' 16-bit type, or be a one-byte fp8 type")
    _require(v_cache.dtype == k_cache.dtype, "k_cache / v_cache dtypes differ")
    sc, st, sh = _cache_strides(k_cache)
    _require(_cache_strides(v_cache) == (sc, st, sh), "k_cache / v_cache strides differ")
    _require(block_table.dtype == torch.int32 and block_table.dim() == 2 and block_table.stride(1) == 1, "bad block_table")
    _require(kv_lens.dtype == torch.int32 and kv_lens.is_contiguous(), "kv_lens must be contiguous int32")
    _require(block_table.size(0) >= R and kv_lens.numel() >= R, "block_table / kv_lens shorter than the batch")
    if fp8:
        _require(k_scales is not None and v_scales is not None, "fp8 cache needs k_scales and v_scales")
        _require(k_scales.dtype == torch.float32 and v_scales.dtype == torch.float32
                 and k_scales.is_contiguous() and v_scales.is_contiguous()
                 and tuple(k_scales.shape) == (N, Hkv) and tuple(v_scales.shape) == (N, Hkv),
                 "scales must be contiguous fp32 [N, Hkv]")
    o3 = _qo_view(out, "out")
    _require(tuple(o3.shape) == (R, Hq, D) and o3.dtype == q3.dtype, "out shape / dtype mismatch")
    if max_kv_len is None:
        max_kv_len = block_table.size(1) * C
    if softmax_scale is None:
        softmax_scale = D ** -0.5
    _lib.check(_native().abi_mi_paged_decode_attention_noalloc(
        q3.data_ptr(), q3.stride(0), q3.stride(1), k_cache.data_ptr(), v_cache.data_ptr(), sc, st, sh,
        block_table.data_ptr(), block_table.stride(0), kv_lens.data_ptr(), o3.data_ptr(), o3.stride(0), o3.stride(1),
        R, Hq, Hkv, D, C, int(max_kv_len), int(split_tokens), float(softmax_scale),
        MI_KV_FP8_E4M3 if fp8 else MI_KV_16BIT, k_scales, v_scales, _dtype_code(q3, "q"), _tuning_arg(),
        stream), "mi_paged_decode_attention_noalloc")
    return out


def paged_mla_decode_attention(q: Tensor, kv_cache: Tensor, kv_lens: Tensor, block_table: Tensor, *,
                               softmax_scale: float, head_dim_v: int = 512, max_kv_len: Optional[int] = None,
                               out: Optional[Tensor] = None) -> Tensor:
    """Absorbed multi-latent decode attention: ``q`` ``[R, (1,) Hq, 576]`` over the latent cache
    ``[N, C, 576]`` (or ``[N, C, 1, 576]``); returns ``[R, (1,) Hq, head_dim_v]``."""
    return _native().paged_mla_decode_attention(q, kv_cache, kv_lens, block_table, softmax_scale, head_dim_v, max_kv_len,
                                                out, _tuning_arg(), _override())


def paged_prefill_attention_mla(q: Tensor, k_cache: Tensor, v_cache: Tensor, cu_seqlens_q: Tensor, kv_lens: Tensor,
                                block_table: Tensor, *, softmax_scale: float, max_kv_len: Optional[int] = None,
                                out: Optional[Tensor] = None) -> Tensor:
    """Varlen causal attention over the decompressed caches of multi-latent attention: ``q`` ``[T, Hq, 192]``,
    ``k_cache`` ``[N, C, H, 192]``, ``v_cache`` ``[N, C, H, 128]`` (each with its own strides) -> ``[T, Hq, 128]``.
    ``max_kv_len`` (an upper bound of ``kv_lens``; default: what the block table can hold) sizes the split of
    the keys when few query rows meet long contexts."""
    return _native().paged_prefill_attention_mla(q, k_cache, v_cache, cu_seqlens_q, kv_lens, block_table, softmax_scale,
                                                 max_kv_len, out, _tuning_arg(), _override())


def paged_prefill_attention(q: Tensor, k_cache: Tensor, v_cache: Tensor, cu_seqlens_q: Tensor, kv_lens: Tensor,
                            block_table: Tensor, *, softmax_scale: Optional[float] = None,
                            max_kv_len: Optional[int] = None, out: Optional[Tensor] = None,
                            k_scales: Optional[Tensor] = None, v_scales: Optional[Tensor] = None,
                            one_row_requests: bool = True) -> Tensor:
    """Varlen causal attention of new tokens over the paged cache (bottom-right aligned mask).
    Byte caches with ``k_scales`` / ``v_scales`` ``[N, Hkv]`` select the fp8-e4m3 path.  ``one_row_requests=False``
    says that no request has exactly one query row, so the decode kernels need not be launched (a request that has
    one all the same is served by the tile kernel)."""
    return _native().paged_prefill_attention(q, k_cache, v_cache, cu_seqlens_q, kv_lens, block_table, softmax_scale,
                                             max_kv_len, out, k_scales, v_scales, _tuning_arg(), _override(),
                                             one_row_requests)


# ---------------------------------------------------------------------------------------------
# fused head norm + rotary embedding (+ append)
# ---------------------------------------------------------------------------------------------
def norm_rope_append(query: Optional[Tensor], key: Optional[Tensor], *, value: Optional[Tensor] = None,
                     q_weight: Optional[Tensor] = None, k_weight: Optional[Tensor] = None,
                     eps: float = 1e-5, norm: Optional[str] = None, rotary_emb: Optional[Tensor] = None,
                     q_positions: Optional[Tensor] = None, k_positions: Optional[Tensor] = None,
                     rotary_interleaved: bool = False, mscale: float = 1.0, query_out: Optional[Tensor] = None,
                     key_out: Optional[Tensor] = None,
                     k_cache: Optional[Tensor] = None, v_cache: Optional[Tensor] = None,
                     token_to_chunk_idx: Optional[Tensor] = None, token_to_local_pos: Optional[Tensor] = None,
                     block_table: Optional[Tensor] = None, kv_lens: Optional[Tensor] = None,
                     faithful_rounding: bool = True) -> None:
    """Norm (none / rms / l2) then RoPE on ``query`` (in place unless ``query_out`` is given) and on
    ``key`` (result to ``key_out`` and/or straight into the cache slot, together with ``value``)."""
    _native().norm_rope_append(query, key, value, q_weight, k_weight, eps, _NORM_KINDS[norm], rotary_emb, q_positions,
                               k_positions, rotary_interleaved, mscale, query_out, key_out, k_cache, v_cache,
                               token_to_chunk_idx, token_to_local_pos, block_table, kv_lens, faithful_rounding,
                               _tuning_arg())


def qkv_norm_rope_append(mixed_qkv: Tensor, *, num_query_heads: int, num_kv_heads: int, query_out: Tensor,
                         key_out: Optional[Tensor] = None, q_weight: Optional[Tensor] = None,
                         k_weight: Optional[Tensor] = None, eps: float = 1e-5, norm: Optional[str] = None,
                         rotary_emb: Optional[Tensor] = None, q_positions: Optional[Tensor] = None,
                         k_positions: Optional[Tensor] = None, rotary_interleaved: bool = False,
                         mscale: float = 1.0, k_cache: Optional[Tensor] = None, v_cache: Optional[Tensor] = None,
                         token_to_chunk_idx: Optional[Tensor] = None, token_to_local_pos: Optional[Tensor] = None,
                         block_table: Optional[Tensor] = None, kv_lens: Optional[Tensor] = None,
                         faithful_rounding: bool = True) -> None:
    """:func:`norm_rope_append` reading the QKV projection's output ``[T, (1,) (Hq + 2 Hkv) * d]`` (per
    query group: its query heads, then its key head, then its value head -- the layout that
    ``get_query_key_value_tensors`` splits, attention.py:985-1030) without materialising the split."""
    _native().qkv_norm_rope_append(mixed_qkv, num_query_heads, num_kv_heads, query_out, key_out, q_weight, k_weight, eps,
                                   _NORM_KINDS[norm], rotary_emb, q_positions, k_positions, rotary_interleaved, mscale,
                                   k_cache, v_cache, token_to_chunk_idx, token_to_local_pos, block_table, kv_lens,
                                   faithful_rounding, _tuning_arg())


def qkv_prefill_supported(head_dim: int, chunk_tokens: int, rotary_emb: Optional[Tensor]) -> bool:
    """Whether :func:`qkv_key_append` and :func:`qkv_prefill_attention` take these sizes: the one-stream tile kernel's,
    and every value of a head rotated (or none).  Tuning overrides ask for the separate calls."""
    return (head_dim in (64, 128) and chunk_tokens % 64 == 0 and _tuning_arg() is None
            and (rotary_emb is None or rotary_emb.size(-1) == head_dim))


def qkv_key_append(mixed_qkv: Tensor, *, num_query_heads: int, num_kv_heads: int, key_out: Optional[Tensor] = None,
                   k_weight: Optional[Tensor] = None, eps: float = 1e-5, norm: Optional[str] = None,
                   rotary_emb: Optional[Tensor] = None, q_positions: Optional[Tensor] = None,
                   k_positions: Optional[Tensor] = None, rotary_interleaved: bool = False, mscale: float = 1.0,
                   k_cache: Optional[Tensor] = None, v_cache: Optional[Tensor] = None,
                   token_to_chunk_idx: Optional[Tensor] = None,
                   token_to_local_pos: Optional[Tensor] = None) -> Optional[Tensor]:
    """The key / value half of :func:`qkv_norm_rope_append`.  Returns cos | sin of every row's query position
    (``None`` without ``rotary_emb``) for :func:`qkv_prefill_attention`, which does the queries' half."""
    return _native().qkv_key_append(mixed_qkv, num_query_heads, num_kv_heads, key_out, k_weight, eps, _NORM_KINDS[norm],
                                    rotary_emb, q_positions, k_positions, rotary_interleaved, mscale, k_cache, v_cache,
                                    token_to_chunk_idx, token_to_local_pos)


def qkv_prefill_attention(mixed_qkv: Tensor, k_cache: Tensor, v_cache: Tensor, cu_seqlens_q: Tensor, kv_lens: Tensor,
                          block_table: Tensor, *, num_query_heads: int, num_kv_heads: int, max_kv_len: int,
                          cos_sin: Optional[Tensor] = None, q_weight: Optional[Tensor] = None, eps: float = 1e-5,
                          norm: Optional[str] = None, rotary_interleaved: bool = False,
                          softmax_scale: Optional[float] = None, k_scales: Optional[Tensor] = None,
                          v_scales: Optional[Tensor] = None) -> Tensor:
    """:func:`paged_prefill_attention` without one-row requests over the raw queries of the QKV projection's output:
    head norm and rotation happen as the tile kernel loads them.  Returns ``[T, 1, Hq, d]``."""
    return _native().qkv_prefill_attention(mixed_qkv, num_query_heads, num_kv_heads, q_weight, eps, _NORM_KINDS[norm],
                                           cos_sin, rotary_interleaved, k_cache, v_cache, cu_seqlens_q, kv_lens,
                                           block_table, softmax_scale, max_kv_len, k_scales, v_scales, _override())


# ---------------------------------------------------------------------------------------------
# context bookkeeping on the GPU
# ---------------------------------------------------------------------------------------------
def decode_step_supported(head_dim: int, rot_dim: int, rotary_interleaved: bool, fp8_cache: bool) -> bool:
    """Whether :func:`decode_step_attention` has a kernel for these shapes (else: the separate calls)."""
    if head_dim not in (64, 96, 128, 192, 256) or (fp8_cache and head_dim != 128):
        return False
    # half-split pairs must sit a whole number of a lane's fragments apart (fp8 key bytes: 64 elements)
    return rot_dim == 0 or rotary_interleaved or (rot_dim // 2) % (64 if fp8_cache else 32) == 0


def decode_step_attention(query: Optional[Tensor], key: Optional[Tensor], value: Optional[Tensor], k_cache: Tensor,
                          v_cache: Tensor, kv_lens: Tensor, block_table: Tensor, *,
                          mixed_qkv: Optional[Tensor] = None, num_query_heads: int = 0, num_kv_heads: int = 0,
                          q_weight: Optional[Tensor] = None, k_weight: Optional[Tensor] = None, eps: float = 1e-5,
                          norm: Optional[str] = None, rotary_emb: Optional[Tensor] = None,
                          positions: Optional[Tensor] = None, rotary_interleaved: bool = False, mscale: float = 1.0,
                          softmax_scale: Optional[float] = None, max_kv_len: Optional[int] = None,
                          split_tokens: int = 0, out: Optional[Tensor] = None, workspace: Optional[Tensor] = None,
                          faithful_rounding: bool = True, k_scales: Optional[Tensor] = None,
                          v_scales: Optional[Tensor] = None, headroom: float = 2.0) -> Tensor:
    """One decode step of a layer in two launches: head norm + RoPE of the raw queries and of the step's new key
    rows, the append of the new key / value rows at position ``kv_lens - 1`` and the attention over the cache --
    what :func:`norm_rope_append` (or :func:`qkv_norm_rope_append`) followed by :func:`paged_decode_attention`
    computes.  Inputs: ``query`` ``[R, (1,) Hq, d]``, ``key`` / ``value`` ``[R, (1,) Hkv, d]``, or ``mixed_qkv``
    ``[R, (1,) (Hq + 2 Hkv) d]`` (the QKV projection's output) with the head counts.  Returns ``[R, (1,) Hq, d]``.
    Byte caches with ``k_scales`` / ``v_scales`` hold e4m3 values: the append then quantises like
    :func:`kv_append_decode_fp8` (``headroom`` as there)."""
    return _native().decode_step_attention(
        query, key, value, mixed_qkv, num_query_heads, num_kv_heads, k_cache, v_cache, kv_lens, block_table, q_weight,
        k_weight, eps, _NORM_KINDS[norm], rotary_emb, positions, rotary_interleaved, mscale, softmax_scale, max_kv_len,
        split_tokens, out, workspace, faithful_rounding, k_scales, v_scales, headroom, _tuning_arg(), _override())


def layer_views(buffer: Tensor, layer: int, pair: bool) -> Tuple[Tensor, Optional[Tensor]]:
    """New views ``buffer[0, layer], buffer[1, layer]`` of a buffer of keys and values, or ``buffer[layer], None``."""
    if buffer.is_cuda:
        return _native().layer_views(buffer, layer, pair)
    return (buffer[0, layer], buffer[1, layer]) if pair else (buffer[layer], None)  # (a context on the host: no library)


def watch(row: Tensor, index: int, value: int, microseconds: int) -> bool:
    """Whether ``row[index]`` (int32 in pinned host memory, written by a kernel) became anything but ``value`` within
    the time; other Python threads run meanwhile."""
    return _native().watch(row, index, value, microseconds)


# Words that the one workgroup of update_requests zeroes on the side: 256 KB take it 2 us or so, a launch of their own costs
# the host five; beyond, many workgroups are the faster way.
UPDATE_CLEARS_AT_MOST = 1 << 16


def update_requests(ctx, mask: Tensor, new_tokens_i64: Tensor, clear: Optional[Tensor] = None) -> None:
    """Enqueue the single-kernel ``update_requests`` on the state tensors of ``ctx`` (results land in
    ``ctx._counters``, pinned host memory, / ``ctx._newly_paused_buf`` / ``ctx._finished_ids_buf`` / ``ctx._paused_tokens_buf``).
    ``clear``: contiguous int32 rows that it zeroes too."""
    table = ctx.request_to_kv_chunk_ids
    _require(table.stride(1) == 1, "request_to_kv_chunk_ids rows must be contiguous")
    native = _native()
    ctx._counters_stream = native.written_by_kernel(ctx._counters, table.device.index)
    update, more = (native.abi_mi_update_requests if mask.dtype == torch.int32 else native.abi_mi_update_requests_mask8), ()
    if clear is not None:
        update, more = native.abi_mi_update_requests_clearing, (mask.element_size(), clear, clear.numel())
    _lib.check(update(
        ctx.request_ids, ctx.request_query_lengths, ctx.request_output_lengths,
        ctx.request_kv_length_offsets, ctx.request_kv_chunk_counts,
        ctx.request_last_kv_chunk_id, ctx.request_last_kv_chunk_offset,
        table, table.stride(0), table.size(1),
        ctx.token_to_input_ids, ctx.token_to_pos_ids, ctx.token_to_request_idx,
        ctx.token_to_position_in_request, ctx.token_to_chunk_idx,
        ctx.token_to_local_position_within_kv_chunk, ctx.chunk_allocator.chunk_bag,
        mask, new_tokens_i64, ctx._paused_tokens_buf,
        ctx._next_tokens_buf, ctx._update_scratch, ctx._newly_paused_buf,
        ctx._finished_ids_buf, ctx._counters, ctx.total_request_count, ctx.paused_request_count,
        ctx.chunk_allocator.chunk_count_avail, ctx.gtd_chunk_count, ctx.gtd_request_count,
        ctx.chunk_size_tokens, ctx.max_requests, *more, _stream(table)), "mi_update_requests")


def add_request(ctx, row: int, token_begin: int, tokens_i64: Tensor, n_chunks: int, stack_first: int,
                request_id: int, output_length: int) -> None:
    """The tensor writes of ``add_request`` in one launch: request row ``row``, its chunk-table entries
    ``chunk_bag[stack_first : stack_first + n_chunks]`` and the token rows from ``token_begin`` on."""
    table = ctx.request_to_kv_chunk_ids
    _require(tokens_i64.dtype == torch.int64 and tokens_i64.is_contiguous() and tokens_i64.device == table.device,
             "prompt tokens must be a contiguous int64 tensor on the context's device")
    _lib.check(_native().abi_mi_add_request(
        ctx.request_ids, ctx.request_query_lengths, ctx.request_output_lengths,
        ctx.request_kv_length_offsets, ctx.request_kv_chunk_counts,
        ctx.request_last_kv_chunk_id, ctx.request_last_kv_chunk_offset, table,
        table.stride(0), ctx.token_to_input_ids, ctx.token_to_pos_ids,
        ctx.token_to_request_idx, ctx.token_to_position_in_request,
        ctx.token_to_chunk_idx, ctx.token_to_local_position_within_kv_chunk,
        ctx.chunk_allocator.chunk_bag, tokens_i64, int(row), int(token_begin),
        tokens_i64.numel(), int(n_chunks), int(stack_first), ctx.chunk_size_tokens, int(request_id),
        int(output_length), _stream(table)), "mi_add_request")


def decode_attention_state(ctx, n_active_requests: int, padded_tokens: int) -> None:
    """Fill the fixed-address length / block-table mirrors and the padded token rows in one launch."""
    table = ctx.request_to_kv_chunk_ids
    mirror = ctx.request_to_kv_chunk_ids_cudagraph_only
    _lib.check(_native().abi_mi_decode_attention_state(
        ctx.request_kv_length_offsets, ctx.request_query_lengths, table,
        table.stride(0), table.size(1), ctx.query_seq_lengths_cudagraph_only,
        ctx.kv_seq_lengths_cudagraph_only, mirror, mirror.stride(0),
        ctx.token_to_chunk_idx, ctx.token_to_local_position_within_kv_chunk,
        ctx.token_to_position_in_request, ctx.paused_request_count, n_active_requests,
        ctx.active_token_count, padded_tokens, ctx.dummy_chunk_idx, _stream(table)), "mi_decode_attention_state")


def step_attention_state(ctx, n_active_requests: int, padded_requests: int, padded_tokens: int) -> None:
    """Prefill / mixed steps: the fixed-address mirrors of lengths, their running sums and the block table, the
    padded token rows and the two maxima (into ``ctx._max_lengths``) in one launch."""
    table = ctx.request_to_kv_chunk_ids
    mirror = ctx.request_to_kv_chunk_ids_cudagraph_only
    ctx._max_lengths_stream = _native().written_by_kernel(ctx._max_lengths, table.device.index)
    _lib.check(_native().abi_mi_step_attention_state(
        ctx.request_kv_length_offsets, ctx.request_query_lengths, table,
        table.stride(0), table.size(1), ctx.query_seq_lengths_cudagraph_only,
        ctx.kv_seq_lengths_cudagraph_only, ctx.cu_query_seq_lengths_cudagraph_only,
        ctx.cu_kv_seq_lengths_cudagraph_only, mirror, mirror.stride(0),
        ctx.token_to_chunk_idx, ctx.token_to_local_position_within_kv_chunk,
        ctx.token_to_position_in_request, ctx._max_lengths, ctx.paused_request_count,
        n_active_requests, padded_requests, ctx.active_token_count, padded_tokens, ctx.dummy_chunk_idx,
        _stream(table)), "mi_step_attention_state")


# ---------------------------------------------------------------------------------------------
# tail of a decode step: last-token rows, sampling, finished-request mask
# ---------------------------------------------------------------------------------------------
def last_token_gather(rows: Tensor, request_query_lengths: Tensor, out: Optional[Tensor] = None) -> Tensor:
    """``rows[cumsum(request_query_lengths) - 1]`` in one launch (``rows`` is ``[T, E]``; the
    lengths are those of the active requests, int32)."""
    return _native().last_token_gather(rows, request_query_lengths, out)


def selected_log_probs(logits: Tensor, token_ids: Tensor) -> Tensor:
    """``log_softmax(logits.float(), -1)[arange(T), token_ids]`` (fp32 ``[T]``) with one read of each row of
    ``logits`` ``[T, V]`` (fp32, bf16 or fp16) and no ``[T, V]`` intermediate."""
    return _native().selected_log_probs(logits, token_ids)


def sample_from_logits(logits: Tensor, *, top_k: int = 0, top_p: float = 0.0, temperature: float = 1.0,
                       uniform: Optional[Tensor] = None, vocab_size: Optional[int] = None,
                       termination_id: Optional[int] = None, kv_length_offsets: Optional[Tensor] = None,
                       query_lengths: Optional[Tensor] = None, output_lengths: Optional[Tensor] = None,
                       return_cut: bool = False):
    """Filter + draw per row of ``logits`` ``[R, V]`` (fp32, bf16 or fp16) and, when
    ``termination_id`` is given, the uint8 mask of requests that go on generating.

    Returns ``(samples int64 [R], mask uint8 [R] or None)`` and, with ``return_cut``, also the
    smallest kept value per row (fp32, -inf where nothing was filtered)."""
    return _native().sample_from_logits(logits, top_k, top_p, temperature, uniform, vocab_size or 0, termination_id,
                                        kv_length_offsets, query_lengths, output_lengths, return_cut, _override())


def attention_layer_decode(hidden: Tensor, qkv_weight: Tensor, qkv_bias: Optional[Tensor], proj_weight: Tensor,
                           proj_bias: Optional[Tensor], num_query_heads: int, num_kv_heads: int, k_cache: Tensor,
                           v_cache: Tensor, kv_lens: Tensor, block_table: Tensor, *, q_weight: Optional[Tensor] = None,
                           k_weight: Optional[Tensor] = None, eps: float = 1e-5, norm: Optional[str] = None,
                           rotary_emb: Optional[Tensor] = None, rotary_interleaved: bool = False,
                           softmax_scale: Optional[float] = None, max_kv_len: Optional[int] = None,
                           k_scales: Optional[Tensor] = None, v_scales: Optional[Tensor] = None,
                           headroom: float = 2.0) -> Tensor:
    """A decode step of one attention layer, hidden states ``[R, 1, hidden]`` in and out: :func:`linear_decode`,
    :func:`decode_step_attention` on its output and :func:`linear_decode` again, without returning to Python in
    between."""
    return _native().attention_layer_decode(
        hidden, qkv_weight, qkv_bias, proj_weight, proj_bias, num_query_heads, num_kv_heads, k_cache, v_cache, kv_lens,
        block_table, q_weight, k_weight, eps, _NORM_KINDS[norm], rotary_emb, rotary_interleaved, softmax_scale, max_kv_len,
        k_scales, v_scales, headroom, _tuning_arg(), _override())


def linear_decode(x: Tensor, weight: Tensor, bias: Optional[Tensor] = None, out: Optional[Tensor] = None) -> Tensor:
    """``x @ weight.T (+ bias)`` for a decode-sized step (at most 256 rows of ``x``): the weight matrix streams from
    HBM once.  ``x`` is ``[..., K]`` (leading dimensions are flattened to rows), ``weight`` ``[N, K]``; the result
    has ``x``'s leading dimensions and ``N`` columns; ``out`` may lie over ``x``.  What ``linear_qkv`` / ``linear_proj``
    of the attention layer compute at tensor-parallel size 1 (``mi_linear_decode`` of the header)."""
    return _native().linear_decode(x, weight, bias, out, _override())
