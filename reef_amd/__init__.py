"""reef_amd: int8 attention for AMD MI355X behind the reef_hip C ABI.

Host-side mirror of the Reef engine's quantization and attention operators
(inference-engine/reference/cpp/include/inference_engine/quant.hpp and
operator/attention.hpp), running on the HIP kernels of libreef_hip.so through
its C ABI (include/reef_hip/attention.h). Tensors are torch tensors on the GPU;
torch only provides device memory and the current stream. There is no CPU
fallback: without the built library every call raises.

Errors follow the engine: shape and argument errors raise InvalidArgument (a
ValueError, as the engine's std::invalid_argument), non-finite input raises
NonFiniteInput (also a ValueError, quant.hpp:72-74), cache capacity raises
CapacityError (an IndexError, the engine's std::length_error).
"""
from __future__ import annotations

import ctypes as C
import math
import os
import struct

PKG = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(PKG, "libreef_hip.so")

OK, INVALID_ARGUMENT, NON_FINITE_INPUT, CAPACITY, HIP_ERROR, UNSUPPORTED, OVERFLOW = range(7)
PER_TENSOR, PER_HEAD, PER_TOKEN = 0, 1, 2
ATTN_PRECISE_PV = 0x1
# prefill schedules (reef_attention_params.flags bits 4-6)
SCHED_AUTO, SCHED_ONE_ITEM, SCHED_SPLIT, SCHED_BALANCED, SCHED_PACKED = (0x00, 0x10, 0x20,
                                                                         0x30, 0x40)
PAGE = 16

EXPORTS = [
    "reef_quantize_int8_per_tensor", "reef_quantize_int8_per_head",
    "reef_quantize_int8_per_token", "reef_quantize_int8_per_token_heads",
    "reef_dequantize_int8", "reef_read_status_word",
    "reef_attention_prefill_workspace_bytes", "reef_attention_prefill_int8", "reef_qk_scores_i32",
    "reef_qk_scores_i32_packed_workspace_bytes", "reef_qk_scores_i32_packed",
    "reef_attention_decode_workspace_bytes", "reef_attention_decode_int8",
    "reef_attention_decode_int8_paged", "reef_attention_decode_int8_paged_noalloc",
    "reef_kv_pack_v_pages", "reef_kv_append_int8",
    "reef_kv_append_int8_paged", "reef_attention_int8_integer", "reef_linear_w8a8_workspace_bytes",
    "reef_linear_w8a8", "reef_gemm_w8a8", "reef_attention_prefill_cache_workspace_bytes",
    "reef_attention_prefill_int8_cache",
]


class ReefError(RuntimeError):
    pass


class InvalidArgument(ReefError, ValueError):
    pass


class NonFiniteInput(ReefError, ValueError):
    pass


class CapacityError(ReefError, IndexError):
    pass


class HipError(ReefError):
    pass


class Unsupported(ReefError, NotImplementedError):
    pass


class Overflow(ReefError, OverflowError):
    pass


_ERRORS = {INVALID_ARGUMENT: InvalidArgument, NON_FINITE_INPUT: NonFiniteInput,
           CAPACITY: CapacityError, HIP_ERROR: HipError, UNSUPPORTED: Unsupported,
           OVERFLOW: Overflow}


class Strides(C.Structure):
    _fields_ = [("batch", C.c_int64), ("head", C.c_int64), ("token", C.c_int64)]


class AttentionParams(C.Structure):
    _fields_ = [("batch", C.c_int64), ("q_heads", C.c_int64), ("kv_heads", C.c_int64),
                ("q_len", C.c_int64), ("kv_len", C.c_int64), ("head_dim", C.c_int64),
                ("query_start", C.c_int64), ("window", C.c_int64),
                ("softmax_scale", C.c_float), ("q_granularity", C.c_int32),
                ("kv_granularity", C.c_int32), ("flags", C.c_uint32)]


class DecodeParams(C.Structure):
    _fields_ = [("batch", C.c_int64), ("q_heads", C.c_int64), ("kv_heads", C.c_int64),
                ("head_dim", C.c_int64), ("max_context", C.c_int64), ("window", C.c_int64),
                ("softmax_scale", C.c_float), ("q_granularity", C.c_int32),
                ("num_splits", C.c_int32), ("flags", C.c_uint32)]


class KvAppendParams(C.Structure):
    _fields_ = [("batch", C.c_int64), ("kv_heads", C.c_int64), ("head_dim", C.c_int64),
                ("new_tokens", C.c_int64), ("max_context", C.c_int64)]


_P = C.c_void_p
_I64 = C.c_int64
_ST, _AP = C.POINTER(Strides), C.POINTER(AttentionParams)
_DP, _KP = C.POINTER(DecodeParams), C.POINTER(KvAppendParams)
_SIGS = {
    "reef_quantize_int8_per_tensor": [_P, _I64, _P, _P, _P, _P],
    "reef_quantize_int8_per_head": [_P, _I64, _I64, _I64, _I64, _ST, _P, _P, _P, _P],
    "reef_quantize_int8_per_token": [_P, _I64, _I64, _I64, _P, _P, _P, _P],
    "reef_quantize_int8_per_token_heads": [_P, _I64, _I64, _I64, _I64, _ST, _P, _P, _P, _P],
    "reef_dequantize_int8": [_P, _I64, _I64, _P, _P, _P],
    "reef_read_status_word": [_P, C.c_int, _P],
    "reef_attention_prefill_workspace_bytes": [_AP],
    "reef_attention_prefill_int8": [_AP, _P, _ST, _P, _ST, _P, _ST, _P, _P, _P, _P, _ST, _P,
                                    C.c_size_t, _P],
    "reef_qk_scores_i32": [_P, _P, _I64, _I64, _I64, _I64, _I64, _I64, _P, _P],
    "reef_qk_scores_i32_packed_workspace_bytes": [_I64, _I64, _I64, _I64, _I64],
    "reef_qk_scores_i32_packed": [_P, _P, _I64, _I64, _I64, _I64, _I64, _P, _P, C.c_size_t, _P],
    "reef_attention_decode_workspace_bytes": [_DP],
    "reef_attention_decode_int8": [_DP, _P, _P, _P, _P, _P, _P, _P, _P, _P, C.c_size_t, _P,
                                   _P],
    "reef_attention_decode_int8_paged": [_DP, _P, _P, _P, _P, _P, _P, _P,
                                         _I64, _I64, _P, _P, _P, C.c_size_t, _P, _P],
    "reef_attention_decode_int8_paged_noalloc": [_DP, _P, _P, _P, _P, _P, _P,
                                                 _P, _I64, _I64, _P, _P, _P, _P],
    "reef_kv_pack_v_pages": [_P, _I64, _I64, _P, _P],
    "reef_linear_w8a8_workspace_bytes": [_I64, _I64],
    "reef_linear_w8a8": [_P, _I64, _I64, _I64, _P, _P, _P, _I64, _P, _I64, _P, C.c_size_t, _P,
                         _P],
    "reef_gemm_w8a8": [_P, _P, _I64, _I64, _P, _P, _P, _I64, _P, _I64, _P, _P],
    "reef_attention_int8_integer": [_AP, _P, _ST, _P, _ST, _P, _ST, C.c_uint32, _P, C.c_uint32,
                                    _P, _ST, _P],
    "reef_kv_append_int8": [_KP, _P, _ST, _P, _ST, _P, _P, _P, _P, _P, _P, _P, _P],
    "reef_kv_append_int8_paged": [_KP, _P, _ST, _P, _ST, _P, _P, _I64, _I64, _P, _P, _P, _P, _P,
                                  _P, _P],
    "reef_attention_prefill_cache_workspace_bytes": [_AP],
    "reef_attention_prefill_int8_cache": [_AP, _P, _ST, _P, _P, _P, _P, _P, _I64, _P, _I64, _I64,
                                          _P, _ST, _P, C.c_size_t, _P, _P],
}

_lib_handle = _plain_handle = None


def _load(plain: bool) -> C.CDLL:
    if not os.path.exists(LIB_PATH):
        raise RuntimeError(f"{LIB_PATH} is missing: build it with python -m reef_amd._build")
    handle = C.CDLL(LIB_PATH)
    for name, args in _SIGS.items():
        fn = getattr(handle, name)
        fn.argtypes = [_P if plain and issubclass(t, C._Pointer) else t for t in args]
        fn.restype = C.c_size_t if name.endswith("_bytes") else C.c_int
    return handle


def lib() -> C.CDLL:
    """The loaded libreef_hip.so. Raises if it has not been built."""
    global _lib_handle
    if _lib_handle is None:
        _lib_handle = _load(plain=False)
    return _lib_handle


def _lib() -> C.CDLL:
    """The same library with structures as plain addresses, for the wrappers below."""
    global _plain_handle
    if _plain_handle is None:
        _plain_handle = _load(plain=True)
    return _plain_handle


def check(status: int, what: str) -> None:
    if status != OK:
        raise _ERRORS.get(status, ReefError)(f"{what}: reef status {status}")


# --- torch plumbing -------------------------------------------------------------------

# The wrappers below run once per layer and token of a serving loop, so the small calls are
# bound by this file: arguments go to the library as plain addresses and packed bytes
# (a ctypes structure costs four times its bytes), and the stream is read as a handle
# rather than through a torch.cuda.Stream (a 1x1x128x64 prefill: 11.4 us a call against
# 20.5, of which 8 us are the kernel's).

_torch_module = None


def _torch():
    global _torch_module
    if _torch_module is None:
        import torch
        _torch_module = torch
    return _torch_module


def _stream():
    """The current device's current stream, as an address."""
    c = _torch()._C
    try:
        return c._cuda_getCurrentRawStream(c._cuda_getDevice())
    except AttributeError:
        return _torch().cuda.current_stream().cuda_stream


def _ptr(t):
    return t.data_ptr() if t is not None else None


def _packed(layout, structure, *fields):
    """The bytes of `structure` (whose members `layout` gives) for the library to read."""
    try:
        return layout.pack(*fields)
    except (struct.error, OverflowError):  # a value outside its member's range
        return C.byref(structure(*fields))


_STRIDES = struct.Struct("=3q")
_ATTENTION = struct.Struct("=8qf2iI")
_DECODE = struct.Struct("=6qf2iI")
_APPEND = struct.Struct("=5q")


def _require(t, dtype, name):
    torch = _torch()
    if isinstance(t, torch.Tensor) and t.is_cuda:
        if t.dtype == dtype:
            return
        raise InvalidArgument(f"{name} must be {dtype}, got {t.dtype}")
    raise InvalidArgument(f"{name} must be a GPU tensor")


def _strides4(t):
    """Strides of a [B, H, S, D] tensor with a contiguous last dimension."""
    st = t.stride()
    if len(st) != 4 or st[3] != 1:
        raise InvalidArgument("expected [batch, heads, tokens, head_dim] with contiguous head_dim")
    return _STRIDES.pack(st[0], st[1], st[2])


class StatusWord:
    """A device status word the kernels flag non-finite input and bad pages in."""

    def __init__(self, device=None):
        torch = _torch()
        self.tensor = torch.zeros(1, dtype=torch.int32, device=device or "cuda")

    @property
    def ptr(self):
        return C.c_void_p(self.tensor.data_ptr())

    def check(self, what: str) -> None:
        check(_lib().reef_read_status_word(self.ptr, 1, _stream()), what)


# --- quantization (quant.hpp) ---------------------------------------------------------

def quantize_per_tensor(x, status: StatusWord | None = None):
    """One scale for the whole tensor (the quant.hpp rule); returns (int8, scale[1])."""
    torch = _torch()
    _require(x, torch.float32, "x")
    x = x.contiguous()
    q = torch.empty(x.shape, dtype=torch.int8, device=x.device)
    s = torch.empty(1, dtype=torch.float32, device=x.device)
    own = status or StatusWord(x.device)
    check(_lib().reef_quantize_int8_per_tensor(_ptr(x), x.numel(), _ptr(q), _ptr(s), _ptr(own.tensor),
                                              _stream()), "quantize_per_tensor")
    if status is None:
        own.check("quantize_per_tensor requires finite values")
    return q, s


def quantize_per_head(x, status: StatusWord | None = None):
    """x [B, H, S, D] (any strides, contiguous D); one scale per head over batch and
    tokens. Returns packed int8 [B, H, S, D] and scales [H]."""
    torch = _torch()
    _require(x, torch.float32, "x")
    st = _strides4(x)
    B, H, S, D = x.shape
    q = torch.empty((B, H, S, D), dtype=torch.int8, device=x.device)
    s = torch.empty(H, dtype=torch.float32, device=x.device)
    own = status or StatusWord(x.device)
    check(_lib().reef_quantize_int8_per_head(_ptr(x), B, H, S, D, st, _ptr(q), _ptr(s),
                                            _ptr(own.tensor), _stream()), "quantize_per_head")
    if status is None:
        own.check("quantize_per_head requires finite values")
    return q, s


def quantize_rows(x, status: StatusWord | None = None):
    """quantize_rows (quant.hpp:112-133) over the last dimension: one scale per row
    (per token). Returns int8 of x's shape and scales of x.shape[:-1]."""
    torch = _torch()
    _require(x, torch.float32, "x")
    shape = x.shape
    width = shape[-1]
    if len(shape) == 4 and not x.is_contiguous() and x.numel() > 0:
        # heads as a projection lays them out: read in place rather than copied first
        sb, sh, st, sd = x.stride()
        if sd == 1 and (sb | sh | st | width) % 4 == 0 and width <= 1024 and x.data_ptr() % 16 == 0:
            q = torch.empty(shape, dtype=torch.int8, device=x.device)
            s = torch.empty(shape[:-1], dtype=torch.float32, device=x.device)
            own = status or StatusWord(x.device)
            ret = _lib().reef_quantize_int8_per_token_heads(
                _ptr(x), *shape, _STRIDES.pack(sb, sh, st), _ptr(q), _ptr(s), _ptr(own.tensor),
                _stream())
            if ret != UNSUPPORTED:  # 2^31 rows or more are copied
                check(ret, "quantize_rows")
                if status is None:
                    own.check("quantize_rows requires finite values")
                return q, s
            del q, s
    x2 = x if len(shape) == 2 else x.reshape(-1, width)
    if x2.stride(1) != 1:
        x2 = x2.contiguous()
    rows = x2.shape[0]
    q = torch.empty(shape, dtype=torch.int8, device=x.device)
    s = torch.empty(shape[:-1], dtype=torch.float32, device=x.device)
    own = status or StatusWord(x.device)
    check(_lib().reef_quantize_int8_per_token(_ptr(x2), rows, width, x2.stride(0), _ptr(q),
                                             _ptr(s), _ptr(own.tensor), _stream()), "quantize_rows")
    if status is None:
        own.check("quantize_rows requires finite values")
    return q, s


quantize_per_token = quantize_rows


def dequantize(q, scales, group: int):
    """x[i] = float(q[i]) * scales[i // group]."""
    torch = _torch()
    _require(q, torch.int8, "q")
    _require(scales, torch.float32, "scales")
    q = q.contiguous()
    x = torch.empty(q.shape, dtype=torch.float32, device=q.device)
    scales = scales.contiguous()
    check(_lib().reef_dequantize_int8(_ptr(q), q.numel(), group, _ptr(scales), _ptr(x),
                                     _stream()), "dequantize")
    return x


# --- attention ------------------------------------------------------------------------

_PREFILL_WS = {}


def prefill_workspace(params: AttentionParams, device):
    """The zero-filled workspace of the balanced prefill schedule, one per (device,
    stream): every launch leaves it zero-filled, so the next launch on that stream
    reuses it."""
    n = lib().reef_attention_prefill_workspace_bytes(C.byref(params))
    return _prefill_workspace(n, _torch().device(device), _stream())


def _prefill_workspace(n, device, stream):
    key = (device.index, stream)
    ws = _PREFILL_WS.get(key)
    if ws is None or ws.numel() < n:
        torch = _torch()
        ws = torch.zeros(max(n, 256), dtype=torch.uint8, device=device)
        _PREFILL_WS[key] = ws
    return ws


def attention_prefill(q, k, v, q_scales, k_scales, v_scales, *, query_start=None, window=0,
                      softmax_scale=None, q_granularity=PER_HEAD, kv_granularity=PER_HEAD,
                      precise=False, schedule=SCHED_AUTO, out=None, workspace=None):
    """Attention::context (attention.hpp:374-432) over int8 heads in one launch.

    q [B, Hq, Sq, D], k and v [B, Hkv, Skv, D] int8 (contiguous head_dim, any other
    strides); scales by granularity. softmax_scale defaults to 1/sqrt(D); pass 1.0
    for the engine's unscaled scores. Returns fp32 [B, Hq, Sq, D]. schedule is one
    of the SCHED_* flags (SCHED_AUTO: the library's choice). workspace: None takes
    this stream's cached one (prefill_workspace), False passes none, or a
    zero-filled uint8 tensor of reef_attention_prefill_workspace_bytes bytes.
    """
    torch = _torch()
    for t, n in ((q, "q"), (k, "k"), (v, "v")):
        _require(t, torch.int8, n)
    for t, n in ((q_scales, "q_scales"), (k_scales, "k_scales"), (v_scales, "v_scales")):
        _require(t, torch.float32, n)
    B, Hq, Sq, D = q.shape
    _, Hkv, Skv, _ = k.shape
    if tuple(v.shape) != tuple(k.shape) or k.shape[0] != B or k.shape[3] != D:
        raise InvalidArgument("attention_prefill shape mismatch")
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(D)
    start = Skv - Sq if query_start is None else query_start
    p = _packed(_ATTENTION, AttentionParams, B, Hq, Hkv, Sq, Skv, D, start, window, softmax_scale,
                q_granularity, kv_granularity, (ATTN_PRECISE_PV if precise else 0) | schedule)
    device = q.device
    if out is None:
        out = torch.empty((B, Hq, Sq, D), dtype=torch.float32, device=device)
    qs, ks, vs, os_ = _strides4(q), _strides4(k), _strides4(v), _strides4(out)
    stream = _stream()
    if workspace is None:
        n = _lib().reef_attention_prefill_workspace_bytes(p)
        workspace = _prefill_workspace(n, device, stream)
    ws_ptr, ws_n = (None, 0) if workspace is False else (_ptr(workspace), workspace.numel()
                                                          * workspace.element_size())
    # (named, so that a copy that contiguous() makes lives until the launch is queued)
    q_scales, k_scales, v_scales = (q_scales.contiguous(), k_scales.contiguous(),
                                    v_scales.contiguous())
    check(_lib().reef_attention_prefill_int8(
        p, _ptr(q), qs, _ptr(k), ks, _ptr(v), vs, _ptr(q_scales), _ptr(k_scales), _ptr(v_scales),
        _ptr(out), os_, ws_ptr, ws_n, stream), "attention_prefill")
    return out


def attention_prefill_cache(q, q_scales, k_cache, v_cache, k_scales, v_scales, kv_len, *,
                            block_table=None, query_start=None, window=0, softmax_scale=None,
                            q_granularity=PER_HEAD, status: StatusWord | None = None, out=None):
    """A prompt chunk over the int8 cache (Attention::forward with query_len > 1 on a
    non-empty cache, attention.hpp:354-372): the cache already holds the chunk's
    keys (kv_append), kv_len tokens per sequence. Contiguous cache (block_table
    None): k_cache [B, Hkv, L, D], v_cache [B, Hkv, L/16, D, 16] (or the same bytes
    in any shape), scales [B, Hkv, L]. Paged: k_cache [P, Hkv, 16, D], v_cache
    [P, Hkv, D, 16], scales [P, Hkv, 16], block_table [B, max_blocks] int32.
    q [B, Hq, q_len, D] int8; returns fp32 [B, Hq, q_len, D]."""
    torch = _torch()
    _require(q, torch.int8, "q")
    B, Hq, Sq, D = q.shape
    Hkv = k_cache.shape[1]
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(D)
    start = kv_len - Sq if query_start is None else query_start
    p = _packed(_ATTENTION, AttentionParams, B, Hq, Hkv, Sq, kv_len, D, start, window,
                softmax_scale, q_granularity, PER_TOKEN, 0)
    if block_table is None:
        max_context, table, max_blocks, pages = k_cache.shape[2], None, 0, 0
    else:
        max_context, table = 0, block_table.contiguous()
        max_blocks, pages = table.shape[1], k_cache.shape[0]
    n = _lib().reef_attention_prefill_cache_workspace_bytes(p)
    device, stream = q.device, _stream()
    key = ("cache", device.index, stream)
    ws = _PREFILL_WS.get(key)
    if ws is None or ws.numel() < n:  # zero-filled once; every call leaves it so
        ws = torch.zeros(max(n, 256), dtype=torch.uint8, device=device)
        _PREFILL_WS[key] = ws
    if out is None:
        out = torch.empty((B, Hq, Sq, D), dtype=torch.float32, device=q.device)
    qs, os_ = _strides4(q), _strides4(out)
    own = status or StatusWord(q.device)
    q_scales, k_cache, v_cache = q_scales.contiguous(), k_cache.contiguous(), v_cache.contiguous()
    k_scales, v_scales = k_scales.contiguous(), v_scales.contiguous()
    check(_lib().reef_attention_prefill_int8_cache(
        p, _ptr(q), qs, _ptr(q_scales), _ptr(k_cache), _ptr(v_cache), _ptr(k_scales),
        _ptr(v_scales), max_context, _ptr(table), max_blocks, pages, _ptr(out), os_, _ptr(ws), n,
        _ptr(own.tensor), stream), "attention_prefill_cache")
    if status is None:
        own.check("attention_prefill_cache")
    return out


def qk_scores_i32(q, k):
    """int32 q . k^T for packed q [B, Hq, Sq, D] and k [B, Hkv, Skv, D]."""
    torch = _torch()
    _require(q, torch.int8, "q")
    _require(k, torch.int8, "k")
    q = q.contiguous()
    k = k.contiguous()
    B, Hq, Sq, D = q.shape
    Hkv, Skv = k.shape[1], k.shape[2]
    acc = torch.empty((B, Hq, Sq, Skv), dtype=torch.int32, device=q.device)
    check(_lib().reef_qk_scores_i32(_ptr(q), _ptr(k), B, Hq, Hkv, Sq, Skv, D, _ptr(acc),
                                   _stream()), "qk_scores_i32")
    return acc


def qk_scores_i32_packed(q, k):
    """int32 q . k^T for packed q [B, Hq, Sq, 128] and k [B, Hkv, Skv, 128], read from
    the packed prefill kernel's own score accumulators."""
    torch = _torch()
    _require(q, torch.int8, "q")
    _require(k, torch.int8, "k")
    q = q.contiguous()
    k = k.contiguous()
    B, Hq, Sq, D = q.shape
    Hkv, Skv = k.shape[1], k.shape[2]
    if D != 128:
        raise ValueError("the packed score hook takes head_dim 128")
    acc = torch.full((B, Hq, Sq, Skv), -1, dtype=torch.int32, device=q.device)
    nbytes = _lib().reef_qk_scores_i32_packed_workspace_bytes(B, Hq, Hkv, Sq, Skv)
    if nbytes == 0:
        raise ValueError("qk_scores_i32_packed: invalid sizes")
    ws = torch.zeros(nbytes, dtype=torch.uint8, device=q.device)
    check(_lib().reef_qk_scores_i32_packed(_ptr(q), _ptr(k), B, Hq, Hkv, Sq, Skv, _ptr(acc),
                                          _ptr(ws), nbytes, _stream()), "qk_scores_i32_packed")
    return acc


def _decode_bytes(q, max_context, kv_heads, window, softmax_scale, q_granularity, num_splits):
    B, Hq, D = q.shape
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(D)
    return _packed(_DECODE, DecodeParams, B, Hq, kv_heads, D, max_context, window, softmax_scale,
                   q_granularity, num_splits, 0)


def _decode_params(q, max_context, kv_heads, window, softmax_scale, q_granularity, num_splits):
    B, Hq, D = q.shape
    if softmax_scale is None:
        softmax_scale = 1.0 / math.sqrt(D)
    return DecodeParams(B, Hq, kv_heads, D, max_context, window, softmax_scale, q_granularity,
                        num_splits, 0)


def decode_workspace(params: DecodeParams, device):
    """A zero-filled decode workspace (its item counters must start at zero; every
    launch leaves them so, so the workspace is reusable without refilling)."""
    return _decode_workspace(lib().reef_attention_decode_workspace_bytes(C.byref(params)), device)


def _decode_workspace(n, device):
    torch = _torch()
    return torch.zeros(max(n, 16) // 4 + 4, dtype=torch.float32, device=device)


def attention_decode(q, q_scales, k_cache, v_pages, k_scales, v_scales, context_lens=None, *,
                     window=0, softmax_scale=None, q_granularity=PER_TOKEN, num_splits=0,
                     workspace=None, status: StatusWord | None = None, out=None):
    """One decode step over a contiguous int8 cache.

    q [B, Hq, D] int8; k_cache [B, Hkv, L, D]; v_pages [B, Hkv, L/16, D, 16] (see
    pack_v_pages); k_scales, v_scales [B, Hkv, L]; context_lens [B] int32 or None.
    """
    torch = _torch()
    _require(q, torch.int8, "q")
    B, Hq, D = q.shape
    Hkv, L = k_cache.shape[1], k_cache.shape[2]
    if tuple(k_cache.shape) != (B, Hkv, L, D) or v_pages.numel() != k_cache.numel():
        raise InvalidArgument("attention_decode cache shape mismatch")
    p = _decode_bytes(q, L, Hkv, window, softmax_scale, q_granularity, num_splits)
    ws = workspace
    if ws is None:
        ws = _decode_workspace(_lib().reef_attention_decode_workspace_bytes(p), q.device)
    if out is None:
        out = torch.empty((B, Hq, D), dtype=torch.float32, device=q.device)
    own = status or StatusWord(q.device)
    cl = context_lens.contiguous() if context_lens is not None else None
    q, q_scales, k_cache, v_pages = (q.contiguous(), q_scales.contiguous(), k_cache.contiguous(),
                                     v_pages.contiguous())
    k_scales, v_scales = k_scales.contiguous(), v_scales.contiguous()
    check(_lib().reef_attention_decode_int8(
        p, _ptr(q), _ptr(q_scales), _ptr(k_cache), _ptr(v_pages), _ptr(k_scales), _ptr(v_scales),
        _ptr(cl), _ptr(out), _ptr(ws), ws.numel() * 4, _ptr(own.tensor), _stream()), "attention_decode")
    if status is None:
        own.check("attention_decode")
    return out


def attention_decode_paged(q, q_scales, k_pages, v_pages, k_scale_pages, v_scale_pages,
                           block_table, context_lens, *, window=0, softmax_scale=None,
                           q_granularity=PER_TOKEN, num_splits=0, workspace=None,
                           status: StatusWord | None = None, out=None):
    """One decode step over a paged int8 cache: k_pages [P, Hkv, 16, D], v_pages
    [P, Hkv, D, 16], scale pages [P, Hkv, 16], block_table [B, max_blocks] int32,
    context_lens [B] int32."""
    torch = _torch()
    _require(q, torch.int8, "q")
    B, Hq, D = q.shape
    P, Hkv = k_pages.shape[0], k_pages.shape[1]
    max_blocks = block_table.shape[1]
    p = _decode_bytes(q, max_blocks * PAGE, Hkv, window, softmax_scale, q_granularity, num_splits)
    ws = workspace
    if ws is None:
        ws = _decode_workspace(_lib().reef_attention_decode_workspace_bytes(p), q.device)
    if out is None:
        out = torch.empty((B, Hq, D), dtype=torch.float32, device=q.device)
    own = status or StatusWord(q.device)
    q, q_scales, block_table, context_lens = (q.contiguous(), q_scales.contiguous(),
                                              block_table.contiguous(), context_lens.contiguous())
    check(_lib().reef_attention_decode_int8_paged(
        p, _ptr(q), _ptr(q_scales), _ptr(k_pages), _ptr(v_pages), _ptr(k_scale_pages),
        _ptr(v_scale_pages), _ptr(block_table), max_blocks, P, _ptr(context_lens), _ptr(out),
        _ptr(ws), ws.numel() * 4, _ptr(own.tensor), _stream()), "attention_decode_paged")
    if status is None:
        own.check("attention_decode_paged")
    return out


def pack_v_pages(v_tokens):
    """Token-major values [..., pages * 16, D] -> transposed pages [..., pages, D, 16]."""
    torch = _torch()
    _require(v_tokens, torch.int8, "v_tokens")
    *lead, L, D = v_tokens.shape
    if L % PAGE:
        raise InvalidArgument("token count must be a multiple of 16")
    src = v_tokens.contiguous()
    pages = src.numel() // (PAGE * D)
    out = torch.empty((*lead, L // PAGE, D, PAGE), dtype=torch.int8, device=src.device)
    check(_lib().reef_kv_pack_v_pages(_ptr(src), pages, D, _ptr(out), _stream()), "pack_v_pages")
    return out


# --- KV-cache append (attention.hpp:290-352) --------------------------------------------

def _append_inputs(k_new, v_new):
    torch = _torch()
    _require(k_new, torch.float32, "k_new")
    _require(v_new, torch.float32, "v_new")
    if k_new.shape != v_new.shape or k_new.dim() != 4:
        raise InvalidArgument("KV cache append shape mismatch")
    return _strides4(k_new), _strides4(v_new)


def kv_append(k_new, v_new, start_positions, k_cache, v_pages, k_scales, v_scales,
              context_lens=None, status: StatusWord | None = None):
    """Quantize fp32 rows k_new, v_new [B, Hkv, T, D] per token and write them into
    the contiguous cache (k_cache [B, Hkv, L, D], v_pages [B, Hkv, L/16, D, 16],
    scales [B, Hkv, L]) at start_positions[b] + t. context_lens, when given, is set
    to start_positions + T afterwards (it may be start_positions itself)."""
    torch = _torch()
    ks, vs = _append_inputs(k_new, v_new)
    B, H, T, D = k_new.shape
    L = k_cache.shape[2]
    if tuple(k_cache.shape) != (B, H, L, D) or v_pages.numel() != k_cache.numel():
        raise InvalidArgument("KV cache append shape mismatch")
    _require(start_positions, torch.int32, "start_positions")
    p = _packed(_APPEND, KvAppendParams, B, H, D, T, L)
    own = status or StatusWord(k_new.device)
    check(_lib().reef_kv_append_int8(
        p, _ptr(k_new), ks, _ptr(v_new), vs, _ptr(start_positions),
        _ptr(k_cache), _ptr(v_pages), _ptr(k_scales), _ptr(v_scales), _ptr(context_lens),
        _ptr(own.tensor), _stream()), "kv_append")
    if status is None:
        own.check("kv_append")


def kv_append_paged(k_new, v_new, start_positions, block_table, k_pages, v_pages,
                    k_scale_pages, v_scale_pages, context_lens=None,
                    status: StatusWord | None = None, max_context=None):
    """kv_append into the paged cache (k_pages [P, Hkv, 16, D], v_pages [P, Hkv, D, 16],
    scale pages [P, Hkv, 16], block_table [B, max_blocks] int32)."""
    torch = _torch()
    ks, vs = _append_inputs(k_new, v_new)
    B, H, T, D = k_new.shape
    P = k_pages.shape[0]
    max_blocks = block_table.shape[1]
    _require(start_positions, torch.int32, "start_positions")
    _require(block_table, torch.int32, "block_table")
    p = _packed(_APPEND, KvAppendParams, B, H, D, T, max_context or max_blocks * PAGE)
    block_table = block_table.contiguous()
    own = status or StatusWord(k_new.device)
    check(_lib().reef_kv_append_int8_paged(
        p, _ptr(k_new), ks, _ptr(v_new), vs, _ptr(start_positions), _ptr(block_table), max_blocks, P, _ptr(k_pages), _ptr(v_pages),
        _ptr(k_scale_pages), _ptr(v_scale_pages), _ptr(context_lens), _ptr(own.tensor), _stream()),
        "kv_append_paged")
    if status is None:
        own.check("kv_append_paged")


# --- integer-only attention (int8.hpp:156-279) -----------------------------------------

def attention_int8_integer(q, k, v, table, *, score_shift, out_shift=8, query_start=None,
                           window=0):
    """attend_head_int8 for every (batch, head): q [B, Hq, Sq, D], k and v
    [B, Hkv, Skv, D] int8, table [256] uint16 (as int16/uint16 torch tensor) on the
    device; returns int8 [B, Hq, Sq, D], bit-identical to the engine."""
    torch = _torch()
    for t, n in ((q, "q"), (k, "k"), (v, "v")):
        _require(t, torch.int8, n)
    if table.numel() != 256 or table.element_size() != 2 or not table.is_cuda:
        raise InvalidArgument("table must hold 256 16-bit entries on the GPU")
    B, Hq, Sq, D = q.shape
    Hkv, Skv = k.shape[1], k.shape[2]
    start = Skv - Sq if query_start is None else query_start
    p = _packed(_ATTENTION, AttentionParams, B, Hq, Hkv, Sq, Skv, D, start, window, 1.0, PER_HEAD,
                PER_HEAD, 0)
    out = torch.empty((B, Hq, Sq, D), dtype=torch.int8, device=q.device)
    sq, sk, sv, so = _strides4(q), _strides4(k), _strides4(v), _strides4(out)
    table = table.contiguous()
    check(_lib().reef_attention_int8_integer(
        p, _ptr(q), sq, _ptr(k), sk, _ptr(v), sv, score_shift, _ptr(table), out_shift, _ptr(out),
        so, _stream()), "attention_int8_integer")
    return out


# --- W8A8 projection (operator/linear.hpp:106-132) ---------------------------------------

def linear_w8a8(x, weight, w_scales, bias=None, status: StatusWord | None = None):
    """y = linear(x, QuantizedWeight{weight, w_scales}, bias): x [rows, in] fp32,
    weight [out, in] int8, w_scales [out] fp32, bias [out] fp32 or None. Rows are
    quantized per row on the device; outputs are bit-identical to the engine's."""
    torch = _torch()
    _require(x, torch.float32, "x")
    _require(weight, torch.int8, "weight")
    _require(w_scales, torch.float32, "w_scales")
    if x.dim() != 2 or x.stride(1) != 1 or weight.dim() != 2 or weight.shape[1] != x.shape[1]:
        raise InvalidArgument("linear_w8a8 shapes: x [rows, in], weight [out, in]")
    rows, fin = x.shape
    fout = weight.shape[0]
    n = _lib().reef_linear_w8a8_workspace_bytes(rows, fin)
    ws = torch.empty(n // 4 + 4, dtype=torch.float32, device=x.device)
    y = torch.empty((rows, fout), dtype=torch.float32, device=x.device)
    own = status or StatusWord(x.device)
    weight, w_scales = weight.contiguous(), w_scales.contiguous()
    bias = bias.contiguous() if bias is not None else None
    check(_lib().reef_linear_w8a8(
        _ptr(x), rows, fin, x.stride(0), _ptr(weight), _ptr(w_scales), _ptr(bias), fout, _ptr(y),
        fout, _ptr(ws), ws.numel() * 4, _ptr(own.tensor), _stream()), "linear_w8a8")
    if status is None:
        own.check("linear_w8a8")
    return y
