"""Host-side mirror of the reference's fused attention API on torch device tensors.

The reference exposes three functions over candle tensors
(crates/ffai-mercury/src/asr/flash_attn.rs):

* ``serves(kt, v) -> bool``                       (:103-129)
* ``attend(q, kt, v, masked) -> Option<Tensor>``   (:212-264, FlashAttnOp :266-413)
* ``attend_merged(q, kt, v) -> Option<Tensor>``    (:131-158, MergedAttnOp :160-210)

This module keeps those names, argument meanings and the decline contract (``None`` where the
reference returns ``Ok(None)``; an exception where it returns ``Err``), and forwards to the C ABI
(``include/ffai_attn.h``) on the caller's current HIP stream. ``attention`` exposes the general
descriptor entry point (batch, bf16/f16, grouped K/V heads, head_dim 128, causal with offset,
ragged key counts, K/V shared across the batch). Torch only provides device memory and streams.
"""

from __future__ import annotations

import ctypes
import struct
from typing import Optional, Sequence

import torch

from . import _lib as L

_DT = {torch.float32: L.F32, torch.float16: L.F16, torch.bfloat16: L.BF16}
_TORCH_DT = {v: k for k, v in _DT.items()}
_VIEW = struct.Struct("@Qii4q4q")  # ffai_tensor's fields
_view_of = L.TensorView.from_buffer_copy


def _stream_handle(t: Optional[torch.Tensor] = None) -> ctypes.c_void_p:
    """The caller's current HIP stream (None for host tensors, which the library declines
    before touching any stream)."""
    if t is not None and not t.is_cuda:
        return ctypes.c_void_p(None)
    if torch.cuda.is_initialized():
        # the handle itself, without a Stream object around it (0.1 against 2.7 us: an eager
        # decode call is bound by its host time)
        return ctypes.c_void_p(torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice()))
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def _view(t: torch.Tensor) -> L.TensorView:
    if t.dim() > 4:
        raise ValueError("tensor views are at most 4-D")
    pad = (1,) * (4 - t.dim())
    # packed in one go (field by field, each array element is a Python call: twice the time)
    return _view_of(_VIEW.pack(t.data_ptr(), _DT.get(t.dtype, -1), t.is_cuda, *t.shape, *pad,
                               *t.stride(), *pad))


def _workspace(nbytes: int, device) -> torch.Tensor | None:
    if nbytes == 0:
        return None
    # the counters start at zero; the partials are written before they are read (zeroing all of it
    # took 10 us beside a 36 us f32 layer of 6 heads x 1500 frames)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=device)
    ws[:L.COUNTER_BYTES].zero_()
    return ws


# -------------------------------------------------------------------------------------------
# Mirrors of the reference functions
# -------------------------------------------------------------------------------------------

def serves(kt: torch.Tensor, v: torch.Tensor) -> bool:
    """flash_attn::serves: whether the decode-shape kernel serves this K/V pair (callers pick the
    cross-attention cache dtype with it)."""
    return L.load().ffai_serves(ctypes.byref(_view(kt)), ctypes.byref(_view(v))) == 1


def attend(q: torch.Tensor, kt: torch.Tensor, v: torch.Tensor,
           masked: bool = False) -> Optional[torch.Tensor]:
    """flash_attn::attend: q (1,H,qlen,64) f32; kt (1,H,64,K) and v (1,H,K,64) f32 (or f16 at
    qlen == 1). Returns (1,H,qlen,64) f32, or None where the reference declines."""
    lib = L.load()
    qv, kv, vv = _view(q), _view(kt), _view(v)
    nbytes = ctypes.c_size_t(0)
    rc = lib.ffai_attend_workspace_bytes(ctypes.byref(qv), ctypes.byref(kv), ctypes.byref(vv),
                                         ctypes.byref(nbytes))
    if masked or rc == L.FFAI_DECLINED:
        # let the C mirror apply (and report) the decline, exactly as it would for a caller
        out = torch.empty(0, device=q.device)
        rc = lib.ffai_attend(ctypes.byref(qv), ctypes.byref(kv), ctypes.byref(vv), int(masked),
                             ctypes.byref(_view(out)), None, 0, _stream_handle(q))
        return None if L.check(rc) == L.FFAI_DECLINED else out
    L.check(rc)
    out = torch.empty(q.shape[0], q.shape[1], q.shape[2], 64, dtype=torch.float32,
                      device=q.device)
    ws = _workspace(nbytes.value, q.device)
    rc = lib.ffai_attend(ctypes.byref(qv), ctypes.byref(kv), ctypes.byref(vv), 0,
                         ctypes.byref(_view(out)),
                         None if ws is None else ws.data_ptr(), nbytes.value, _stream_handle())
    if L.check(rc) == L.FFAI_DECLINED:
        return None
    return out


def attend_merged(q: torch.Tensor, kt: torch.Tensor,
                  v: torch.Tensor) -> Optional[torch.Tensor]:
    """flash_attn::attend_merged: encoder attention writing (1,T,H*64) f32 directly, or None."""
    lib = L.load()
    qv, kv, vv = _view(q), _view(kt), _view(v)
    heads, seq = q.shape[1], q.shape[2]
    out = torch.empty(1, seq, heads * 64, dtype=torch.float32, device=q.device)
    nbytes = ctypes.c_size_t(0)
    rc = lib.ffai_attend_merged_workspace_bytes(ctypes.byref(qv), ctypes.byref(kv),
                                                ctypes.byref(vv), ctypes.byref(nbytes))
    ws = _workspace(nbytes.value, q.device) if rc == L.FFAI_OK else None
    rc = lib.ffai_attend_merged(ctypes.byref(qv), ctypes.byref(kv), ctypes.byref(vv),
                                ctypes.byref(_view(out)),
                                None if ws is None else ws.data_ptr(), nbytes.value,
                                _stream_handle(q))
    if L.check(rc) == L.FFAI_DECLINED:
        return None
    return out


def decode_min_keys() -> int:
    return L.load().ffai_get_decode_min_keys()


def set_decode_min_keys(n: int) -> None:
    """knobs::DECODE_MIN_KEYS.set (knobs.rs:163-168)."""
    L.load().ffai_set_decode_min_keys(int(n))


# -------------------------------------------------------------------------------------------
# General descriptor entry point
# -------------------------------------------------------------------------------------------

def make_desc(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, out: torch.Tensor, *,
              k_transposed: bool, scale: float, causal: bool, q_offset: int,
              kv_lens: Optional[torch.Tensor]) -> L.AttnDesc:
    """Descriptor for q (B,Hq,Tq,D), k (B,Hkv,D,Tk) if k_transposed else (B,Hkv,Tk,D),
    v (B,Hkv,Tk,D), out (B,Hq,Tq,D); any strides with a unit innermost stride. A K/V batch
    dimension of size 1 broadcasts (stride 0) across the batch."""
    b, hq, tq, d = q.shape
    hkv = v.shape[1]
    tk = v.shape[2]
    desc = L.AttnDesc()
    desc.q_dtype = _DT[q.dtype]
    desc.kv_dtype = _DT[k.dtype]
    desc.out_dtype = _DT[out.dtype]
    desc.batch, desc.heads_q, desc.heads_kv = b, hq, hkv
    desc.q_len, desc.kv_len, desc.head_dim = tq, tk, d
    desc.k_layout = L.K_TRANSPOSED if k_transposed else L.K_ROWS
    desc.causal = int(causal)
    desc.q_offset = int(q_offset)
    desc.scale = float(scale)

    def strides(t: torch.Tensor):
        s = t.stride()
        return (0,) + s[1:] if t.shape[0] == 1 and b > 1 else s

    desc.q_strides, desc.k_strides = strides(q), strides(k)
    desc.v_strides, desc.o_strides = strides(v), strides(out)
    desc.kv_lens = None if kv_lens is None else kv_lens.data_ptr()
    return desc


def attention(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, *, k_transposed: bool = False,
              scale: float = 1.0, causal: bool = False, q_offset: int = 0,
              kv_lens: Optional[torch.Tensor] = None, out: Optional[torch.Tensor] = None,
              out_dtype: Optional[torch.dtype] = None,
              workspace: Optional[torch.Tensor] = None) -> Optional[torch.Tensor]:
    """O = softmax(scale * Q K^T [+ causal mask]) V through ffai_attn_fwd. Returns the output, or
    None when the descriptor is not served. `workspace` (see workspace_bytes) may be reused by
    stream-ordered calls and graph replays."""
    lib = L.load()
    if out is None:
        od = out_dtype or (torch.float32 if q.dtype == torch.float32 else q.dtype)
        out = torch.empty(q.shape[0], q.shape[1], q.shape[2], v.shape[3], dtype=od,
                          device=q.device)
    if kv_lens is not None:
        assert kv_lens.dtype == torch.int32 and kv_lens.is_cuda
    desc = make_desc(q, k, v, out, k_transposed=k_transposed, scale=scale, causal=causal,
                     q_offset=q_offset, kv_lens=kv_lens)
    nbytes = ctypes.c_size_t(0)
    rc = L.check(lib.ffai_attn_workspace_bytes(ctypes.byref(desc), ctypes.byref(nbytes)))
    if rc == L.FFAI_DECLINED:
        return None
    if nbytes.value and (workspace is None or workspace.numel() * workspace.element_size()
                         < nbytes.value):
        # row blocks use none (at head_dim 128 whether the call runs so depends on its alignment)
        if desc.head_dim != 64 or lib.ffai_attn_row_block(ctypes.byref(desc)) == 0:
            workspace = _workspace(nbytes.value, q.device)
    rc = lib.ffai_attn_fwd(ctypes.byref(desc), q.data_ptr(), k.data_ptr(), v.data_ptr(),
                           out.data_ptr(),
                           None if workspace is None else workspace.data_ptr(),
                           0 if workspace is None else workspace.numel() * workspace.element_size(),
                           _stream_handle())
    if L.check(rc) == L.FFAI_DECLINED:
        return None
    return out


def workspace_bytes(q, k, v, out, **kw) -> int:
    desc = make_desc(q, k, v, out, k_transposed=kw.get("k_transposed", False),
                     scale=kw.get("scale", 1.0), causal=kw.get("causal", False),
                     q_offset=kw.get("q_offset", 0), kv_lens=kw.get("kv_lens"))
    n = ctypes.c_size_t(0)
    L.check(L.load().ffai_attn_workspace_bytes(ctypes.byref(desc), ctypes.byref(n)))
    return n.value


def plan(q, k, v, out, **kw) -> dict:
    """The launch plan ffai_attn_fwd uses for these operands, or the row blocks ("row_block") that
    it runs as instead: see _lib.plan_info. K and V 16-byte aligned is assumed (at head_dim 64 it does
    not matter)."""
    desc = make_desc(q, k, v, out, k_transposed=kw.get("k_transposed", False),
                     scale=kw.get("scale", 1.0), causal=kw.get("causal", False),
                     q_offset=kw.get("q_offset", 0), kv_lens=kw.get("kv_lens"))
    return L.plan_info(desc)


def serves_desc(q_dtype: torch.dtype, kv_dtype: torch.dtype, out_dtype: torch.dtype,
                shape: Sequence[int], *, k_transposed: bool = False, causal: bool = False) -> bool:
    """ffai_attn_serves for packed operands: shape = (batch, heads_q, heads_kv, q_len, kv_len,
    head_dim)."""
    b, hq, hkv, tq, tk, d = shape
    desc = L.AttnDesc()
    L.load().ffai_attn_desc_init(ctypes.byref(desc), _DT[q_dtype], _DT[kv_dtype], _DT[out_dtype],
                                 b, hq, hkv, tq, tk, d,
                                 L.K_TRANSPOSED if k_transposed else L.K_ROWS)
    desc.causal = int(causal)
    return L.load().ffai_attn_serves(ctypes.byref(desc)) == 1
