"""Torch-facing entry points of the HIP attention library.

All tensors must live on the GPU; outputs and workspaces are allocated with
PyTorch's caching allocator and every launch goes on
`torch.cuda.current_stream()`. There is no CPU path: calling these with CPU
tensors raises.

Layouts (any strides, last dim contiguous):
  dense   q [B, Tq, Hq, D], k/v [B, Tk, Hkv, D]
  varlen  q [total_q, Hq, D], k/v [total_k, Hkv, D] with int32 cu_seqlens
The reference's kernel layout [B, H, T, D] is passed as `x.transpose(1, 2)`.
"""

from __future__ import annotations

import ctypes
import math
from typing import NamedTuple

import torch

from . import _lib

_DTYPES = {
    torch.float32: _lib.DTYPE_F32,
    torch.float16: _lib.DTYPE_F16,
    torch.bfloat16: _lib.DTYPE_BF16,
}


def _ptr(t: torch.Tensor | None) -> int | None:
    return None if t is None else t.data_ptr()


# The current stream's handle without the Stream object that
# torch.cuda.current_stream() builds (about 4 us of a call's host time).
_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream() -> int:
    if _raw_stream is None:
        return torch.cuda.current_stream().cuda_stream
    return _raw_stream(torch.cuda.current_device())


def _require_gpu(name: str, t: torch.Tensor) -> None:
    if not t.is_cuda:
        raise ValueError(f"goda_amd: {name} must be a GPU tensor (got {t.device})")


def _require_last_contig(name: str, t: torch.Tensor) -> None:
    if t.stride(-1) != 1:
        raise ValueError(f"goda_amd: {name} must be contiguous in its last dimension")


def _i32_vec(name: str, t: torch.Tensor | None, n: int, device: torch.device) -> torch.Tensor | None:
    if t is None:
        return None
    if t.dtype != torch.int32 or t.dim() != 1 or t.numel() != n:
        raise ValueError(f"goda_amd: {name} must be an int32 vector of length {n}")
    if t.device != device:
        raise ValueError(f"goda_amd: {name} must be on {device}")
    return t.contiguous()


def _f32_vec(name: str, t: torch.Tensor | None, n: int, device: torch.device) -> torch.Tensor | None:
    if t is None:
        return None
    if t.dtype == torch.float32 and t.dim() == 1 and t.shape[0] == n and t.is_contiguous() and t.device == device:
        return t  # (the usual weight, as it is)
    t = t.detach().reshape(-1)
    if t.numel() != n:
        raise ValueError(f"goda_amd: {name} must have {n} elements")
    return t.to(device=device, dtype=torch.float32).contiguous()


class PackedMask(NamedTuple):
    """A boolean attention mask bit-packed along the key axis for the C-ABI
    (goda_prefill_args.mask_bits): int32 words [Bm, Hm, Lqm, W] with
    W = 2 * ceil(seqlen_k / 64); bit j % 32 of word j // 32 is key j. Strides
    are in words, 0 where the mask broadcasts (Bm, Hm or Lqm of 1)."""

    bits: torch.Tensor
    stride_b: int
    stride_h: int
    stride_q: int
    seqlen_k: int


def pack_mask(
    mask: torch.Tensor, batch: int, heads_q: int, seqlen_q: int, seqlen_k: int, device, *, allow_short_keys: bool = False
) -> PackedMask:
    """Bit-pack goda's boolean `base_attn_mask` (mint/nn/flashattn.py:242-243),
    broadcastable to the attention-weight shape [B, Hq, Lq, Lk]: its key
    dimension is seqlen_k or 1 (broadcast over every key), as SDPA requires.
    `allow_short_keys` is for KV-cache launches, sized by a bound past the
    keys the mask names: a shorter key dimension then hides the rest."""
    if isinstance(mask, PackedMask):
        if mask.seqlen_k < seqlen_k:
            raise ValueError(f"goda_amd: packed mask covers {mask.seqlen_k} keys, the launch has {seqlen_k}")
        return mask
    if mask.dtype != torch.bool:
        raise ValueError(f"goda_amd: base_attn_mask must be boolean (got {mask.dtype})")
    m = mask
    while m.dim() < 4:
        m = m.unsqueeze(0)
    if m.dim() != 4:
        raise ValueError(f"goda_amd: base_attn_mask {tuple(mask.shape)} has more than 4 dimensions")
    for size, full, name in zip(m.shape[:3], (batch, heads_q, seqlen_q), ("batch", "heads", "query")):
        if size not in (1, full):
            raise ValueError(f"goda_amd: base_attn_mask {tuple(mask.shape)} does not broadcast over {name} size {full}")
    if m.shape[3] != 1 and m.shape[3] > seqlen_k:
        raise ValueError(f"goda_amd: base_attn_mask has {m.shape[3]} keys, more than the {seqlen_k} attended")
    if m.shape[3] not in (1, seqlen_k) and not allow_short_keys:
        raise ValueError(f"goda_amd: base_attn_mask has {m.shape[3]} keys; the attention has {seqlen_k}")
    m = m.to(device)
    # a dimension expanded to its size (stride 0) is one mask for all of it
    for dim in range(3):
        if m.shape[dim] > 1 and m.stride(dim) == 0:
            m = m.narrow(dim, 0, 1)
    bm, hm, qm, lk = m.shape
    if not m.is_cuda:
        bits = _pack_bits_cpu(m, seqlen_k)
        return PackedMask(bits, *(bits.stride(i) if m.shape[i] > 1 else 0 for i in range(3)), seqlen_k)
    bits = torch.empty(bm, hm, qm, 2 * ((seqlen_k + 63) // 64), dtype=torch.int32, device=m.device)
    a = _lib.PackMaskArgs()
    a.mask, a.bits = m.data_ptr(), bits.data_ptr()
    a.stride_b, a.stride_h, a.stride_q = m.stride(0), m.stride(1), m.stride(2)
    a.stride_k = 0 if lk == 1 else m.stride(3)  # one byte for every key
    a.batch, a.heads, a.rows, a.keys, a.mask_keys = bm, hm, qm, seqlen_k, seqlen_k if lk == 1 else lk
    _lib.check(_lib.load().goda_attn_pack_mask(ctypes.byref(a), _stream()))
    return PackedMask(bits, *(bits.stride(i) if m.shape[i] > 1 else 0 for i in range(3)), seqlen_k)


def _pack_bits_cpu(m: torch.Tensor, seqlen_k: int) -> torch.Tensor:
    bm, hm, qm, lk = m.shape
    words = 2 * ((seqlen_k + 63) // 64)
    u8 = torch.zeros(bm, hm, qm, words * 32, dtype=torch.uint8)
    u8[..., : seqlen_k if lk == 1 else lk] = m
    weights = torch.tensor([1, 2, 4, 8, 16, 32, 64, 128], dtype=torch.uint8)
    by = (u8.view(bm, hm, qm, words * 4, 8) * weights).sum(-1, dtype=torch.uint8)
    return by.contiguous().view(torch.int32)  # little-endian: byte k holds keys 8k .. 8k+7


def _rope_tables(cos: torch.Tensor | None, sin: torch.Tensor | None, head_dim: int, device):
    if cos is None and sin is None:
        return None, None, 0
    if cos is None or sin is None:
        raise ValueError("goda_amd: rope_cos and rope_sin go together")
    if (
        cos.dtype == sin.dtype == torch.float32
        and cos.dim() == 2
        and cos.shape == sin.shape
        and cos.shape[1] == head_dim // 2
        and cos.is_contiguous()
        and sin.is_contiguous()
        and cos.device == device
        and sin.device == device
    ):
        return cos, sin, cos.shape[0]  # (the usual tables, as they are)
    cos = cos.reshape(-1, head_dim // 2).to(device=device, dtype=torch.float32).contiguous()
    sin = sin.reshape(-1, head_dim // 2).to(device=device, dtype=torch.float32).contiguous()
    if cos.shape != sin.shape:
        raise ValueError("goda_amd: rope_cos and rope_sin shapes differ")
    return cos, sin, cos.shape[0]


class Launch:
    """A validated, ready-to-run C-ABI call: the argument struct, the tensors
    it points to (kept alive here), and the outputs. Calling it enqueues the
    kernels on the current stream again; nothing is allocated or checked on
    the Python side, so a serving loop can reuse one plan per shape.

    `timing` optionally takes two hipEvent_t handles (e.g. the `cuda_event`
    of two recorded torch.cuda.Event(enable_timing=True)) that the library
    records right around its main kernel."""

    def __init__(self, fn_name: str, args, keep: tuple, result, grads=None):
        self._fn = getattr(_lib.load(), fn_name)
        self.args = args
        self.grads = grads  # the backward's second struct (it carries the timing events)
        self._keep = keep
        self.result = result

    def __call__(self, timing: tuple[int, int] | None = None):
        a = self.args
        t = self.grads if self.grads is not None else a
        if timing is not None:
            t.timing_begin, t.timing_end = timing
        try:
            if self.grads is not None:
                _lib.check(self._fn(ctypes.byref(a), ctypes.byref(self.grads), _stream()))
            else:
                _lib.check(self._fn(ctypes.byref(a), _stream()))
        finally:
            if timing is not None:
                t.timing_begin = t.timing_end = None
        return self.result


def attention_prefill(*args, **kwargs):
    """Prefill attention through `goda_attn_prefill_fwd`; see `plan_prefill`
    for the arguments. Returns `o` (and the fp32 `lse` if `return_lse`)."""
    return plan_prefill(*args, **kwargs)()


def plan_prefill(q: torch.Tensor, k: torch.Tensor, v: torch.Tensor, **kwargs):
    """Validate the arguments of `goda_attn_prefill_fwd`, allocate outputs
    and workspace, and return the `Launch` that runs it.

    Semantics are those of goda's eager path (mint/nn/flashattn.py:221-273):
    GQA head mapping h -> h // (Hq/Hkv), bottom-right causal alignment, left
    window only with causal (or a single query), ALiBi as
    slope_h * (j - i_abs), RoPE as mint/nn/pos.py:90-112 using the given
    fp32 cos/sin tables. Returns `o` (and `lse` fp32 if `return_lse`).
    Keyword arguments: see `_prefill_args`.
    """
    a, keep, o, lse = _prefill_args(q, k, v, **kwargs)
    lib = _lib.load()
    need = lib.goda_attn_prefill_workspace_size(ctypes.byref(a))
    if need < 0:
        _lib.check(int(need))
    ws = None
    if need > 0:
        ws = torch.empty(int(need), dtype=torch.uint8, device=q.device)
        a.workspace, a.workspace_bytes = ws.data_ptr(), int(need)
    # The plan keeps every tensor the struct points to alive. Once a plan is
    # dropped, the caching allocator only reuses that memory for work
    # ordered after the launch on this stream.
    return Launch("goda_attn_prefill_fwd", a, keep + (ws,), (o, lse) if lse is not None else o)


def _prefill_args(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    *,
    causal: bool,
    softmax_scale: float | None = None,
    window_left: int = -1,
    alibi_slopes: torch.Tensor | None = None,
    rope_cos: torch.Tensor | None = None,
    rope_sin: torch.Tensor | None = None,
    rope_q: bool = False,
    rope_k: bool = False,
    rope_q_offset: int = 0,
    rope_k_offset: int = 0,
    rope_pos_abs: bool = False,
    rope_packed_rows: bool = False,
    q_norm_weight: torch.Tensor | None = None,
    k_norm_weight: torch.Tensor | None = None,
    norm_eps: float = 1e-6,
    attn_mask: torch.Tensor | PackedMask | None = None,
    cu_seqlens_q: torch.Tensor | None = None,
    cu_seqlens_k: torch.Tensor | None = None,
    max_seqlen_q: int | None = None,
    max_seqlen_k: int | None = None,
    seqused_k: torch.Tensor | None = None,
    return_lse: bool = False,
    out: torch.Tensor | None = None,
    lse_in: torch.Tensor | None = None,
):
    """Validated `PrefillArgs` for q, k, v and the options, with `o` (`out`
    or a new tensor) and `lse` (`lse_in`, a new tensor if `return_lse`, or
    None). Returns (args, tensors to keep alive, o, lse); no workspace.
    `attn_mask` is a boolean mask broadcastable to [B, Hq, Lq, Lk] (or a
    `PackedMask`), composed with causal / window like goda's base_attn_mask;
    `rope_pos_abs` rotates query row i at rope_q_offset + i instead of
    rope_q_offset + (Lk - Lq) + i; `rope_packed_rows` (varlen) rotates packed
    query and key rows at their index modulo the length of the tables."""
    for name, t in (("q", q), ("k", k), ("v", v)):
        _require_gpu(name, t)
        _require_last_contig(name, t)
    if not (q.dtype == k.dtype == v.dtype):
        raise ValueError(f"goda_amd: q/k/v dtypes differ ({q.dtype}, {k.dtype}, {v.dtype})")
    if q.dtype not in _DTYPES:
        raise ValueError(f"goda_amd: unsupported dtype {q.dtype}")
    varlen = cu_seqlens_q is not None
    if (cu_seqlens_k is not None) != varlen:
        raise ValueError("goda_amd: cu_seqlens_q and cu_seqlens_k go together")
    dev = q.device
    if varlen:
        if q.dim() != 3 or k.dim() != 3 or v.dim() != 3:
            raise ValueError("goda_amd: varlen q/k/v must be [total, H, D]")
        batch = cu_seqlens_q.numel() - 1
        cu_q = _i32_vec("cu_seqlens_q", cu_seqlens_q, batch + 1, dev)
        cu_k = _i32_vec("cu_seqlens_k", cu_seqlens_k, batch + 1, dev)
        if max_seqlen_q is None or max_seqlen_k is None:
            raise ValueError("goda_amd: varlen needs max_seqlen_q and max_seqlen_k")
        tq, tk = int(max_seqlen_q), int(max_seqlen_k)
        hq, d = q.shape[1], q.shape[2]
        hkv = k.shape[1]
        qs = (0, q.stride(0), q.stride(1))
        ks = (0, k.stride(0), k.stride(1))
        vs = (0, v.stride(0), v.stride(1))
        if v.shape[1] != hkv or k.shape[2] != d or v.shape[2] != d or k.shape[0] != v.shape[0]:
            raise ValueError("goda_amd: k/v shapes do not match q")
    else:
        if q.dim() != 4 or k.dim() != 4 or v.dim() != 4:
            raise ValueError("goda_amd: dense q/k/v must be [B, T, H, D]")
        batch, tq, hq, d = q.shape
        _, tk, hkv, _ = k.shape
        if k.shape[0] != batch or v.shape != k.shape or k.shape[3] != d:
            raise ValueError(f"goda_amd: k {tuple(k.shape)} / v {tuple(v.shape)} do not match q {tuple(q.shape)}")
        cu_q = cu_k = None
        qs, ks, vs = q.stride()[:3], k.stride()[:3], v.stride()[:3]
    if hq % hkv != 0:
        raise ValueError(f"goda_amd: heads_q {hq} is not a multiple of heads_kv {hkv}")
    used = _i32_vec("seqused_k", seqused_k, batch, dev)

    if out is None:
        o = torch.empty(q.shape, dtype=q.dtype, device=dev)
    else:
        if out.shape != q.shape or out.dtype != q.dtype or out.device != dev:
            raise ValueError("goda_amd: out must match q's shape, dtype and device")
        _require_last_contig("out", out)
        o = out
    os_ = (0, o.stride(0), o.stride(1)) if varlen else (o.stride(0), o.stride(1), o.stride(2))

    lse = None
    lse_shape = (hq, q.shape[0]) if varlen else (batch, hq, tq)
    if lse_in is not None:
        if tuple(lse_in.shape) != lse_shape or lse_in.dtype != torch.float32 or lse_in.device != dev:
            raise ValueError(f"goda_amd: lse must be fp32 {lse_shape} on {dev}")
        if lse_in.stride(-1) != 1:
            raise ValueError("goda_amd: lse rows must be contiguous")
        lse = lse_in
    elif return_lse:
        lse = torch.empty(lse_shape, dtype=torch.float32, device=dev)

    slopes = _f32_vec("alibi_slopes", alibi_slopes, hq, dev)
    cos, sin, rope_len = _rope_tables(rope_cos, rope_sin, d, dev)
    if (rope_q or rope_k) and cos is None:
        raise ValueError("goda_amd: rope_q/rope_k need rope_cos and rope_sin")

    a = _lib.PrefillArgs()
    a.dtype = _DTYPES[q.dtype]
    a.batch, a.heads_q, a.heads_kv, a.head_dim = batch, hq, hkv, d
    a.seqlen_q, a.seqlen_k = tq, tk
    a.causal = int(bool(causal))
    a.window_left = int(window_left)
    a.softmax_scale = float(softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d))
    a.q, a.k, a.v, a.o = q.data_ptr(), k.data_ptr(), v.data_ptr(), o.data_ptr()
    a.q_stride_b, a.q_stride_t, a.q_stride_h = qs
    a.k_stride_b, a.k_stride_t, a.k_stride_h = ks
    a.v_stride_b, a.v_stride_t, a.v_stride_h = vs
    a.o_stride_b, a.o_stride_t, a.o_stride_h = os_
    if lse is not None:
        a.lse = lse.data_ptr()
        if varlen:
            a.lse_stride_b, a.lse_stride_h = 0, lse.stride(0)
        else:
            a.lse_stride_b, a.lse_stride_h = lse.stride(0), lse.stride(1)
    a.cu_seqlens_q, a.cu_seqlens_k = _ptr(cu_q), _ptr(cu_k)
    a.seqused_k = _ptr(used)
    a.alibi_slopes = _ptr(slopes)
    a.rope_cos, a.rope_sin, a.rope_len = _ptr(cos), _ptr(sin), rope_len
    a.rope_q, a.rope_k = int(bool(rope_q)), int(bool(rope_k))
    a.rope_q_offset, a.rope_k_offset = int(rope_q_offset), int(rope_k_offset)
    a.rope_pos_abs, a.rope_packed_rows = int(bool(rope_pos_abs)), int(bool(rope_packed_rows))
    qn = _f32_vec("q_norm_weight", q_norm_weight, d, dev)
    kn = _f32_vec("k_norm_weight", k_norm_weight, d, dev)
    a.q_norm_weight, a.k_norm_weight, a.norm_eps = _ptr(qn), _ptr(kn), float(norm_eps)
    pm = None
    if attn_mask is not None:
        if varlen:
            raise ValueError("goda_amd: attn_mask needs dense q/k/v (not cu_seqlens)")
        pm = pack_mask(attn_mask, batch, hq, tq, tk, dev)
        a.mask_bits = pm.bits.data_ptr()
        a.mask_stride_b, a.mask_stride_h, a.mask_stride_q = pm.stride_b, pm.stride_h, pm.stride_q

    keep = (q, k, v, o, lse, slopes, cos, sin, cu_q, cu_k, used, qn, kn, pm)
    return a, keep, o, lse


def doc_segments(doc_ids: torch.Tensor) -> tuple[torch.Tensor, int, bool] | None:
    """cu_seqlens (int32, on the GPU) of the maximal runs of equal ids inside
    each row of doc_ids [B, T], the longest run, and whether every id occupies
    one run of its row, through `goda_attn_doc_segments`: two launches and one
    read of three words. None where the kernel leaves the last question open
    (over 1024 runs of ids in no order) or does not take the ids."""
    _require_gpu("doc_ids", doc_ids)
    if doc_ids.dim() != 2 or doc_ids.dtype not in (torch.int32, torch.int64) or not 0 < doc_ids.numel() < 1 << 31:
        return None
    if doc_ids.stride(1) != 1:
        doc_ids = doc_ids.contiguous()
    b, t = doc_ids.shape
    lib = _lib.load()
    need = int(lib.goda_attn_doc_segments_scratch_bytes(b, t))
    scratch = torch.empty(need, dtype=torch.uint8, device=doc_ids.device)
    out = torch.empty(3 + b * t + 1, dtype=torch.int32, device=doc_ids.device)
    result, cu = out[:3], out[3:]
    _lib.check(lib.goda_attn_doc_segments(doc_ids.data_ptr(), doc_ids.element_size(), doc_ids.stride(0), b, t, cu.data_ptr(),
                                          result.data_ptr(), scratch.data_ptr(), need, _stream()))
    count, longest, recurring = result.tolist()  # launch sizes (the reference synchronizes here too)
    if recurring == 2:
        return None
    return cu[: count + 1], longest, recurring == 0


def attention_prefill_bwd(q, k, v, o, lse, d_o, **kwargs):
    """Gradients (dq, dk, dv) of `attention_prefill` through
    `goda_attn_prefill_bwd`, from the forward's o and lse and the upstream
    gradient d_o. Takes the forward's own keyword arguments (causal, window,
    ALiBi, RoPE, fused QK-RMSNorm, varlen, seqused_k, scale), so the scores
    are recomputed exactly as the forward computed them. dk/dv have Hkv heads
    (summed over each KV head's query group) and are zero for keys past
    seqused_k. With `q_norm_weight` / `k_norm_weight` the result is
    (dq, dk, dv, d_q_norm_weight, d_k_norm_weight): dq / dk are the gradients
    of the rows before the norm, the weight gradients fp32 [head_dim] (None
    for a norm not given)."""
    return plan_prefill_bwd(q, k, v, o, lse, d_o, **kwargs)()


def plan_prefill_bwd(
    q: torch.Tensor,
    k: torch.Tensor,
    v: torch.Tensor,
    o: torch.Tensor,
    lse: torch.Tensor,
    d_o: torch.Tensor,
    **kwargs,
):
    """Validate and allocate once for `goda_attn_prefill_bwd`; returns the
    `Launch` whose result is (dq, dk, dv)."""
    kwargs.pop("return_lse", None)
    kwargs.pop("out", None)
    a, keep, o, lse = _prefill_args(q, k, v, out=o, lse_in=lse, **kwargs)
    _require_gpu("d_o", d_o)
    if d_o.shape != o.shape or d_o.dtype != o.dtype:
        raise ValueError(f"goda_amd: d_o {tuple(d_o.shape)} {d_o.dtype} must match o {tuple(o.shape)} {o.dtype}")
    if d_o.stride(-1) != 1:
        d_o = d_o.contiguous()
    dq = torch.empty_like(q)
    dk = torch.empty_like(k)
    dv = torch.empty_like(v)
    for name, t in (("dq", dq), ("dk", dk), ("dv", dv)):
        _require_last_contig(name, t)
    g = _lib.PrefillGrads()
    varlen = q.dim() == 3

    def strides(t):
        return (0, t.stride(0), t.stride(1)) if varlen else (t.stride(0), t.stride(1), t.stride(2))

    g.d_o = d_o.data_ptr()
    g.do_stride_b, g.do_stride_t, g.do_stride_h = strides(d_o)
    g.dq = dq.data_ptr()
    g.dq_stride_b, g.dq_stride_t, g.dq_stride_h = strides(dq)
    g.dk = dk.data_ptr()
    g.dk_stride_b, g.dk_stride_t, g.dk_stride_h = strides(dk)
    g.dv = dv.data_ptr()
    g.dv_stride_b, g.dv_stride_t, g.dv_stride_h = strides(dv)
    result = (dq, dk, dv)
    norm = (kwargs.get("q_norm_weight"), kwargs.get("k_norm_weight"))
    dw = [None, None]
    if norm[0] is not None or norm[1] is not None:
        for i, w in enumerate(norm):
            if w is not None:
                dw[i] = torch.empty(q.shape[-1], dtype=torch.float32, device=q.device)
        g.dq_norm_weight, g.dk_norm_weight = _ptr(dw[0]), _ptr(dw[1])
        result = (dq, dk, dv, dw[0], dw[1])
    lib = _lib.load()
    need = lib.goda_attn_prefill_bwd_workspace_size(ctypes.byref(a))
    if need < 0:
        _lib.check(int(need))
    ws = None
    if need > 0:
        ws = torch.empty(int(need), dtype=torch.uint8, device=q.device)
        g.workspace, g.workspace_bytes = ws.data_ptr(), int(need)
    return Launch("goda_attn_prefill_bwd", a, keep + (d_o, dq, dk, dv, ws, *dw), result, grads=g)


def attention_decode(*args, **kwargs):
    """One-token decode through `goda_attn_decode`; see `plan_decode`.
    Returns `o` (and the fp32 `lse` [B, Hq] if `return_lse`)."""
    return plan_decode(*args, **kwargs)()


def plan_decode(
    q: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    cache_seqlens: torch.Tensor,
    *,
    softmax_scale: float | None = None,
    window_left: int = -1,
    alibi_slopes: torch.Tensor | None = None,
    rope_cos: torch.Tensor | None = None,
    rope_sin: torch.Tensor | None = None,
    rope_q: bool = False,
    rope_q_offset: int = 0,
    rope_pos_abs: bool = False,
    q_norm_weight: torch.Tensor | None = None,
    norm_eps: float = 1e-6,
    split_size: int = 0,
    cache_layout: str = "bthd",
    return_lse: bool = False,
    out: torch.Tensor | None = None,
    noalloc: bool = False,
):
    """Validate and prepare a one-token decode over a KV cache with
    per-sequence lengths; returns the `Launch`.

    q: [B, Hq, D] (or [B, 1, Hq, D]); caches [B, Lmax, Hkv, D] when
    cache_layout == "bthd" (goda's KVCache, mint/kvcache/base.py:22-31) or
    [B, Hkv, Lmax, D] when "bhtd"; cache_seqlens int32 [B] = valid keys
    (the new token included). The query sits at position cache_seqlens[b]-1
    and is rotated there (+ rope_q_offset), or at rope_q_offset itself with
    `rope_pos_abs` (a caller-given position, goda's start_pos).
    With `noalloc` the launch goes through `goda_attn_decode_noalloc`, whose
    split-K partials live in the library's fixed device-resident array (no
    workspace; calls overlapping on one GPU race).
    """
    squeeze = False
    if q.dim() == 4:
        if q.shape[1] != 1:
            raise ValueError("goda_amd: decode takes one query token per sequence")
        q = q[:, 0]
        squeeze = True
    for name, t in (("q", q), ("k_cache", k_cache), ("v_cache", v_cache)):
        _require_gpu(name, t)
        _require_last_contig(name, t)
    if not (q.dtype == k_cache.dtype == v_cache.dtype) or q.dtype not in _DTYPES:
        raise ValueError("goda_amd: q and caches must share a supported dtype")
    if k_cache.shape != v_cache.shape:
        raise ValueError("goda_amd: k_cache and v_cache shapes differ")
    b, hq, d = q.shape
    if cache_layout == "bthd":
        _, lmax, hkv, dk = k_cache.shape
        ks = k_cache.stride()[:3]
        vs = v_cache.stride()[:3]
    elif cache_layout == "bhtd":
        _, hkv, lmax, dk = k_cache.shape
        ks = (k_cache.stride(0), k_cache.stride(2), k_cache.stride(1))
        vs = (v_cache.stride(0), v_cache.stride(2), v_cache.stride(1))
    else:
        raise ValueError(f"goda_amd: unknown cache_layout {cache_layout!r}")
    if k_cache.shape[0] < b or dk != d:
        raise ValueError("goda_amd: cache shape does not match q")
    if hq % hkv != 0:
        raise ValueError(f"goda_amd: heads_q {hq} is not a multiple of heads_kv {hkv}")
    dev = q.device
    seqlens = _i32_vec("cache_seqlens", cache_seqlens[:b] if cache_seqlens.numel() > b else cache_seqlens, b, dev)
    if out is None:
        o = torch.empty_like(q)
    else:
        if out.shape != q.shape or out.dtype != q.dtype or out.device != dev:
            raise ValueError(f"goda_amd: out must be {tuple(q.shape)} {q.dtype} on {dev}")
        _require_last_contig("out", out)
        o = out
    lse = torch.empty((b, hq), dtype=torch.float32, device=dev) if return_lse else None
    slopes = _f32_vec("alibi_slopes", alibi_slopes, hq, dev)
    cos, sin, rope_len = _rope_tables(rope_cos, rope_sin, d, dev)
    if rope_q and cos is None:
        raise ValueError("goda_amd: rope_q needs rope_cos and rope_sin")

    a = _lib.DecodeArgs()
    a.dtype = _DTYPES[q.dtype]
    a.batch, a.heads_q, a.heads_kv, a.head_dim = b, hq, hkv, d
    a.max_seqlen = lmax
    a.window_left = int(window_left)
    a.split_size = int(split_size)
    a.softmax_scale = float(softmax_scale if softmax_scale is not None else 1.0 / math.sqrt(d))
    a.q, a.q_stride_b, a.q_stride_h = q.data_ptr(), q.stride(0), q.stride(1)
    a.k_cache = k_cache.data_ptr()
    a.k_stride_b, a.k_stride_t, a.k_stride_h = ks
    a.v_cache = v_cache.data_ptr()
    a.v_stride_b, a.v_stride_t, a.v_stride_h = vs
    a.cache_seqlens = seqlens.data_ptr()
    a.o, a.o_stride_b, a.o_stride_h = o.data_ptr(), o.stride(0), o.stride(1)
    if lse is not None:
        a.lse, a.lse_stride_b = lse.data_ptr(), lse.stride(0)
    a.alibi_slopes = _ptr(slopes)
    a.rope_cos, a.rope_sin, a.rope_len = _ptr(cos), _ptr(sin), rope_len
    a.rope_q, a.rope_q_offset = int(bool(rope_q)), int(rope_q_offset)
    a.rope_pos_abs = int(bool(rope_pos_abs))
    qn = _f32_vec("q_norm_weight", q_norm_weight, d, dev)
    a.q_norm_weight, a.norm_eps = _ptr(qn), float(norm_eps)

    lib = _lib.load()
    need = lib.goda_attn_decode_workspace_size(ctypes.byref(a))
    if need < 0:
        _lib.check(int(need))
    ws = None
    if need > 0 and not noalloc:
        ws = torch.empty(int(need), dtype=torch.uint8, device=dev)
        a.workspace, a.workspace_bytes = ws.data_ptr(), int(need)
    ov = o.unsqueeze(1) if squeeze else o
    keep = (q, k_cache, v_cache, seqlens, o, lse, ws, slopes, cos, sin, qn)
    fn = "goda_attn_decode_noalloc" if noalloc else "goda_attn_decode"
    return Launch(fn, a, keep, (ov, lse) if return_lse else ov)


def kv_append(
    k_new: torch.Tensor,
    v_new: torch.Tensor,
    k_cache: torch.Tensor,
    v_cache: torch.Tensor,
    cache_seqlens: torch.Tensor,
    *,
    rope_cos: torch.Tensor | None = None,
    rope_sin: torch.Tensor | None = None,
    rope_k: bool = False,
    rope_k_offset: int = 0,
    rope_pos_abs: bool = False,
    k_norm_weight: torch.Tensor | None = None,
    norm_eps: float = 1e-6,
    status: torch.Tensor | None = None,
) -> None:
    """Write k_new/v_new [B, Tn, Hkv, D] into caches [Bmax, Lmax, Hkv, D] at
    each sequence's own position cache_seqlens[b], then advance the lengths —
    all on the device, with no host read of the lengths. k rows are
    optionally RMS-normalised (goda's RMSNorm with weight 1 + k_norm_weight)
    and then rotated before they are stored: row t at its cache position
    (+ rope_k_offset), or at rope_k_offset + t with `rope_pos_abs`.
    A sequence whose rows would pass Lmax keeps the rows that fit, its length
    stops at Lmax, and 1 is stored into `status` (an int32 GPU tensor the
    caller clears and checks) when given."""
    for name, t in (("k_new", k_new), ("v_new", v_new), ("k_cache", k_cache), ("v_cache", v_cache)):
        _require_gpu(name, t)
        _require_last_contig(name, t)
    if not (k_new.dtype == v_new.dtype == k_cache.dtype == v_cache.dtype) or k_new.dtype not in _DTYPES:
        raise ValueError("goda_amd: kv_append tensors must share a supported dtype")
    b, tn, hkv, d = k_new.shape
    if v_new.shape != k_new.shape or k_cache.shape[2:] != (hkv, d) or k_cache.shape != v_cache.shape:
        raise ValueError("goda_amd: kv_append shapes do not match")
    if k_cache.shape[0] < b:
        raise ValueError(f"goda_amd: kv_append of {b} sequences into a cache of {k_cache.shape[0]}")
    if status is not None and (status.dtype != torch.int32 or status.numel() < 1 or status.device != k_new.device):
        raise ValueError("goda_amd: status must be an int32 tensor on the cache's device")
    if cache_seqlens.dtype != torch.int32 or cache_seqlens.numel() < b or not cache_seqlens.is_contiguous():
        raise ValueError("goda_amd: cache_seqlens must be a contiguous int32 vector")
    dev = k_new.device
    cos, sin, rope_len = _rope_tables(rope_cos, rope_sin, d, dev)
    if rope_k and cos is None:
        raise ValueError("goda_amd: rope_k needs rope_cos and rope_sin")
    a = _lib.KvAppendArgs()
    a.dtype = _DTYPES[k_new.dtype]
    a.batch, a.heads_kv, a.head_dim = b, hkv, d
    a.max_seqlen, a.seqlen_new = k_cache.shape[1], tn
    a.k_new, a.v_new = k_new.data_ptr(), v_new.data_ptr()
    a.kn_stride_b, a.kn_stride_t, a.kn_stride_h, _ = k_new.stride()
    a.vn_stride_b, a.vn_stride_t, a.vn_stride_h, _ = v_new.stride()
    a.k_cache, a.v_cache = k_cache.data_ptr(), v_cache.data_ptr()
    a.k_stride_b, a.k_stride_t, a.k_stride_h, _ = k_cache.stride()
    a.v_stride_b, a.v_stride_t, a.v_stride_h, _ = v_cache.stride()
    a.cache_seqlens = cache_seqlens.data_ptr()
    a.rope_cos, a.rope_sin, a.rope_len = _ptr(cos), _ptr(sin), rope_len
    a.rope_k, a.rope_k_offset = int(bool(rope_k)), int(rope_k_offset)
    a.rope_pos_abs = int(bool(rope_pos_abs))
    a.status = _ptr(status)
    kn = _f32_vec("k_norm_weight", k_norm_weight, d, dev)
    a.k_norm_weight, a.norm_eps = _ptr(kn), float(norm_eps)
    _lib.check(_lib.load().goda_attn_kv_append(ctypes.byref(a), _stream()))
    del kn  # ordered after the launch by the caching allocator

