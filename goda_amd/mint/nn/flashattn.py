"""Drop-in for goda's attention dispatcher (mint/nn/flashattn.py:14-273),
backed entirely by the HIP kernels.

`FlashAttention.forward(q, k, v, *, causal, window_size, kv_cache,
base_attn_mask, doc_ids)` keeps the reference signature and its results
(mint/nn/flashattn.py:21-53), with the reference's restrictions lifted:

  - real GQA/MQA (Hq != Hkv) runs on the fused kernel instead of falling back
    to SDPA (the reference's custom path needs Hq == Hkv, :139);
  - left sliding windows run on the kernel (the reference sends them to SDPA);
  - `doc_ids` packing runs as a varlen launch over the document segments of
    each row (the reference's varlen branch needs flash_attn, :98-137) when
    every id occupies one run of its row, which is how goda's loader writes
    them; ids that recur in separate runs take the dense document mask;
  - the KV-cache path appends on the device at each sequence's own length
    (no `.item()` sync, :202) and decodes with the split-K kernel. With
    doc_ids it follows the reference's SDPA path instead (:202-218): every
    sequence appends at sequence 0's length, and the document mask over the
    new tokens needs an empty cache unless there is one new token.

Without a KV cache the attention is differentiable: under autograd the
backward runs on the HIP backward kernels (goda's training path,
pretrain.py / sfttrain.py). The KV-cache path is inference only.

`base_attn_mask` (a boolean mask broadcastable to [B, Hq, Lq, Lk], composed
with the causal, window and doc masks as mint/nn/flashattn.py:236-255 does) is
bit-packed and applied inside the forward and backward kernels. A float mask
is SDPA's additive one: as in the reference it is taken only without causal
and doc_ids, and here only with values 0 and -inf. A right
window is ignored, as the reference's SDPA path ignores it
(mint/nn/flashattn.py:251-253).

Extra keyword arguments fuse the positional encoding into the kernels:
`rope=(cos, sin)` fp32 tables with `start_pos` (q and k are then passed
UNROTATED), or `alibi_slopes` [Hq]; `qk_norm=(q_scale, k_scale, eps)` fuses
goda's QK-RMSNorm (mint/nn/norm.py:17-27, weight 1 + scale, before RoPE) into
the kernels' q/k loads, forward and backward (the backward also returns the
two scales' gradients); over a KV cache with doc_ids, or in a differentiable
call, it runs as ordinary torch ops instead. There is no SDPA or CPU
fallback.
"""

from __future__ import annotations

import torch
from torch import nn

import math

from ... import autograd, headdim, ops
from ..kvcache.base import KVCache


def _segments(doc_ids: torch.Tensor) -> tuple[torch.Tensor, int, bool]:
    """cu_seqlens of the maximal runs of equal ids inside each row of
    doc_ids [B, T] (a run never crosses a row), the longest run, and whether
    every id occupies one run per row. Only then do the runs equal goda's
    mask doc_ids[i] == doc_ids[j] over the whole row
    (mint/nn/flashattn.py:238-240); goda's packing loader writes ids that way
    (mint/data/dist/pretrain.py:243-273). On the GPU by `ops.doc_segments`; the
    torch form below serves CPU tensors and what that one leaves open."""
    if doc_ids.is_cuda:
        found = ops.doc_segments(doc_ids)
        if found is not None:
            return found
    b, t = doc_ids.shape
    starts = torch.ones(b, t, dtype=torch.bool, device=doc_ids.device)
    starts[:, 1:] = doc_ids[:, 1:] != doc_ids[:, :-1]
    first = starts.reshape(-1).nonzero().reshape(-1).to(torch.int32)
    cu = torch.cat([first, torch.tensor([b * t], dtype=torch.int32, device=doc_ids.device)])
    srt = doc_ids.sort(dim=1).values
    distinct = 1 + (srt[:, 1:] != srt[:, :-1]).sum(1)
    recurring = (distinct != starts.sum(1)).any()
    # launch size and the recurrence flag (the reference syncs here too, :121)
    max_len, rec = torch.stack([(cu[1:] - cu[:-1]).max(), recurring.to(cu.dtype)]).tolist()
    return cu, int(max_len), not rec


def _bool_base_mask(mask: torch.Tensor | None, *, causal: bool, doc_ids) -> torch.Tensor | None:
    """goda's base_attn_mask as the boolean mask the kernels take. A float
    mask is additive (SDPA's convention); the reference accepts one only
    where it reaches SDPA untouched, i.e. without causal and doc_ids: with
    either it is combined with a boolean mask by `&`, which raises
    (mint/nn/flashattn.py:236-255), and so does this. The kernels apply
    visibility bits, so an additive mask must hold only 0 (visible) and -inf
    (hidden); other values are refused."""
    if mask is None or mask.dtype == torch.bool:
        return mask
    if not mask.is_floating_point():
        raise ValueError(f"goda_amd FlashAttention: base_attn_mask must be boolean or float (got {mask.dtype})")
    if causal or doc_ids is not None:
        raise TypeError(
            "goda_amd FlashAttention: a float base_attn_mask combines with the causal or document mask by '&', "
            "which needs a boolean mask (mint/nn/flashattn.py:242-253)"
        )
    if bool(((mask != 0) & ~torch.isneginf(mask)).any()):
        raise ValueError("goda_amd FlashAttention: a float base_attn_mask may hold only 0 and -inf")
    return mask == 0


class FlashAttention(nn.Module):
    def __init__(self, *, use_custom_fa: bool = True) -> None:
        super().__init__()
        self.use_custom_fa = use_custom_fa  # accepted for signature compatibility

    def forward(
        self,
        q: torch.Tensor,
        k: torch.Tensor,
        v: torch.Tensor,
        *,
        causal: bool = False,
        window_size: tuple[int, int] = (-1, -1),
        kv_cache: KVCache | None = None,
        base_attn_mask: torch.Tensor = None,
        doc_ids: torch.Tensor = None,
        rope: tuple[torch.Tensor, torch.Tensor] | None = None,
        start_pos: int | None = None,
        alibi_slopes: torch.Tensor | None = None,
        qk_norm: tuple[torch.Tensor, torch.Tensor, float] | None = None,
    ) -> torch.Tensor:
        # Only the left window is used: the reference's SDPA path reads
        # window_size[0] alone (mint/nn/flashattn.py:251-253, 258-264).
        window_left = window_size[0] if window_size[0] >= 0 else -1
        if qk_norm is not None and kv_cache is not None and (doc_ids is not None or _needs_grad(q, k, *qk_norm[:2])):
            # documents or a differentiable call over a KV cache: plain torch.
            q, k = headdim.rms_norm(q, qk_norm[0], qk_norm[2]), headdim.rms_norm(k, qk_norm[1], qk_norm[2])
            qk_norm = None
        base_attn_mask = _bool_base_mask(base_attn_mask, causal=causal, doc_ids=doc_ids)
        if kv_cache is None:
            return self._attention(q, k, v, causal=causal, window_left=window_left, doc_ids=doc_ids,
                                   base_attn_mask=base_attn_mask, rope=rope, start_pos=start_pos or 0,
                                   alibi_slopes=alibi_slopes, qk_norm=qk_norm)
        if doc_ids is not None:
            base_attn_mask = self._cache_doc_mask(q, kv_cache, doc_ids, base_attn_mask)
        return self._attention_with_kvcache(q, k, v, kv_cache, causal=causal, window_left=window_left,
                                            base_attn_mask=base_attn_mask, rope=rope, start_pos=start_pos,
                                            alibi_slopes=alibi_slopes, qk_norm=qk_norm)

    @staticmethod
    def _cache_doc_mask(q, kv_cache: KVCache, doc_ids, base_attn_mask):
        """doc_ids on the KV-cache path, as mint/nn/flashattn.py:202-218 treats
        them: every sequence appends at sequence 0's length, and the document
        mask compares the new tokens' ids with each other ([B, 1, T, T]), so
        it is all true for one token and otherwise needs the keys to be the
        new tokens alone, i.e. an empty cache (the reference's broadcast of
        that mask against T + cached keys fails otherwise). Returns the mask
        to combine with the causal/window ones."""
        b, tq = q.shape[0], q.shape[1]
        seqlens = kv_cache.cache_seqlens
        seqlens[:b].copy_(seqlens[:1].expand(b))
        if tq == 1:
            return base_attn_mask
        if int(seqlens[0].item()) != 0:  # (the reference reads it too, :202)
            raise ValueError(
                "goda_amd FlashAttention: doc_ids over a KV cache that already holds tokens; the document mask "
                "covers only the new tokens (mint/nn/flashattn.py:238-240)"
            )
        docs = doc_ids[:, None, :, None] == doc_ids[:, None, None, :]
        return docs if base_attn_mask is None else docs & base_attn_mask

    # mint/nn/flashattn.py:87-172
    def _attention(self, q, k, v, *, causal, window_left, doc_ids, base_attn_mask, rope, start_pos, alibi_slopes,
                   qk_norm):
        b, t, hq, d = q.shape
        hkv = k.shape[2]
        segments = None
        if doc_ids is not None and base_attn_mask is None:
            segments = _segments(doc_ids)
            if not segments[2]:
                segments = None  # an id recurs in separate runs of a row: the dense mask below
        if segments is not None:
            kw = _norm_kwargs(qk_norm, q=True, k=True)
            if not headdim.is_native(d) or _rope_in_torch(rope, t):
                # norm and RoPE as torch ops, before the packing (and the
                # zero-padding of a head dim without kernels)
                if qk_norm is not None:
                    q, k = headdim.rms_norm(q, qk_norm[0], qk_norm[2]), headdim.rms_norm(k, qk_norm[1], qk_norm[2])
                    kw = {}
                if rope is not None:
                    q, k = _rotate(q, rope, start_pos), _rotate(k, rope, start_pos)
            elif rope is not None:
                # Positions are row positions, not document positions: the
                # kernels take a packed row's index modulo the row length
                # (RoPE comes before attention in goda too, mint/nn/attn.py:60).
                tables = [x[start_pos : start_pos + t] for x in rope]
                if any(x.shape[0] != t for x in tables):
                    raise ValueError(f"goda_amd FlashAttention: RoPE tables of {rope[0].shape[0]} positions; rows "
                                     f"{start_pos} .. {start_pos + t - 1} are needed")
                if t < 64:  # (the kernels' least table: the same positions over and over)
                    tables = [x.repeat(-(-64 // t), 1) for x in tables]
                kw.update(rope_cos=tables[0], rope_sin=tables[1], rope_q=True, rope_k=True, rope_packed_rows=True)
            cu, max_len, _ = segments
            o = autograd.attention_prefill(
                q.reshape(b * t, hq, d),
                k.reshape(b * t, hkv, d),
                v.reshape(b * t, hkv, d),
                causal=causal,
                window_left=window_left,
                alibi_slopes=alibi_slopes,
                cu_seqlens_q=cu,
                cu_seqlens_k=cu,
                max_seqlen_q=max_len,
                max_seqlen_k=max_len,
                **kw,
            )
            return o.reshape(b, t, hq, d)
        kw = _norm_kwargs(qk_norm, q=True, k=True)
        if rope is not None:
            kw.update(rope_cos=rope[0], rope_sin=rope[1], rope_q=True, rope_k=True,
                      rope_q_offset=start_pos, rope_k_offset=start_pos)
        mask = base_attn_mask
        if doc_ids is not None:
            # The document mask over whole rows (with base_attn_mask, their
            # conjunction), as the reference builds it
            # (mint/nn/flashattn.py:238-243), on the dense kernel.
            docs = doc_ids[:, None, :, None] == doc_ids[:, None, None, :]
            mask = docs if mask is None else docs & mask
        if mask is not None:
            kw["attn_mask"] = mask
        return autograd.attention_prefill(q, k, v, causal=causal, window_left=window_left,
                                          alibi_slopes=alibi_slopes, **kw)

    # mint/nn/flashattn.py:174-219
    def _attention_with_kvcache(self, q, k, v, kv_cache: KVCache, *, causal, window_left, base_attn_mask, rope,
                                start_pos, alibi_slopes, qk_norm):
        """Append k/v at each sequence's cache length, then attend over the
        visible cache. With fused RoPE and an integer `start_pos` (what goda's
        attention layer passes), q and the new k rotate at start_pos + t, as
        goda's RoPE(q, k, start_pos) does (mint/nn/pos.py:100-112); with
        start_pos None they rotate at their cache positions."""
        b, tq, d = q.shape[0], q.shape[1], q.shape[-1]
        rope_kw = {}
        if rope is not None:
            rope_kw = dict(rope_cos=rope[0], rope_sin=rope[1], rope_q=True)
            if start_pos is not None:
                rope_kw.update(rope_q_offset=int(start_pos), rope_pos_abs=True)
        kv_cache.append(k, v, **({} if rope is None else dict(rope_cos=rope[0], rope_sin=rope[1],
                                                              start_pos=start_pos)),
                        **_norm_kwargs(qk_norm, q=False, k=True))
        k_cache, v_cache, seqlens = kv_cache.cache_tensors()
        used = seqlens[:b]
        native = headdim.is_native(d)
        if native:
            kw = _norm_kwargs(qk_norm, q=True, k=False)
            kw.update(rope_kw)
        else:
            # A head dim without kernels: norm and RoPE as torch ops at the
            # kernel's positions, q zero-padded like the stored rows, the
            # real head dim's scale, the output sliced back.
            if qk_norm is not None:
                q = headdim.rms_norm(q, qk_norm[0], qk_norm[2])
            if rope is not None:
                tt = torch.arange(tq, device=q.device)
                pos = int(start_pos) + tt if start_pos is not None else used[:, None].long() - tq + tt
                q = headdim.rotate(q, rope[0].float(), rope[1].float(), pos)
            q = headdim.pad(q, k_cache.shape[-1])
            kw = {"softmax_scale": 1.0 / math.sqrt(d)}
        if tq == 1 and base_attn_mask is None:
            # One new token: the bottom-right causal mask admits every cached
            # key, so causal and non-causal coincide (mint/nn/flashattn.py:245-264).
            o = ops.attention_decode(q, k_cache, v_cache, used, window_left=window_left,
                                     alibi_slopes=alibi_slopes, **kw)
            return o if native else o[..., :d]
        # Chunked prefill over the cache: the launch covers the keys the cache
        # can hold now (its host-side length bound), not max_seq_len.
        lk = kv_cache.max_seq_len if kv_cache.len_bound is None else max(1, kv_cache.len_bound)
        if base_attn_mask is not None:
            # the mask names the keys up to the cache's current end; the launch
            # may reach past them (to the host bound), where keys are hidden
            kw["attn_mask"] = ops.pack_mask(base_attn_mask, b, q.shape[2], tq, lk, q.device, allow_short_keys=True)
        o = ops.attention_prefill(q, k_cache[:b, :lk], v_cache[:b, :lk], causal=causal, window_left=window_left,
                                  alibi_slopes=alibi_slopes, seqused_k=used, **kw)
        return o if native else o[..., :d]


def _needs_grad(*ts) -> bool:
    return torch.is_grad_enabled() and any(t.requires_grad for t in ts)


def _norm_kwargs(qk_norm, *, q: bool, k: bool) -> dict:
    if qk_norm is None:
        return {}
    kw = {"norm_eps": float(qk_norm[2])}
    if q:
        kw["q_norm_weight"] = qk_norm[0]
    if k:
        kw["k_norm_weight"] = qk_norm[1]
    return kw


def _rope_in_torch(rope, t: int) -> bool:
    """Documents' RoPE that the kernels do not take: tables that receive
    gradients, and a single position for every row."""
    return rope is not None and (_needs_grad(*rope) or (t > 1 and any(x.shape[0] == 1 for x in rope)))


def _rotate(x: torch.Tensor, rope: tuple[torch.Tensor, torch.Tensor], start_pos: int) -> torch.Tensor:
    # (documents whose RoPE does not run in the kernels)
    t = x.shape[1]
    cos = rope[0][start_pos : start_pos + t][None, :, None, :].to(x.dtype)
    sin = rope[1][start_pos : start_pos + t][None, :, None, :].to(x.dtype)
    h = x.shape[-1] // 2
    x1, x2 = x[..., :h], x[..., h:]
    return torch.cat([x1 * cos - x2 * sin, x1 * sin + x2 * cos], dim=-1)
