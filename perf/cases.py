"""The workloads that the attention path's speed is judged by: single passes
through the public entry points, over the sizes, directions, dtypes and options
that the framework's users run.

A case is a dict of plain values; its "kind" names the entry point and fixes
which of the other keys apply:

  step     one new token per sequence through `FlashAttention` with a `KVCache`
           (QK-RMSNorm and RoPE fused; append, then decode)
  decode   one decode token over a resident cache, a kept `ops.plan_decode`
  prefill  dense causal prefill, a kept `ops.plan_prefill` (RoPE or ALiBi)
  eval     dense causal forward through `FlashAttention` without gradients
  mix      a serving step: packed prefill of one set of sequences and a decode
           token of another, both through kept plans
  chunk    a chunk of new tokens per sequence through `FlashAttention` with a
           `KVCache` that already holds a prefix
  masked   dense forward through `FlashAttention` with a boolean mask
  train    forward and backward through `FlashAttention` (RoPE, QK-RMSNorm,
           optional left window), or through `FlashAttentionMQAKernel` ("kernel")
  docs     forward and backward of packed documents (`doc_ids`)

Inputs are drawn on the GPU from the seed alone. Ragged lengths are part of the
case (drawn from its "lengths" seed), so that its work is known without inputs.
"""

from __future__ import annotations

import math
import random
from types import SimpleNamespace

import torch

from goda_amd import ops
from goda_amd.kernels_ import FlashAttentionMQAKernel
from goda_amd.mint.kvcache import KVCache
from goda_amd.mint.nn import FlashAttention
from goda_amd.mint.nn.pos import alibi_slopes, rope_tables

DEVICE = "cuda"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
NORM_EPS = 1e-6
ROPE_BASE = 10000.0


# ---- the cases ----------------------------------------------------------------
def listed() -> list[dict]:
    return [
        # Token-by-token generation with the small model's heads: a few short
        # sequences, where launches and latency are all there is.
        dict(name="step_small", kind="step", dtype="bf16", batch=8, hq=6, hkv=2, d=128,
             lo=64, hi=2000, capacity=2048, lengths=11),
        # A decode step of a loaded server: 64 long sequences of unequal length.
        dict(name="decode_ragged", kind="decode", dtype="bf16", batch=64, hq=32, hkv=8, d=128,
             lo=1024, hi=32768, capacity=32768, lengths=405),
        # Evaluation of the small fp32 model (its default dtype) at its
        # training length.
        dict(name="eval_fp32_small", kind="eval", dtype="fp32", batch=2, t=512, hq=6, hkv=2, d=128, window=-1),
        # Long prompts of a grouped-query model: the benchmark's own workload.
        dict(name="prefill_gqa_8k", kind="prefill", dtype="bf16", batch=4, t=8192, hq=32, hkv=8, d=128, pos="rope"),
        # Prompts of a multi-query model with wide heads and ALiBi.
        dict(name="prefill_mqa_alibi", kind="prefill", dtype="bf16", batch=8, t=4096, hq=16, hkv=1, d=256, pos="alibi"),
        # Continuous batching: new prompts of all lengths packed into one
        # prefill, and a token for the sequences already running.
        dict(name="mix_ragged", kind="mix", dtype="bf16", hq=8, hkv=1, d=256, batch=16, lo=128, hi=4096,
             dec_batch=48, dec_lo=512, dec_hi=16384, capacity=16384, lengths=506),
        # Chunked prefill: the next 256 tokens of prompts of which a part is
        # cached already.
        dict(name="chunk_256", kind="chunk", dtype="bf16", batch=8, new=256, hq=32, hkv=8, d=128,
             lo=512, hi=8192, capacity=8448, lengths=21),
        # Prompts of unequal lengths in one padded batch, each with a prefix
        # that all its rows see, as a caller's own boolean mask.
        dict(name="masked_prefix", kind="masked", dtype="bf16", batch=4, t=2048, hq=16, hkv=4, d=128, full=True),
        # A training step's attention at length 4096, grouped queries, under
        # bf16 autocast.
        dict(name="train_gqa_4k", kind="train", dtype="bf16", batch=2, t=4096, hq=32, hkv=8, d=128, window=-1,
             norm=True, kernel=False),
        # The small model trained as shipped: fp32, length 512, full heads, a
        # sliding window of a quarter of the length on every other layer.
        dict(name="train_fp32_window", kind="train", dtype="fp32", batch=16, t=512, hq=4, hkv=4, d=128, window=128,
             norm=True, kernel=False),
        # Wide multi-query heads trained in the default dtype.
        dict(name="train_fp32_wide", kind="train", dtype="fp32", batch=1, t=2048, hq=16, hkv=1, d=256, window=-1,
             norm=False, kernel=False),
        # Pretraining on documents packed into rows, fp16 autocast, narrow
        # heads.
        dict(name="train_docs", kind="docs", dtype="fp16", batch=4, t=2048, hq=16, hkv=16, d=64, docs=6, lengths=31),
    ]


def _log_int(rng: random.Random, lo: int, hi: int) -> int:
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


# (query heads, KV heads, head dim) of the small, grouped, multi-query, full
# and wide models above.
_HEADS = [(6, 2, 128), (4, 4, 128), (32, 8, 128), (16, 4, 128), (8, 1, 256), (16, 1, 256), (16, 16, 64), (32, 4, 64),
          (8, 2, 256), (16, 1, 128)]


def draw(rng: random.Random) -> dict:
    """One more case of the same ranges: any kind, sizes spread over their
    logarithm, odd ones among them; the batch is cut so that no case costs
    more than the largest listed ones."""
    kind = rng.choice(["step", "decode", "eval", "prefill", "mix", "chunk", "masked", "train", "docs"])
    hq, hkv, d = rng.choice(_HEADS)
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    lengths = rng.randrange(1, 1 << 30)
    if kind == "step":
        capacity = _log_int(rng, 64, 8192)
        return dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 32), hq=hq, hkv=hkv, d=d, lo=max(1, capacity // 32),
                    hi=capacity - 1, capacity=capacity, lengths=lengths)
    if kind == "decode":
        capacity = _log_int(rng, 256, 32768)
        most = int(4.0e9 / (2 * capacity * hkv * d * 2))  # bytes of the cache's K and V
        return dict(kind=kind, dtype=rng.choice(["bf16", "fp16", "fp32"]), batch=min(_log_int(rng, 1, 64), max(1, most // 2)),
                    hq=hq, hkv=hkv, d=d, lo=max(1, capacity // 16), hi=capacity, capacity=capacity, lengths=lengths)
    if kind == "mix":
        hi = _log_int(rng, 128, 4096)
        capacity = _log_int(rng, 512, 16384)
        most = int(16 * 8 * 256 * 4096**2 / (hq * d * hi**2))
        return dict(kind=kind, dtype=dtype, hq=hq, hkv=hkv, d=d, batch=min(_log_int(rng, 2, 24), max(1, most)),
                    lo=max(1, hi // 32), hi=hi, dec_batch=_log_int(rng, 1, 48), dec_lo=max(1, capacity // 32),
                    dec_hi=capacity, capacity=capacity, lengths=lengths)
    if kind == "chunk":
        new = _log_int(rng, 2, 512)
        hi = _log_int(rng, 256, 8192)
        return dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 8), new=new, hq=hq, hkv=hkv, d=d,
                    lo=max(1, hi // 16), hi=hi, capacity=hi + new, lengths=lengths)
    t = _log_int(rng, 64, 4096)
    if kind == "eval":
        dtype = rng.choice(["fp32", "fp32", "bf16"])
        t = min(t, 2048)
        most = 2.0e10 / (hq * d * t * t)
        return dict(kind=kind, dtype=dtype, batch=max(1, min(_log_int(rng, 1, 8), int(most))), t=t, hq=hq, hkv=hkv, d=d,
                    window=rng.choice([-1, -1, max(1, t // 4)]))
    if kind == "prefill":
        t = _log_int(rng, 64, 8192)
        most = 4 * 32 * 128 * 8192**2 / (hq * d * t * t)
        return dict(kind=kind, dtype=dtype, batch=max(1, min(_log_int(rng, 1, 16), int(most))), t=t, hq=hq, hkv=hkv, d=d,
                    pos=rng.choice(["rope", "alibi"]))
    if kind == "masked":
        t = min(t, 2048)
        return dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 4), t=t, hq=hq, hkv=hkv, d=d, full=rng.random() < 0.5)
    if kind == "docs":
        t = min(t, 2048)
        return dict(kind=kind, dtype=dtype, batch=_log_int(rng, 1, 4), t=t, hq=hq, hkv=hkv, d=d,
                    docs=max(1, min(t // 16, _log_int(rng, 1, 12))), lengths=lengths)
    dtype = rng.choice(["bf16", "bf16", "fp16", "fp32"])
    if dtype == "fp32":
        t = min(t, 1024)
        most = 16 * 256 * 2048**2 / (hq * d * t * t)
    else:
        most = 2 * 32 * 128 * 4096**2 / (hq * d * t * t)
    kernel = rng.random() < 0.25
    return dict(kind="train", dtype=dtype, batch=max(1, min(_log_int(rng, 1, 16), int(most))), t=t, hq=hq, hkv=hkv, d=d,
                window=rng.choice([-1, -1, max(1, t // 4)]), norm=(not kernel) and rng.random() < 0.5, kernel=kernel)


# ---- geometry -----------------------------------------------------------------
def _lens(case: dict, n: int, lo: int, hi: int, salt: int = 0) -> list[int]:
    r = random.Random(case["lengths"] * 7 + salt)
    return [r.randint(lo, hi) for _ in range(n)]


def _doc_lens(case: dict) -> list[list[int]]:
    """Lengths of the documents of each row: `docs` pieces that fill it."""
    rows = []
    r = random.Random(case["lengths"])
    for _ in range(case["batch"]):
        cuts = sorted(r.sample(range(1, case["t"]), case["docs"] - 1))
        rows.append([b - a for a, b in zip([0, *cuts], [*cuts, case["t"]])])
    return rows


def _tri(n: int) -> int:
    return n * (n + 1) // 2


def _window_pairs(t: int, window: int) -> int:
    """Visible pairs of a causal sequence with a left window (key >= row - window)."""
    return _tri(t) if window < 0 or window >= t else _tri(t) - _tri(t - window - 1)


def _prefixes(case: dict) -> list[tuple[int, int]]:
    """(prefix, valid length) of each sequence of a masked batch."""
    t = case["t"]
    return [(max(1, t // 8 * (b % 4) + t // 16), max(1, t - (t // 5) * (b % 3))) for b in range(case["batch"])]


def _mask(case: dict) -> torch.Tensor:
    """full: [B, 1, T, T], row i sees its prefix and the keys up to itself,
    never padding; else [B, 1, 1, T], the valid keys alone."""
    t = case["t"]
    j = torch.arange(t, device=DEVICE)
    rows = []
    for prefix, valid in _prefixes(case):
        ok = (j < valid)[None]
        if case["full"]:
            ok = ok & ((j[None] < prefix) | (j[None] <= j[:, None]))
        rows.append(ok[None])
    return torch.stack(rows)


def work(case: dict) -> dict:
    """Each input read once and each output written once; 4 * D * Hq flops per
    visible pair forward, 10 backward (five products)."""
    kind, es = case["kind"], 4 if case["dtype"] == "fp32" else 2
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    if kind in ("step", "decode"):
        n = sum(_lens(case, case["batch"], case["lo"], case["hi"])) + (case["batch"] if kind == "step" else 0)
        return dict(bytes=(2 * n * hkv + 2 * case["batch"] * hq) * d * es, flops=4 * d * hq * n)
    if kind == "chunk":
        starts, new = _lens(case, case["batch"], case["lo"], case["hi"]), case["new"]
        keys = sum(starts) + new * len(starts)
        pairs = sum(new * s + _tri(new) for s in starts)
        return dict(bytes=(2 * keys * hkv + 2 * new * len(starts) * (hq + hkv)) * d * es, flops=4 * d * hq * pairs)
    if kind == "mix":
        lens = _lens(case, case["batch"], case["lo"], case["hi"])
        n = sum(_lens(case, case["dec_batch"], case["dec_lo"], case["dec_hi"], 1))
        return dict(bytes=(2 * sum(lens) * (hq + hkv) + 2 * n * hkv + 2 * case["dec_batch"] * hq) * d * es,
                    flops=4 * d * hq * (sum(_tri(x) for x in lens) + n))
    b, t = case["batch"], case["t"]
    elems = 2 * b * t * (hq + hkv) * d
    if kind == "masked":
        if case["full"]:
            pairs = sum(sum(min(v, max(p, i + 1)) for i in range(t)) for p, v in _prefixes(case))
        else:
            pairs = sum(_tri(v) + (t - v) * v for _, v in _prefixes(case))
        return dict(bytes=elems * es + b * t * (t if case["full"] else 1), flops=4 * d * hq * pairs)
    if kind in ("eval", "prefill"):
        return dict(bytes=elems * es, flops=4 * d * hq * b * _window_pairs(t, case.get("window", -1)))
    if kind == "docs":
        pairs = sum(_tri(n) for row in _doc_lens(case) for n in row)
    else:
        pairs = b * _window_pairs(t, case["window"])
    # forward: q, k, v in, o out; backward: q, k, v, o, dO in, dq, dk, dv out
    return dict(bytes=(2 * elems + b * t * hq * d) * es, flops=14 * d * hq * pairs)


def tolerance(case: dict) -> dict:
    # About four times the largest error seen against `exact`: 3.4e-6 (fp32
    # gradients), 6.2e-4 (fp16 gradients of documents, rotated in fp16), 4.1e-3
    # (bf16 gradients). "max" in units of the result's root mean square.
    if case["dtype"] == "fp32":
        return {"rel": 2e-5, "max": 1e-3}
    if case["dtype"] == "fp16":
        return {"rel": 3e-3, "max": 0.1}
    return {"rel": 2e-2, "max": 0.4}


# ---- inputs -------------------------------------------------------------------
class _Draws:
    def __init__(self, case: dict, seed: int):
        self.gen = torch.Generator(device=DEVICE)
        self.gen.manual_seed(seed * 1000003 + 17)
        self.dtype = DTYPES[case["dtype"]]

    def __call__(self, *shape, std: float = 0.5, dtype=None) -> torch.Tensor:
        out = torch.empty(shape, dtype=dtype or self.dtype, device=DEVICE)
        flat = out.view(-1)
        for part in flat.split(1 << 28):
            part.copy_(torch.randn(part.shape, generator=self.gen, device=DEVICE).mul_(std))
        return out


def _inputs(case: dict, seed: int) -> SimpleNamespace:
    s = SimpleNamespace(case=case)
    rnd, kind = _Draws(case, seed), case["kind"]
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    positions = case.get("capacity", 0) if kind in ("step", "chunk") else max(case.get("t", 0), case.get("hi", 0), case.get("capacity", 0))
    cos, sin = rope_tables(positions, d, ROPE_BASE)
    s.rope = (cos.to(DEVICE), sin.to(DEVICE))
    if kind in ("step", "chunk"):
        b, new = case["batch"], case.get("new", 1)
        s.q, s.k, s.v = rnd(b, new, hq, d), rnd(b, new, hkv, d), rnd(b, new, hkv, d)
        s.q_scale, s.k_scale = rnd(d, std=0.1, dtype=torch.float32), rnd(d, std=0.1, dtype=torch.float32)
        s.start = torch.tensor(_lens(case, b, case["lo"], case["hi"]), dtype=torch.int32, device=DEVICE)
        s.cached_k, s.cached_v = (rnd(b, hkv, case["capacity"], d) for _ in range(2))
        return s
    if kind == "mix":
        lens = _lens(case, case["batch"], case["lo"], case["hi"])
        s.lens = lens
        s.q, s.k, s.v = (rnd(sum(lens), h, d) for h in (hq, hkv, hkv))
    if kind in ("decode", "mix"):
        b = case["dec_batch"] if kind == "mix" else case["batch"]
        lo, hi, salt = (case["dec_lo"], case["dec_hi"], 1) if kind == "mix" else (case["lo"], case["hi"], 0)
        s.dec_q = rnd(b, hq, d)
        s.k_cache, s.v_cache = (rnd(b, hkv, case["capacity"], d) for _ in range(2))
        s.dec_lens = torch.tensor(_lens(case, b, lo, hi, salt), dtype=torch.int32, device=DEVICE)
        return s
    b, t = case["batch"], case["t"]
    if case.get("kernel"):  # goda's kernel layout [B, H, T, D]
        s.q, s.k, s.v, s.d_o = rnd(b, hq, t, d), rnd(b, hkv, t, d), rnd(b, hkv, t, d), rnd(b, hq, t, d)
    else:
        s.q, s.k, s.v, s.d_o = rnd(b, t, hq, d), rnd(b, t, hkv, d), rnd(b, t, hkv, d), rnd(b, t, hq, d)
    if case.get("pos") == "alibi":
        s.slopes = torch.tensor(alibi_slopes(hq), dtype=torch.float32, device=DEVICE)
    if case.get("norm"):
        s.q_scale, s.k_scale = rnd(d, std=0.1, dtype=torch.float32), rnd(d, std=0.1, dtype=torch.float32)
    if kind == "masked":
        s.mask = _mask(case)
    if kind == "docs":
        s.doc_ids = torch.stack([
            torch.repeat_interleave(torch.arange(len(row)), torch.tensor(row)) for row in _doc_lens(case)
        ]).to(DEVICE)
    return s


def prepare(case: dict, seed: int) -> SimpleNamespace:
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("step", "chunk"):
        s.attn = FlashAttention()
        s.cache = KVCache(case["batch"], case["capacity"], case["hkv"], case["d"], DTYPES[case["dtype"]], DEVICE)
        # the program sets the lengths itself, so it holds the raw tensors
        k_cache, v_cache, s.lengths = s.cache.get_cache_tensors()
        k_cache.copy_(s.cached_k.transpose(1, 2))
        v_cache.copy_(s.cached_v.transpose(1, 2))
        del s.cached_k, s.cached_v
        s.norm = (s.q_scale, s.k_scale, NORM_EPS)
    elif kind == "prefill":
        kw = dict(alibi_slopes=s.slopes) if case["pos"] == "alibi" else dict(
            rope_cos=s.rope[0], rope_sin=s.rope[1], rope_q=True, rope_k=True)
        s.plan = ops.plan_prefill(s.q, s.k, s.v, causal=True, **kw)
    if kind == "mix":
        cu = [0]
        for n in s.lens:
            cu.append(cu[-1] + n)
        cu = torch.tensor(cu, dtype=torch.int32, device=DEVICE)
        s.plan = ops.plan_prefill(s.q, s.k, s.v, causal=True, rope_cos=s.rope[0], rope_sin=s.rope[1], rope_q=True, rope_k=True,
                                  cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=max(s.lens), max_seqlen_k=max(s.lens))
    if kind in ("decode", "mix"):
        kw = dict(rope_cos=s.rope[0], rope_sin=s.rope[1], rope_q=True) if kind == "mix" else {}
        s.dec_plan = ops.plan_decode(s.dec_q, s.k_cache, s.v_cache, s.dec_lens, cache_layout="bhtd", **kw)
    if kind in ("eval", "masked"):
        s.attn = FlashAttention()
    if kind in ("train", "docs"):
        s.attn = FlashAttention()
        for x in (s.q, s.k, s.v):
            x.requires_grad_(True)
        if case.get("norm"):
            s.q_scale.requires_grad_(True)
            s.k_scale.requires_grad_(True)
    return s


def run(s: SimpleNamespace):
    case = s.case
    kind = case["kind"]
    if kind in ("step", "chunk"):
        # back to the accepted length, as a program does that samples several
        # continuations of one prefix
        s.lengths.copy_(s.start)
        with torch.no_grad():
            o = s.attn(s.q, s.k, s.v, causal=True, kv_cache=s.cache, rope=s.rope, qk_norm=s.norm)
        return o, s.cache.k_cache, s.cache.v_cache, s.lengths
    if kind == "decode":
        return s.dec_plan()
    if kind == "prefill":
        return s.plan()
    if kind == "mix":
        return s.plan(), s.dec_plan()
    if kind == "eval":
        with torch.no_grad():
            return s.attn(s.q, s.k, s.v, causal=True, window_size=(case["window"], -1), rope=s.rope)
    if kind == "masked":
        # a mask that shows a prefix replaces the causal one; padding is on top of it
        with torch.no_grad():
            return s.attn(s.q, s.k, s.v, causal=not case["full"], base_attn_mask=s.mask, rope=s.rope)
    if kind == "docs":
        o = s.attn(s.q, s.k, s.v, causal=True, doc_ids=s.doc_ids, rope=s.rope)
        return o, *torch.autograd.grad(o, (s.q, s.k, s.v), s.d_o)
    leaves = [s.q, s.k, s.v]
    if case["kernel"]:
        o = FlashAttentionMQAKernel.apply(s.q, s.k, s.v, True, case["d"] ** -0.5, s.rope[0], s.rope[1], None, case["window"])
    else:
        norm = None
        if case["norm"]:
            norm = (s.q_scale, s.k_scale, NORM_EPS)
            leaves += [s.q_scale, s.k_scale]
        o = s.attn(s.q, s.k, s.v, causal=True, window_size=(case["window"], -1), rope=s.rope, qk_norm=norm)
    return o, *torch.autograd.grad(o, leaves, s.d_o)


# ---- the same results in 64 bits ----------------------------------------------
def _norm64(x, scale):
    return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + NORM_EPS) * (1.0 + scale)


def _rope64(x, rope, pos):
    """Half-split rotation of x [B, T, H, D] at positions [T] or [B, T]."""
    c, s = rope[0].double()[pos], rope[1].double()[pos]
    if c.dim() == 2:
        c, s = c[None], s[None]
    c, s = c[:, :, None], s[:, :, None]
    a, b = x.chunk(2, -1)
    return torch.cat([a * c - b * s, a * s + b * c], -1)


def _head64(q, k, v, hidden, bias=None):
    """Attention of one head: q [Lq, D], k, v [Lk, D]; hidden [Lq, Lk] or None."""
    s = (q @ k.t()) * q.shape[-1] ** -0.5
    if bias is not None:
        s = s + bias
    if hidden is not None:
        s.masked_fill_(hidden, -math.inf)
    p = torch.softmax(s, -1)
    return p, p @ v


def _heads64(q, k, v, hidden, slopes=None, d_o=None):
    """q [Lq, Hq, D], k, v [Lk, Hkv, D] of one sequence; o, and with d_o also
    (dq, dk, dv), a head at a time."""
    lq, hq, d = q.shape
    lk, hkv, _ = k.shape
    group = hq // hkv
    o = torch.empty_like(q)
    dq, dk, dv = torch.empty_like(q), torch.zeros_like(k), torch.zeros_like(v)
    off = None
    if slopes is not None:
        off = (torch.arange(lk, device=q.device)[None] - (torch.arange(lq, device=q.device)[:, None] + lk - lq)).double()
    for h in range(hq):
        qh, kh, vh = q[:, h].contiguous(), k[:, h // group].contiguous(), v[:, h // group].contiguous()
        p, oh = _head64(qh, kh, vh, hidden, None if off is None else off * slopes[h].double())
        o[:, h] = oh
        if d_o is not None:
            g = d_o[:, h].contiguous()
            dv[:, h // group] += p.t().contiguous() @ g
            ds = g @ vh.t().contiguous()
            ds -= (g * oh).sum(-1, keepdim=True)
            ds *= p
            ds *= d**-0.5
            dq[:, h] = ds @ kh
            dk[:, h // group] += ds.t().contiguous() @ qh
    return (o, dq, dk, dv) if d_o is not None else o


def _causal_hidden(lq: int, lk: int, window: int = -1) -> torch.Tensor:
    i = torch.arange(lq, device=DEVICE)[:, None] + (lk - lq)
    j = torch.arange(lk, device=DEVICE)[None]
    hidden = j > i
    if window >= 0:
        hidden |= j < i - window
    return hidden


def _decode64(q, k_cache, v_cache, lens, rope=None):
    """q [B, Hq, D] over caches [B, Hkv, L, D]."""
    o = torch.empty(q.shape, dtype=torch.float64, device=q.device)
    for b, n in enumerate(lens.tolist()):
        x = q[b : b + 1, None].double()
        if rope is not None:
            x = _rope64(x, rope, torch.tensor([n - 1], device=q.device))
        for h in range(k_cache.shape[1]):
            group = q.shape[1] // k_cache.shape[1]
            rows = slice(h * group, (h + 1) * group)
            o[b, rows] = _head64(x[0, 0, rows], k_cache[b, h, :n].double(), v_cache[b, h, :n].double(), None)[1]
    return o


def exact(case: dict, seed: int):
    s = _inputs(case, seed)
    kind = case["kind"]
    if kind in ("step", "chunk"):
        new = case.get("new", 1)
        pos = s.start.long()[:, None] + torch.arange(new, device=DEVICE)
        q = _rope64(_norm64(s.q.double(), s.q_scale.double()), s.rope, pos)
        k = _rope64(_norm64(s.k.double(), s.k_scale.double()), s.rope, pos)
        v = s.v.double()
        ck, cv = s.cached_k.transpose(1, 2).double(), s.cached_v.transpose(1, 2).double()
        o = torch.empty(q.shape, dtype=torch.float64, device=DEVICE)
        for b, n in enumerate(s.start.tolist()):
            ck[b, n : n + new], cv[b, n : n + new] = k[b], v[b]
            o[b] = _heads64(q[b], ck[b, : n + new], cv[b, : n + new], _causal_hidden(new, n + new))
        return o, ck, cv, s.start + new
    if kind == "decode":
        return _decode64(s.dec_q, s.k_cache, s.v_cache, s.dec_lens)
    if kind == "mix":
        o, at = torch.empty(s.q.shape, dtype=torch.float64, device=DEVICE), 0
        for n in s.lens:
            pos = torch.arange(n, device=DEVICE)
            q, k = (_rope64(x[None, at : at + n].double(), s.rope, pos)[0] for x in (s.q, s.k))
            o[at : at + n] = _heads64(q, k, s.v[at : at + n].double(), _causal_hidden(n, n))
            at += n
        return o, _decode64(s.dec_q, s.k_cache, s.v_cache, s.dec_lens, s.rope)

    t = case["t"]
    leaves = [x.double() for x in (s.q, s.k, s.v)]
    if case.get("norm"):
        leaves += [s.q_scale.double(), s.k_scale.double()]
    grad = kind in ("train", "docs")
    with torch.enable_grad():
        for x in leaves:
            x.requires_grad_(grad)
        q, k, v = leaves[:3]
        if case.get("kernel"):
            q, k, v = (x.transpose(1, 2) for x in (q, k, v))
        if case.get("norm"):
            q, k = _norm64(q, leaves[3]), _norm64(k, leaves[4])
        if case.get("pos") != "alibi":
            pos = torch.arange(t, device=DEVICE)
            q, k = _rope64(q, s.rope, pos), _rope64(k, s.rope, pos)
    d_o = (s.d_o.transpose(1, 2) if case.get("kernel") else s.d_o).double() if grad else None
    hidden = _causal_hidden(t, t, case.get("window", -1))
    outs = []
    with torch.no_grad():
        for b in range(case["batch"]):
            hid = hidden
            if kind == "docs":
                hid = hidden | (s.doc_ids[b][:, None] != s.doc_ids[b][None])
            elif kind == "masked":
                hid = ~s.mask[b, 0] if case["full"] else hidden | ~s.mask[b, 0]
            outs.append(_heads64(q[b], k[b], v[b], hid, getattr(s, "slopes", None), d_o[b] if grad else None))
        if not grad:
            return torch.stack(outs)
        o, dq, dk, dv = (torch.stack(x) for x in zip(*outs))
    grads = torch.autograd.grad((q, k, v), leaves, (dq, dk, dv))
    if case.get("kernel"):
        o = o.transpose(1, 2)
    return o, *grads
