"""Backward parity: dq, dk, dv from goda_attn_prefill_bwd (through the C-ABI)
against the CPU oracle's gradients (torch autograd through the SDPA
restatement, pinned by tests/test_oracle.py against finite differences).

Tolerance: the north-star absolute bounds (1e-4 fp32, 2e-2 bf16/fp16) on top of
the gradient's own storage rounding at the largest reference value (2^-8 |x|
in bf16, 2^-11 |x| in fp16, 2^-24 |x| in fp32): gradient magnitudes grow with
the number of rows and group heads that feed one key, and a 16-bit output
cannot hold x more closely than its rounding.
"""

from __future__ import annotations

import math
import re

import numpy as np
import pytest
import torch

from goda_amd import autograd, ops
from goda_amd import workloads as wl
from goda_amd.kernels_ import FlashAttentionGQAKernel, FlashAttentionMQAKernel
from goda_amd.mint.nn import FlashAttention, GroupedQueryAttention, RoPE
from oracle import attention as ref
from oracle import brute
from tests.helpers import TOL

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _rand(shape, dtype, seed, std=0.5):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).to(dtype)


# Largest rounding error of a stored value x relative to |x|: a 16-bit
# gradient cannot hold x more closely than that.
STORAGE = {torch.float32: 2.0**-24, torch.bfloat16: 2.0**-8, torch.float16: 2.0**-11}


def grad_bound(x_ref: torch.Tensor, dtype) -> float:
    """The north-star absolute bound on top of the output's own storage
    rounding at the largest reference gradient (which alone reaches 2e-2 in
    bf16 once |x| >= 8: bench-shape dv reaches 7.7 and 16.5)."""
    return TOL[dtype] + STORAGE[dtype] * x_ref.abs().max().item()


def _check(grads, refs, dtype, what=""):
    for name, g, r in zip(("dq", "dk", "dv"), grads, refs):
        r = r.to("cpu", torch.float32)
        e = (g.to("cpu", torch.float32) - r).abs().max().item()
        bound = grad_bound(r, dtype)
        assert e <= bound, f"{what} {name} err {e} > {bound} (max |ref| {r.abs().max().item()})"


def _case(b, tq, tk, hq, hkv, d, dtype, *, causal, window=-1, alibi=False, rope=False, seed=0):
    q = _rand((b, tq, hq, d), dtype, seed)
    k = _rand((b, tk, hkv, d), dtype, seed + 1)
    v = _rand((b, tk, hkv, d), dtype, seed + 2)
    d_o = _rand((b, tq, hq, d), dtype, seed + 3, std=1.0)
    kw, okw = {}, {}
    if alibi:
        slopes = torch.tensor(wl.alibi_slopes(hq), dtype=torch.float32)
        kw["alibi_slopes"] = slopes.to(DEV)
        okw["alibi_slopes"] = slopes
    if rope:
        cos, sin = wl.rope_tables(tk + 8, d, 10000.0)
        kw.update(rope_cos=cos.to(DEV), rope_sin=sin.to(DEV), rope_q=True, rope_k=True)
        okw["rope"] = (cos, sin, torch.arange(tk - tq, tk), torch.arange(tk))
    qg, kg, vg = q.to(DEV), k.to(DEV), v.to(DEV)
    o, lse = ops.attention_prefill(qg, kg, vg, causal=causal, window_left=window, return_lse=True, **kw)
    dq, dk, dv = ops.attention_prefill_bwd(qg, kg, vg, o, lse, d_o.to(DEV), causal=causal, window_left=window, **kw)
    torch.cuda.synchronize()
    refs = ref.attention_grads(q.float(), k.float(), v.float(), d_o.float(), causal=causal,
                               window_size=(window, -1), **okw)
    _check((dq, dk, dv), refs, dtype, f"b{b} tq{tq} tk{tk} h{hq}/{hkv} d{d} {dtype} causal={causal}")
    assert dq.shape == q.shape and dk.shape == k.shape and dv.shape == v.shape


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("hq,hkv", [(8, 2), (4, 4), (6, 1)])
@pytest.mark.parametrize("causal", [True, False])
def test_backward_shapes(dtype, d, hq, hkv, causal):
    _case(2, 70, 70, hq, hkv, d, dtype, causal=causal, seed=d + hq)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("window", [0, 5, 40])
def test_backward_window(dtype, window):
    _case(2, 96, 96, 4, 2, 128, dtype, causal=True, window=window, seed=window)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward_bottom_right_and_long(dtype):
    _case(1, 50, 90, 8, 2, 128, dtype, causal=True, seed=5)  # Lq < Lk
    _case(1, 300, 300, 4, 1, 128, dtype, causal=True, seed=6)  # several key blocks


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward_alibi_and_rope(dtype):
    _case(2, 64, 64, 8, 2, 128, dtype, causal=True, alibi=True, seed=7)
    _case(2, 64, 64, 8, 2, 128, dtype, causal=True, rope=True, seed=8)
    _case(1, 40, 72, 4, 1, 256, dtype, causal=True, rope=True, seed=9)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_backward_d256_paths(dtype):
    """head_dim 256 runs its own dk/dv kernel: one query tile (each key block
    writes dk/dv directly), MQA with ALiBi over several key blocks (the walk is
    split over workgroups whose partials a reduction sums), a window, and
    Lq < Lk."""
    _case(1, 20, 90, 4, 4, 256, dtype, causal=True, seed=11)
    _case(2, 100, 300, 16, 1, 256, dtype, causal=True, alibi=True, seed=12)
    _case(1, 96, 96, 4, 2, 256, dtype, causal=True, window=40, seed=13)
    _case(1, 50, 170, 8, 2, 256, dtype, causal=True, rope=True, seed=14)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_backward_d256_dq_from_stored_ds(dtype):
    """At head_dim 256 with an even query-head group, dq is one product over
    the dS tiles the dk/dv kernel stored: causal batches keep only the visible
    key tiles (Lq < Lk shifts the diagonal by whole and partial tiles), others
    keep all; workgroups whose four waves cover several query tiles (group 2,
    6) walk key tiles some waves do not see. An odd group (5, 3) recomputes
    S and dP instead."""
    _case(2, 70, 70, 6, 1, 256, dtype, causal=True, seed=41)
    _case(1, 33, 101, 4, 2, 256, dtype, causal=True, seed=42)  # diagonal 68 keys in
    _case(1, 64, 128, 2, 1, 256, dtype, causal=True, seed=43)  # diagonal 2 whole tiles in
    _case(2, 90, 40, 4, 2, 256, dtype, causal=True, seed=44)  # Lq > Lk: all tiles kept
    _case(1, 75, 75, 2, 2, 256, dtype, causal=False, seed=45)
    _case(1, 96, 96, 6, 3, 256, dtype, causal=True, window=33, seed=46)
    _case(2, 60, 60, 5, 1, 256, dtype, causal=True, seed=47)
    _case(1, 60, 60, 3, 3, 256, dtype, causal=False, seed=48)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_backward_d256_varlen_and_seqused(dtype):
    """Stored dS tiles of ragged batches: packed sequences (all key tiles of
    the longest kept per sequence) and seqused_k (a dense causal batch whose
    sequences see fewer keys than its tile rows hold)."""
    lens = [33, 1, 70, 12]
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    tot, hq, hkv, d = int(cu[-1]), 8, 2, 256
    q, k, v = _rand((tot, hq, d), dtype, 51), _rand((tot, hkv, d), dtype, 52), _rand((tot, hkv, d), dtype, 53)
    d_o = _rand((tot, hq, d), dtype, 54, std=1.0)
    kw = dict(causal=True, cu_seqlens_q=cu.to(DEV), cu_seqlens_k=cu.to(DEV), max_seqlen_q=max(lens), max_seqlen_k=max(lens))
    o, lse = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), return_lse=True, **kw)
    dq, dk, dv = ops.attention_prefill_bwd(q.to(DEV), k.to(DEV), v.to(DEV), o, lse, d_o.to(DEV), **kw)
    for s, e in zip(cu[:-1].tolist(), cu[1:].tolist()):
        refs = ref.attention_grads(q[s:e][None].float(), k[s:e][None].float(), v[s:e][None].float(),
                                   d_o[s:e][None].float(), causal=True)
        _check((dq[s:e][None], dk[s:e][None], dv[s:e][None]), refs, dtype, f"segment {s}:{e}")

    b, tq, tk = 2, 40, 100
    q, k, v = _rand((b, tq, hq, d), dtype, 55), _rand((b, tk, hkv, d), dtype, 56), _rand((b, tk, hkv, d), dtype, 57)
    d_o = _rand((b, tq, hq, d), dtype, 58, std=1.0)
    used = torch.tensor([45, 100], dtype=torch.int32)
    kw = dict(causal=True, seqused_k=used.to(DEV))
    o, lse = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), return_lse=True, **kw)
    dq, dk, dv = ops.attention_prefill_bwd(q.to(DEV), k.to(DEV), v.to(DEV), o, lse, d_o.to(DEV), **kw)
    for i, L in enumerate(used.tolist()):
        refs = ref.attention_grads(q[i : i + 1].float(), k[i : i + 1, :L].float(), v[i : i + 1, :L].float(),
                                   d_o[i : i + 1].float(), causal=True)
        _check((dq[i : i + 1], dk[i : i + 1, :L], dv[i : i + 1, :L]), refs, dtype, f"seq {i}")
        assert torch.all(dk[i, L:].cpu() == 0) and torch.all(dv[i, L:].cpu() == 0)


def test_backward_workgroup_order_partial_chunks():
    """The dk/dv and dq grids are walked in chunks of 8 (head group or pair)
    units, heaviest block of each unit first; unit counts that leave a partial
    last chunk (3 x 6 = 18 units at head_dim 128; 5 x 2 x splits at 256 with
    the split dk/dv walk) must still visit every block exactly once."""
    _case(3, 160, 160, 12, 6, 128, torch.bfloat16, causal=True, seed=21)
    _case(5, 130, 130, 8, 2, 256, torch.bfloat16, causal=True, rope=True, seed=22)
    _case(3, 70, 70, 12, 6, 128, torch.float32, causal=True, seed=23)


@pytest.mark.parametrize("d,hq,hkv,alibi", [(128, 8, 2, False), (256, 16, 1, True)])
def test_forward_backward_run_to_run_bit_identical(d, hq, hkv, alibi):
    """No atomics or order-dependent sums anywhere on the path: two calls on
    the same inputs give the same bits (o, lse, dq, dk, dv), including the
    head_dim-256 dk/dv walk split over workgroups whose fp32 partials a
    separate pass sums in a fixed order."""
    b, t, dtype = 2, 1000, torch.bfloat16
    q = _rand((b, t, hq, d), dtype, 31).to(DEV)
    k = _rand((b, t, hkv, d), dtype, 32).to(DEV)
    v = _rand((b, t, hkv, d), dtype, 33).to(DEV)
    d_o = _rand((b, t, hq, d), dtype, 34, std=1.0).to(DEV)
    kw = {"alibi_slopes": torch.tensor(wl.alibi_slopes(hq), dtype=torch.float32, device=DEV)} if alibi else {}
    runs = []
    for _ in range(2):
        o, lse = ops.attention_prefill(q, k, v, causal=True, return_lse=True, **kw)
        runs.append((o, lse) + tuple(ops.attention_prefill_bwd(q, k, v, o, lse, d_o, causal=True, **kw)))
    torch.cuda.synchronize()
    for name, x, y in zip(("o", "lse", "dq", "dk", "dv"), runs[0], runs[1]):
        assert torch.isfinite(x).all() and x.abs().max().item() > 0, name
        assert torch.equal(x, y), f"{name} differs between two calls (d={d})"


def test_backward_rows_without_keys():
    """Lq > Lk with causal: the first Lq - Lk rows see no key; their o is 0
    and they contribute nothing (checked against the float64 brute force)."""
    b, tq, tk, hq, hkv, d = 1, 12, 8, 2, 1, 64
    q, k, v = (_rand(s, torch.float32, i) for i, s in enumerate([(b, tq, hq, d), (b, tk, hkv, d), (b, tk, hkv, d)]))
    d_o = _rand((b, tq, hq, d), torch.float32, 9, std=1.0)
    o, lse = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), causal=True, return_lse=True)
    dq, dk, dv = ops.attention_prefill_bwd(q.to(DEV), k.to(DEV), v.to(DEV), o, lse, d_o.to(DEV), causal=True)
    bq, bk, bv = brute.attention_backward(q.numpy(), k.numpy(), v.numpy(), d_o.numpy(), causal=True)
    for g, r in ((dq, bq), (dk, bk), (dv, bv)):
        assert (g.cpu().double() - torch.from_numpy(r)).abs().max().item() <= 1e-4
    assert torch.all(dq[:, : tq - tk].cpu() == 0)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward_varlen(dtype):
    lens = [33, 1, 70, 12]
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32)
    tot, hq, hkv, d = int(cu[-1]), 8, 2, 128
    q, k, v = _rand((tot, hq, d), dtype, 1), _rand((tot, hkv, d), dtype, 2), _rand((tot, hkv, d), dtype, 3)
    d_o = _rand((tot, hq, d), dtype, 4, std=1.0)
    kw = dict(causal=True, cu_seqlens_q=cu.to(DEV), cu_seqlens_k=cu.to(DEV), max_seqlen_q=max(lens), max_seqlen_k=max(lens))
    o, lse = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), return_lse=True, **kw)
    dq, dk, dv = ops.attention_prefill_bwd(q.to(DEV), k.to(DEV), v.to(DEV), o, lse, d_o.to(DEV), **kw)
    for s, e in zip(cu[:-1].tolist(), cu[1:].tolist()):
        refs = ref.attention_grads(q[s:e][None].float(), k[s:e][None].float(), v[s:e][None].float(),
                                   d_o[s:e][None].float(), causal=True)
        _check((dq[s:e][None], dk[s:e][None], dv[s:e][None]), refs, dtype, f"segment {s}:{e}")


def test_backward_seqused_k_zeroes_unused_keys():
    b, tq, tk, hq, hkv, d = 2, 16, 64, 4, 2, 128
    q, k, v = _rand((b, tq, hq, d), torch.float32, 1), _rand((b, tk, hkv, d), torch.float32, 2), _rand((b, tk, hkv, d), torch.float32, 3)
    d_o = _rand((b, tq, hq, d), torch.float32, 4, std=1.0)
    used = torch.tensor([40, 64], dtype=torch.int32)
    kw = dict(causal=True, seqused_k=used.to(DEV))
    o, lse = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), return_lse=True, **kw)
    dq, dk, dv = ops.attention_prefill_bwd(q.to(DEV), k.to(DEV), v.to(DEV), o, lse, d_o.to(DEV), **kw)
    for i, L in enumerate(used.tolist()):
        refs = ref.attention_grads(q[i : i + 1], k[i : i + 1, :L], v[i : i + 1, :L], d_o[i : i + 1], causal=True)
        _check((dq[i : i + 1], dk[i : i + 1, :L], dv[i : i + 1, :L]), refs, torch.float32, f"seq {i}")
        assert torch.all(dk[i, L:].cpu() == 0) and torch.all(dv[i, L:].cpu() == 0)


@pytest.mark.parametrize("cls", [FlashAttentionGQAKernel, FlashAttentionMQAKernel])
def test_kernels_apply_backward(cls):
    """kernels_/flash_attn_gqa/cuda.py:577-658: loss.backward() through
    apply(Q, K, V, causal, tau) on [B, H, T, D] gives dQ, dK, dV."""
    b, hq, hkv, t, d = 2, 8, 2, 80, 128
    q = _rand((b, hq, t, d), torch.bfloat16, 1).to(DEV).requires_grad_(True)
    k = _rand((b, hkv, t, d), torch.bfloat16, 2).to(DEV).requires_grad_(True)
    v = _rand((b, hkv, t, d), torch.bfloat16, 3).to(DEV).requires_grad_(True)
    d_o = _rand((b, hq, t, d), torch.bfloat16, 4, std=1.0)
    o = cls.apply(q, k, v, True, 1.0 / math.sqrt(d))
    o.backward(d_o.to(DEV))
    refs = ref.attention_grads(q.detach().transpose(1, 2).float(), k.detach().transpose(1, 2).float(),
                               v.detach().transpose(1, 2).float(), d_o.transpose(1, 2).float(), causal=True)
    _check((q.grad.transpose(1, 2), k.grad.transpose(1, 2), v.grad.transpose(1, 2)), refs, torch.bfloat16)


@pytest.mark.parametrize("with_rope", [False, True])
def test_flashattention_doc_ids_backward(with_rope):
    b, t, hq, hkv, d = 2, 64, 4, 2, 128
    q = _rand((b, t, hq, d), torch.float32, 1)
    k = _rand((b, t, hkv, d), torch.float32, 2)
    v = _rand((b, t, hkv, d), torch.float32, 3)
    d_o = _rand((b, t, hq, d), torch.float32, 4, std=1.0)
    doc = torch.tensor([[0] * 20 + [1] * 30 + [2] * 14, [5] * 64])
    kw, okw = {}, {}
    if with_rope:
        cos, sin = wl.rope_tables(t, d, 10000.0)
        kw["rope"] = (cos.to(DEV), sin.to(DEV))
        okw["rope"] = (cos, sin, torch.arange(t), torch.arange(t))
    qg, kg, vg = (x.to(DEV).requires_grad_(True) for x in (q, k, v))
    o = FlashAttention()(qg, kg, vg, causal=True, doc_ids=doc.to(DEV), **kw)
    o.backward(d_o.to(DEV))
    refs = ref.attention_grads(q, k, v, d_o, causal=True, doc_ids=doc, **okw)
    _check((qg.grad, kg.grad, vg.grad), refs, torch.float32)


def test_autograd_entry_is_plain_forward_without_grad():
    q = _rand((1, 16, 2, 64), torch.bfloat16, 1).to(DEV)
    with torch.no_grad():
        o = autograd.attention_prefill(q, q[:, :, :1], q[:, :, :1], causal=True)
    assert o.grad_fn is None


def test_gqa_layer_training_step_matches_cpu_reference():
    """One training step of GroupedQueryAttention (mint/nn/attn.py:39-77) with
    fused RoPE: parameter gradients from the HIP forward + backward equal those
    of the same layer on the CPU with the oracle attention (fp32)."""
    torch.manual_seed(0)
    e, hq, hkv, d, t = 256, 4, 2, 128, 48
    rope = RoPE(seq_len=64, head_dim=d, rope_base_theta=10000)
    layer = GroupedQueryAttention(hq, hkv, d, e, rope, torch.float32)
    with torch.no_grad():
        for p_ in layer.parameters():
            p_.normal_(0, 0.05)
    x = torch.randn(2, t, e) * 0.5
    gy = torch.randn(2, t, e)

    layer_g = layer.to(DEV)
    y = layer_g(x.to(DEV))
    y.backward(gy.to(DEV))
    grads = {n: p_.grad.detach().cpu() for n, p_ in layer_g.named_parameters()}

    # CPU reference: the same computation with the oracle attention.
    sd = {n: p_.detach().cpu().float().requires_grad_(True) for n, p_ in layer_g.named_parameters()}

    def rms(z, scale):
        return z * torch.rsqrt(z.pow(2).mean(-1, keepdim=True) + 1e-6) * (1.0 + scale)

    qf = (x @ sd["wq.weight"].T).view(2, t, hq, d)
    kf = (x @ sd["wk.weight"].T).view(2, t, hkv, d)
    vf = (x @ sd["wv.weight"].T).view(2, t, hkv, d)
    qf, kf = rms(qf, sd["q_norm.scale"]), rms(kf, sd["k_norm.scale"])
    pos = torch.arange(t)
    qf = ref.apply_rope(qf, rope.cos.cpu(), rope.sin.cpu(), pos)
    kf = ref.apply_rope(kf, rope.cos.cpu(), rope.sin.cpu(), pos)
    o = ref.attention(qf, kf, vf, causal=True)
    y_ref = o.reshape(2, t, -1) @ sd["wo.weight"].T
    y_ref.backward(gy)
    for n, g in grads.items():
        # parameter gradients sum over every row: compared relative to their size
        r = sd[n].grad
        e = ((g.cpu().float() - r).abs().max() / max(1.0, r.abs().max().item())).item()
        assert e <= 1e-4, f"{n}"


def _xhat(x: torch.Tensor, eps: float) -> torch.Tensor:
    xf = x.float()
    return xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)


def _check_norm_weight(dw, dw_ref, x, dn_ref, dtype, what):
    """dw = sum over rows of x^ * dy: each term carries the error of dy (the
    gradient of the normalized row, stored in the input dtype), so the bound
    per head-dim element is sum_rows |x^| * (TOL + STORAGE * max|dy|)."""
    xh = _xhat(x, 1e-6).reshape(-1, x.shape[-1]).abs().sum(0)
    bound = xh * (TOL[dtype] + STORAGE[dtype] * dn_ref.abs().max().item())
    err = (dw.cpu().float() - dw_ref.float()).abs()
    worst = (err / bound).max().item()
    print(f"{what}: max |d_w err| {err.max().item():.3e}, max |d_w| {dw_ref.abs().max().item():.3e}, "
          f"err/bound {worst:.3f}", flush=True)
    assert worst <= 1.0, f"{what}: weight gradient err {err.max().item()} over its bound"


def _check_normed_rows(got, dx_ref, x, w, dn_ref, dtype, what, eps=1e-6):
    """dx = r (g dy - x^ mean(x^ g dy)) (g = 1 + w) turns an error |d dy| <= e
    of the normalized row's gradient (e = TOL + STORAGE max|dy|: dy is held in
    the input dtype, as on the unfused path) into
    |d dx_i| <= r (|g_i| + |x^_i| mean_j |x^_j g_j|) e, plus dx's own storage
    rounding. A structural mistake (a wrong r, a dropped 1 +, a missing mean
    term) errs by the size of dx itself."""
    xf = x.float()
    r = torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)
    xh = xf * r
    g = 1.0 + w.float()
    e_dy = TOL[dtype] + STORAGE[dtype] * dn_ref.abs().max().item()
    m = (xh * g).abs().mean(-1, keepdim=True)
    bound = r * (g.abs() + xh.abs() * m) * e_dy + STORAGE[dtype] * dx_ref.abs().max().item()
    err = (got.cpu().float() - dx_ref.float()).abs()
    worst = (err / bound).max().item()
    print(f"{what}: max err {err.max().item():.3e} (max |ref| {dx_ref.abs().max().item():.3e}), "
          f"err/bound {worst:.3f}", flush=True)
    assert worst <= 1.0, f"{what}: err {err.max().item()} over its propagated bound"


def _norm_case(b, tq, tk, hq, hkv, d, dtype, *, rope, seed, varlen_lens=None):
    eps = 1e-6
    g = torch.Generator().manual_seed(seed + 100)
    wq = torch.randn(d, generator=g) * 0.3
    wk = torch.randn(d, generator=g) * 0.3
    if varlen_lens is None:
        q = _rand((b, tq, hq, d), dtype, seed)
        k = _rand((b, tk, hkv, d), dtype, seed + 1)
        v = _rand((b, tk, hkv, d), dtype, seed + 2)
        d_o = _rand((b, tq, hq, d), dtype, seed + 3, std=1.0)
        segs = [(None, None)]
        kw = dict(causal=True)
    else:
        cu = torch.tensor([0] + list(np.cumsum(varlen_lens)), dtype=torch.int32)
        tot = int(cu[-1])
        q = _rand((tot, hq, d), dtype, seed)
        k = _rand((tot, hkv, d), dtype, seed + 1)
        v = _rand((tot, hkv, d), dtype, seed + 2)
        d_o = _rand((tot, hq, d), dtype, seed + 3, std=1.0)
        segs = list(zip(cu[:-1].tolist(), cu[1:].tolist()))
        kw = dict(causal=True, cu_seqlens_q=cu.to(DEV), cu_seqlens_k=cu.to(DEV), max_seqlen_q=max(varlen_lens),
                  max_seqlen_k=max(varlen_lens))
        tq = tk = max(varlen_lens)
    kw.update(q_norm_weight=wq.to(DEV), k_norm_weight=wk.to(DEV), norm_eps=eps)
    if rope:
        cos, sin = wl.rope_tables(tk + 8, d, 10000.0)
        kw.update(rope_cos=cos.to(DEV), rope_sin=sin.to(DEV), rope_q=True, rope_k=True)
    qg, kg, vg = q.to(DEV), k.to(DEV), v.to(DEV)
    o, lse = ops.attention_prefill(qg, kg, vg, return_lse=True, **kw)
    dq, dk, dv, dwq, dwk = ops.attention_prefill_bwd(qg, kg, vg, o, lse, d_o.to(DEV), **kw)
    torch.cuda.synchronize()
    acc_wq, acc_wk = torch.zeros(d, dtype=torch.float64), torch.zeros(d, dtype=torch.float64)
    dnq_max, dnk_max = 0.0, 0.0
    for s, e in segs:
        sl = slice(s, e)
        qs, ks, vs, gs = ((x[sl][None] if s is not None else x) for x in (q, k, v, d_o))
        okw = {}
        if rope:
            n_q, n_k = qs.shape[1], ks.shape[1]
            okw["rope"] = (cos, sin, torch.arange(n_k - n_q, n_k), torch.arange(n_k))
        rq, rk, rv, rwq, rwk = ref.attention_grads(qs.float(), ks.float(), vs.float(), gs.float(), causal=True,
                                                   qk_norm=(wq, wk, eps), **okw)
        got = [x[sl][None] if s is not None else x for x in (dq, dk, dv)]
        what = f"norm d{d} {dtype} rope={rope} seg {s}:{e}"
        _check(got[2:], (rv,), dtype, what)  # _check names its first tensor dq: here it is dv
        acc_wq += rwq.double()
        acc_wk += rwk.double()
        # gradients of the normalized rows (dy of the bounds)
        dn = ref.attention_grads(ref.rms_norm(qs.float(), wq, eps), ref.rms_norm(ks.float(), wk, eps), vs.float(),
                                 gs.float(), causal=True, **okw)
        _check_normed_rows(got[0], rq, qs, wq, dn[0], dtype, what + " dq")
        _check_normed_rows(got[1], rk, ks, wk, dn[1], dtype, what + " dk")
        dnq_max, dnk_max = max(dnq_max, dn[0].abs().max().item()), max(dnk_max, dn[1].abs().max().item())
    _check_norm_weight(dwq, acc_wq, q, torch.tensor(dnq_max), dtype, f"norm d{d} {dtype} rope={rope} d_q_norm_weight")
    _check_norm_weight(dwk, acc_wk, k, torch.tensor(dnk_max), dtype, f"norm d{d} {dtype} rope={rope} d_k_norm_weight")
    return (dq, dk, dv, dwq, dwk), (qg, kg, vg, o, lse, d_o, kw)


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.bfloat16, 256),
                                     (torch.float16, 128), (torch.float32, 128), (torch.float32, 256)])
@pytest.mark.parametrize("rope", [False, True])
def test_backward_fused_qk_norm(dtype, d, rope):
    """The fused QK-RMSNorm (goda's RMSNorm before RoPE, mint/nn/attn.py:57-60)
    through the backward: dq / dk of the rows before the norm and both scales'
    gradients against the oracle's autograd."""
    _norm_case(2, 96, 96, 8, 2, d, dtype, rope=rope, seed=41)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_backward_fused_qk_norm_varlen_mqa(dtype):
    _norm_case(1, 0, 0, 6, 1, 128, dtype, rope=True, seed=43, varlen_lens=[40, 1, 75, 9])


def test_backward_fused_qk_norm_weight_gradients_are_deterministic():
    grads, (qg, kg, vg, o, lse, d_o, kw) = _norm_case(2, 300, 300, 8, 2, 128, torch.bfloat16, rope=True, seed=47)
    again = ops.attention_prefill_bwd(qg, kg, vg, o, lse, d_o.to(DEV), **kw)
    for a_, b_ in zip(grads[3:], again[3:]):
        assert torch.equal(a_, b_)


@pytest.mark.parametrize("b,t,hq,hkv", [(1, 1, 1, 1), (1, 63, 2, 1), (1, 65, 33, 1), (3, 129, 32, 8)])
@pytest.mark.parametrize("d", [64, 256])
def test_backward_fused_qk_norm_partial_sums(b, t, hq, hkv, d):
    """The rows of a norm workgroup (64) and the partials of a reduction round
    (64), one less, one more and several rounds, on both sides."""
    _norm_case(b, t, t, hq, hkv, d, torch.bfloat16, rope=False, seed=53)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,tq,tk,hq,hkv,causal,window", [
    (1, 1, 1, 1, 1, True, -1),  # one row, one key
    (1, 33, 97, 3, 1, True, -1),  # partial tiles on both sides, more keys than rows
    (2, 65, 65, 6, 2, True, -1),  # a third tile of one row, idle waves
    (1, 160, 160, 5, 5, True, 32),  # windowed
    (1, 40, 130, 4, 1, False, -1),
])
def test_backward_fp32_streamed(d, b, tq, tk, hq, hkv, causal, window):
    """fp32 at the edges of its 32-row tiles, with the walks of dk/dv and dq
    split over several waves and workgroups."""
    _case(b, tq, tk, hq, hkv, d, torch.float32, causal=causal, seed=d + tq, window=window)


def _least_workspace(plan) -> int:
    """The bytes that a refused workspace is told it needs; the plan is left
    with a workspace of just that."""
    plan.grads.workspace_bytes = 0
    with pytest.raises(Exception, match="workspace of") as e:
        plan()
    plan.grads.workspace_bytes = int(re.search(r"workspace of (\d+) bytes", str(e.value))[1])
    return plan.grads.workspace_bytes


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,tq,tk,hq,hkv,causal,window,alibi,masked", [
    (2, 97, 97, 4, 2, True, -1, False, False),
    (1, 40, 130, 6, 1, True, -1, True, False),  # the diagonal 90 keys in
    (1, 130, 40, 2, 2, True, -1, False, True),  # rows without a key
    (1, 300, 300, 3, 1, True, 0, False, False),  # one key a row: bands of two tiles
    (1, 300, 300, 2, 1, True, 1, True, False),
    (1, 290, 323, 2, 2, True, 34, False, True),
    (1, 300, 300, 2, 1, True, 290, False, False),  # a window that leaves no band
    (2, 1, 300, 4, 1, False, 70, False, False),
    (1, 70, 100, 4, 4, False, -1, True, True),
])
def test_backward_fp32_stored_and_recomputed(d, b, tq, tk, hq, hkv, causal, window, alibi, masked):
    """dq from stored dS tiles (a triangle, a window's band, or all of them) and,
    in the least workspace the call accepts, from S and dP formed again, with a
    walk of dk/dv that is not split: both within the oracle's bounds. A byte less
    is refused."""
    q, k, v, d_o = (_rand((b, t, h, d), torch.float32, s) for s, (t, h) in enumerate(((tq, hq), (tk, hkv), (tk, hkv), (tq, hq))))
    kw, okw = dict(causal=causal, window_left=window), dict(causal=causal, window_size=(window, -1))
    if alibi:
        okw["alibi_slopes"] = torch.tensor(wl.alibi_slopes(hq), dtype=torch.float32)
        kw["alibi_slopes"] = okw["alibi_slopes"].to(DEV)
    if masked:
        okw["base_attn_mask"] = torch.rand(b, 1, tq, tk, generator=torch.Generator().manual_seed(d)) < 0.8
        kw["attn_mask"] = okw["base_attn_mask"].to(DEV)
    x = [y.to(DEV) for y in (q, k, v)]
    o, lse = ops.attention_prefill(*x, return_lse=True, **kw)
    plan = ops.plan_prefill_bwd(*x, o, lse, d_o.to(DEV), **kw)
    refs = ref.attention_grads(q, k, v, d_o, **okw)
    _check(plan(), refs, torch.float32, f"stored d{d} {tq}/{tk}")
    full, least = plan.grads.workspace_bytes, _least_workspace(plan)
    assert least < full
    for y in plan.result:
        y.fill_(float("nan"))
    _check(plan(), refs, torch.float32, f"recomputed d{d} {tq}/{tk}")
    plan.grads.workspace_bytes = least - 1
    with pytest.raises(Exception, match="workspace of"):
        plan()


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("window", [-1, 20])
@pytest.mark.parametrize("same", [True, False])  # one cu_seqlens array (a triangle of dS tiles), or two
def test_backward_fp32_packed_in_a_smaller_workspace(same, window, norm):
    """Packed documents in the workspace of a smaller call than the query's
    (no dS tiles) and in the whole one: the same gradients, those of the norm
    weights among them. The two forms differ in the order of fp32 sums."""
    lens, hq, hkv, d = [70, 1, 160, 0, 33], 4, 2, 128
    n, m = sum(lens), max(lens)
    cu = torch.tensor([sum(lens[:i]) for i in range(len(lens) + 1)], dtype=torch.int32, device=DEV)
    q, k, v, d_o = (_rand((n, h, d), torch.float32, s).to(DEV) for s, h in enumerate((hq, hkv, hkv, hq)))
    kw = dict(causal=True, window_left=window, cu_seqlens_q=cu, cu_seqlens_k=cu if same else cu.clone(), max_seqlen_q=m, max_seqlen_k=m)
    if norm:
        kw.update(q_norm_weight=_rand((d,), torch.float32, 8).to(DEV), k_norm_weight=_rand((d,), torch.float32, 9).to(DEV))
    o, lse = ops.attention_prefill(q, k, v, return_lse=True, **kw)
    plan = ops.plan_prefill_bwd(q, k, v, o, lse, d_o, **kw)
    full, want = plan.grads.workspace_bytes, [y.clone() for y in plan()]
    assert _least_workspace(plan) < full
    for got, w in zip(plan(), want):
        assert (got - w).abs().max().item() <= 1e-5 * max(1.0, w.abs().max().item())


def test_backward_fp32_workspace_of_the_largest_batch_serves_smaller_ones():
    """One workspace, as the query gives it for the largest batch of a program,
    at smaller batches: the split of dk/dv's walk, which the query's size turns
    on, ends between 31 and 32 sequences, so that 31 ask for more than 32. None
    is refused, and the gradients are those of a workspace of their own (up to
    the order of fp32 sums)."""
    t, d = 1024, 64
    q, k, v, d_o = (_rand((32, t, 1, d), torch.float32, s).to(DEV) for s in range(4))
    largest, sizes = None, []
    for b in (32, 31, 5):
        o, lse = ops.attention_prefill(q[:b], k[:b], v[:b], causal=True, return_lse=True)
        plan = ops.plan_prefill_bwd(q[:b], k[:b], v[:b], o, lse, d_o[:b], causal=True)
        sizes.append(plan.grads.workspace_bytes)
        want = [y.clone() for y in plan()]
        largest = largest or plan
        plan.grads.workspace, plan.grads.workspace_bytes = largest.grads.workspace, sizes[0]
        for got, w in zip(plan(), want):
            assert (got - w).abs().max().item() <= 1e-5 * max(1.0, w.abs().max().item())
    assert sizes[1] > sizes[0] > sizes[2]


def test_backward_fp32_without_stored_ds():
    """Past 4 GiB of dS tiles the pairs of a batch run in several launches: the
    gradients of the whole batch are those of its halves, and those of the dq
    kernel that forms S and dP again, for want of room. The last two forms
    differ in the order of dq's fp32 sums and in the rounding of the exponents'
    bias terms: slopes of at most 0.707 / 64 over 4608 keys keep those under 74
    log2 units, so two roundings change a probability by 2 * 74 * 2^-24 * ln 2
    = 6.1e-6 of itself (at the slopes themselves it would be 3.9e-4), and
    gradients of at most 1 stay within 1e-4."""
    b, t, hq, d = 8, 4608, 16, 64
    g = torch.Generator(device=DEV).manual_seed(5)
    q, k, v, d_o = (torch.randn(b, t, h, d, device=DEV, generator=g) * 0.5 for h in (hq, 4, 4, hq))
    slopes = torch.tensor(wl.alibi_slopes(hq), dtype=torch.float32, device=DEV) / 64
    mask = torch.rand(b, 1, 1, t, device=DEV, generator=g) < 0.9

    def grads(rows, least=False):
        x = [y[rows].contiguous() for y in (q, k, v)]
        kw = dict(causal=False, alibi_slopes=slopes, attn_mask=mask[rows])
        o, lse = ops.attention_prefill(*x, return_lse=True, **kw)
        plan = ops.plan_prefill_bwd(*x, o, lse, d_o[rows].contiguous(), **kw)
        ws = plan.grads.workspace_bytes
        if least:
            assert _least_workspace(plan) < 1 << 30
        return plan(), ws

    whole, ws = grads(slice(0, b))
    half, ws_half = grads(slice(0, 4))
    assert ws < 8 << 30 and ws_half > 4 << 30  # (four launches, two)
    for w, h in zip(whole, grads(slice(0, 4), least=True)[0]):
        assert (w[:4] - h).abs().max().item() <= 1e-4 * max(1.0, h.abs().max().item())
    for w, h in zip(whole, half):
        assert (w[:4] - h).abs().max().item() <= 1e-4 * max(1.0, h.abs().max().item())
