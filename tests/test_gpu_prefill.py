"""Prefill parity: HIP path (through the C-ABI) vs the CPU oracle."""

from __future__ import annotations

import ctypes
import math

import pytest
import torch

from goda_amd import _lib, ops
from goda_amd import workloads as wl
from oracle import attention as ref
from tests.helpers import TOL, lse_err, max_err, report, rope_oracle, wave_block_rows

pytestmark = pytest.mark.gpu

DEV = "cuda"


def _rand(shape, dtype, seed, std=0.5):
    g = torch.Generator().manual_seed(seed)
    return (torch.randn(shape, generator=g) * std).to(dtype)


def _run_case(
    b, tq, tk, hq, hkv, d, dtype, causal, *, seed=0, window=-1, alibi=False, rope=False, layout="bthd"
):
    q = _rand((b, tq, hq, d), dtype, seed)
    k = _rand((b, tk, hkv, d), dtype, seed + 1)
    v = _rand((b, tk, hkv, d), dtype, seed + 2)
    kw = {}
    slopes = None
    cos = sin = None
    if alibi:
        slopes = torch.tensor(wl.alibi_slopes(hq), dtype=torch.float32)
        kw["alibi_slopes"] = slopes.to(DEV)
    if rope:
        cos, sin = wl.rope_tables(tk + 8, d, 10000.0)
        kw.update(rope_cos=cos.to(DEV), rope_sin=sin.to(DEV), rope_q=True, rope_k=True)
    if layout == "bhtd":
        # the reference kernel layout [B, H, T, D], passed as strided views
        qg = q.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)
        kg = k.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)
        vg = v.transpose(1, 2).contiguous().to(DEV).transpose(1, 2)
    else:
        qg, kg, vg = q.to(DEV), k.to(DEV), v.to(DEV)
    o, lse = ops.attention_prefill(qg, kg, vg, causal=causal, window_left=window, return_lse=True, **kw)
    torch.cuda.synchronize()

    qr, kr = q.float(), k.float()
    if rope:
        qr = rope_oracle(q, cos, sin, torch.arange(tk - tq, tk))
        kr = rope_oracle(k, cos, sin, torch.arange(tk))
    o_ref, lse_ref = ref.attention_rows(
        qr, kr, v.float(), torch.arange(tq), causal=causal, window_left=window, alibi_slopes=slopes
    )
    tol = TOL[dtype]
    eo = max_err(o, o_ref)
    el = lse_err(lse, lse_ref)
    assert eo <= tol, f"o max err {eo} > {tol}"
    assert el <= max(tol, 1e-3 if dtype != torch.float32 else 1e-4) * 4, f"lse max err {el}"
    return eo


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_head_dims(dtype, d, causal):
    _run_case(2, 128, 128, 8, 2, d, dtype, causal, seed=d)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("hq,hkv", [(4, 4), (8, 2), (8, 1), (6, 1), (12, 4), (6, 2), (16, 1)])
def test_prefill_gqa_groups(dtype, hq, hkv):
    _run_case(2, 96, 96, hq, hkv, 128, dtype, True, seed=hq * 10 + hkv)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("tq,tk", [(100, 100), (1, 1), (37, 150), (1, 77), (200, 333), (65, 64)])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_ragged_lengths(dtype, tq, tk, causal):
    if tq > tk and causal:
        pytest.skip("rows with no visible key are covered by test_prefill_empty_rows")
    _run_case(2, tq, tk, 8, 2, 128, dtype, causal, seed=tq + tk)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("window", [0, 5, 31, 64, 200])
def test_prefill_window(dtype, window):
    _run_case(2, 160, 160, 8, 2, 128, dtype, True, seed=window, window=window)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,hq,hkv", [(128, 8, 2), (256, 16, 1), (64, 6, 6)])
def test_prefill_alibi(dtype, d, hq, hkv):
    _run_case(2, 130, 130, hq, hkv, d, dtype, True, seed=d + hq, alibi=True)
    _run_case(1, 70, 70, hq, hkv, d, dtype, False, seed=d + hq + 1, alibi=True)


@pytest.mark.parametrize(
    "dtype,d", [(torch.bfloat16, 128), (torch.bfloat16, 256), (torch.float16, 128), (torch.float16, 256), (torch.float32, 128)]
)
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_rescale_margin(dtype, d, causal):
    """The lazy rescale's margin (P entries up to 2^14 for fp16 operands, 2^60
    for bf16/fp32): steep ALiBi slopes move every row's max by up to ~6 log2
    units per key, large-magnitude scores put entries near the margin, and
    values of std 300 stress the fp32 accumulators. Against the oracle, with
    the error relative to the values' scale. Bounds per dtype: at this scale
    the output's own rounding alone is 0.013 (bf16) / 0.0017 (fp16) of it, and
    the rounding of P adds about as much; a margin of 8 gives the same errors
    (measured 0.020-0.032 bf16, 0.0035-0.0046 fp16, <= 0.0004 fp32)."""
    b, t, hq, hkv = 1, 700, 4, 1
    q = _rand((b, t, hq, d), dtype, 71, std=2.0)
    k = _rand((b, t, hkv, d), dtype, 72, std=2.0)
    v = _rand((b, t, hkv, d), dtype, 73, std=300.0)
    slopes = torch.tensor([4.0, 1.0, 0.25, 0.0625], dtype=torch.float32)
    o, lse = ops.attention_prefill(
        q.to(DEV), k.to(DEV), v.to(DEV), causal=causal, alibi_slopes=slopes.to(DEV), return_lse=True
    )
    torch.cuda.synchronize()
    assert torch.isfinite(o.float()).all() and torch.isfinite(lse).all()
    o_ref, lse_ref = ref.attention_rows(
        q.float(), k.float(), v.float(), torch.arange(t), causal=causal, alibi_slopes=slopes
    )
    tol_o = {torch.bfloat16: 0.05, torch.float16: 0.01, torch.float32: 2e-3}[dtype]
    tol_l = {torch.bfloat16: 2e-2, torch.float16: 5e-3, torch.float32: 1e-4}[dtype]
    eo = max_err(o, o_ref) / 300.0
    assert eo <= tol_o, f"o err {eo} (relative to the values' scale)"
    # lse reaches ~2800 here (steep slopes, non-causal): compared relative to
    # max(1, |lse|), since a few fp32 ulps there are ~1e-3 absolute
    el = ((lse.cpu().float() - lse_ref).abs() / lse_ref.abs().clamp(min=1.0)).max().item()
    assert el <= tol_l, f"lse err {el} (relative)"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d", [64, 128, 256])
def test_prefill_rope(dtype, d):
    _run_case(2, 120, 120, 8, 2, d, dtype, True, seed=d + 7, rope=True)
    _run_case(1, 24, 90, 4, 1, d, dtype, True, seed=d + 8, rope=True)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_prefill_kernel_layout_strides(dtype):
    _run_case(2, 130, 130, 8, 2, 128, dtype, True, seed=5, layout="bhtd")


def test_prefill_empty_rows():
    """Lq > Lk with causal alignment: the first Lq - Lk rows see no key and
    give o = 0, lse = -inf (a documented convention)."""
    b, tq, tk, hq, hkv, d = 1, 40, 16, 4, 2, 128
    q = _rand((b, tq, hq, d), torch.bfloat16, 1)
    k = _rand((b, tk, hkv, d), torch.bfloat16, 2)
    v = _rand((b, tk, hkv, d), torch.bfloat16, 3)
    o, lse = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), causal=True, return_lse=True)
    o = o.cpu().float()
    lse = lse.cpu()
    assert torch.all(o[:, : tq - tk] == 0)
    assert torch.all(torch.isneginf(lse[:, :, : tq - tk]))
    o_ref, _ = ref.attention_rows(q.float(), k.float(), v.float(), torch.arange(tq - tk, tq), causal=True)
    assert max_err(o[:, tq - tk :], o_ref) <= 2e-2


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("d,hq,hkv", [(128, 8, 2), (256, 8, 1)])
def test_prefill_varlen(dtype, d, hq, hkv):
    lens = [1, 17, 64, 65, 130, 3]
    cu = torch.zeros(len(lens) + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(lens), 0)
    total = int(cu[-1])
    q = _rand((total, hq, d), dtype, 11)
    k = _rand((total, hkv, d), dtype, 12)
    v = _rand((total, hkv, d), dtype, 13)
    o = ops.attention_prefill(
        q.to(DEV),
        k.to(DEV),
        v.to(DEV),
        causal=True,
        cu_seqlens_q=cu.to(DEV),
        cu_seqlens_k=cu.to(DEV),
        max_seqlen_q=max(lens),
        max_seqlen_k=max(lens),
    )
    o_ref = ref.varlen_attention(q, k, v, cu, cu, causal=True)
    assert max_err(o, o_ref) <= TOL[dtype]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("d,hq,hkv", [(128, 8, 2), (256, 8, 1)])
@pytest.mark.parametrize("window", [-1, 50, 200])
def test_prefill_alibi_varlen_window(dtype, d, hq, hkv, window):
    """ALiBi walks each item's key tiles from the last down; with packed
    sequences and a left window the walk starts and ends away from tile 0.
    (fp32 at head_dim 256 streams its operands, checked the same way.)"""
    lens = [1, 37, 64, 65, 300, 129, 5]
    cu = torch.zeros(len(lens) + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(lens), 0)
    total = int(cu[-1])
    q = _rand((total, hq, d), dtype, 21)
    k = _rand((total, hkv, d), dtype, 22)
    v = _rand((total, hkv, d), dtype, 23)
    slopes = torch.tensor(wl.alibi_slopes(hq), dtype=torch.float32)
    o = ops.attention_prefill(
        q.to(DEV),
        k.to(DEV),
        v.to(DEV),
        causal=True,
        window_left=window,
        alibi_slopes=slopes.to(DEV),
        cu_seqlens_q=cu.to(DEV),
        cu_seqlens_k=cu.to(DEV),
        max_seqlen_q=max(lens),
        max_seqlen_k=max(lens),
    )
    o_ref = ref.varlen_attention(q, k, v, cu, cu, causal=True, window_left=window, alibi_slopes=slopes)
    assert max_err(o, o_ref) <= TOL[dtype]


@pytest.mark.parametrize("nseq", [40, 70])
def test_prefill_varlen_many_sequences(nseq):
    """Packed batches walk their (sequence, head) pairs longest sequence first
    when there are at most 64 sequences (ranked on the device, ties by index)
    and in index order above that; both must cover every query tile once.
    Lengths include repeats (rank ties), an empty sequence and a long one."""
    g = torch.Generator().manual_seed(nseq)
    lens = torch.randint(1, 160, (nseq,), generator=g)
    lens[3] = lens[7] = lens[11]  # ties
    lens[5] = 0
    lens[nseq - 2] = 700
    lens = lens.tolist()
    hq, hkv, d = 4, 2, 128
    cu = torch.zeros(nseq + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(lens), 0)
    total = int(cu[-1])
    q = _rand((total, hq, d), torch.bfloat16, 31)
    k = _rand((total, hkv, d), torch.bfloat16, 32)
    v = _rand((total, hkv, d), torch.bfloat16, 33)
    o = ops.attention_prefill(
        q.to(DEV), k.to(DEV), v.to(DEV), causal=True,
        cu_seqlens_q=cu.to(DEV), cu_seqlens_k=cu.to(DEV), max_seqlen_q=max(lens), max_seqlen_k=max(lens),
    )
    o_ref = ref.varlen_attention(q, k, v, cu, cu, causal=True)
    assert max_err(o, o_ref) <= TOL[torch.bfloat16]


@pytest.mark.parametrize("nseq,d,hq,hkv,maxlen", [(5, 256, 8, 1, 1500), (16, 256, 8, 1, 1300), (33, 128, 8, 2, 1700),
                                                  (64, 256, 8, 1, 700), (12, 128, 32, 8, 2100)])
def test_prefill_varlen_tail_levels(nseq, d, hq, hkv, maxlen):
    """Packed batches of at most 64 sequences deal the query tiles of their
    shortest sequences level by level at the end of each XCD's walk; every
    tile of every sequence must still be computed once. Lengths span several
    tile levels per XCD (so the level search and the per-level sequence rank
    both matter), with ties, an empty sequence and one-token sequences."""
    g = torch.Generator().manual_seed(1000 + nseq)
    lens = torch.randint(1, maxlen, (nseq,), generator=g)
    if nseq > 4:
        lens[1] = lens[2]  # a rank tie
        lens[3] = 0
        lens[4] = 1
    lens = lens.tolist()
    cu = torch.zeros(nseq + 1, dtype=torch.int32)
    cu[1:] = torch.cumsum(torch.tensor(lens), 0)
    total = int(cu[-1])
    q = _rand((total, hq, d), torch.bfloat16, 41)
    k = _rand((total, hkv, d), torch.bfloat16, 42)
    v = _rand((total, hkv, d), torch.bfloat16, 43)
    o = ops.attention_prefill(
        q.to(DEV), k.to(DEV), v.to(DEV), causal=True,
        cu_seqlens_q=cu.to(DEV), cu_seqlens_k=cu.to(DEV), max_seqlen_q=max(lens), max_seqlen_k=max(lens),
    )
    o_ref = ref.varlen_attention(q, k, v, cu, cu, causal=True)
    assert max_err(o, o_ref) <= TOL[torch.bfloat16]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_prefill_seqused_k(dtype):
    """Per-sequence key counts from the device (chunked prefill over a cache)."""
    b, tq, lmax, hq, hkv, d = 3, 20, 200, 8, 2, 128
    used = torch.tensor([20, 150, 77], dtype=torch.int32)
    q = _rand((b, tq, hq, d), dtype, 21)
    k = _rand((b, lmax, hkv, d), dtype, 22)
    v = _rand((b, lmax, hkv, d), dtype, 23)
    o = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), causal=True, seqused_k=used.to(DEV))
    for i in range(b):
        L = int(used[i])
        o_ref, _ = ref.attention_rows(
            q[i : i + 1].float(), k[i : i + 1, :L].float(), v[i : i + 1, :L].float(), torch.arange(tq), causal=True
        )
        assert max_err(o[i : i + 1], o_ref) <= TOL[dtype]


def test_prefill_softmax_scale():
    b, t, hq, hkv, d = 1, 64, 4, 2, 128
    q = _rand((b, t, hq, d), torch.bfloat16, 31)
    k = _rand((b, t, hkv, d), torch.bfloat16, 32)
    v = _rand((b, t, hkv, d), torch.bfloat16, 33)
    o = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), causal=True, softmax_scale=0.3)
    o_ref, _ = ref.attention_rows(q.float(), k.float(), v.float(), torch.arange(t), causal=True, scale=0.3)
    assert max_err(o, o_ref) <= 2e-2


def test_prefill_rejects_bad_args():
    q = torch.zeros(1, 8, 6, 128, dtype=torch.bfloat16, device=DEV)
    k = torch.zeros(1, 8, 4, 128, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(ValueError):
        ops.attention_prefill(q, k, k, causal=True)  # 6 % 4 != 0
    q2 = torch.zeros(1, 8, 4, 96, dtype=torch.bfloat16, device=DEV)
    with pytest.raises(Exception):
        ops.attention_prefill(q2, q2, q2, causal=True)  # unsupported head_dim
    with pytest.raises(ValueError):
        ops.attention_prefill(q.cpu(), k.cpu(), k.cpu(), causal=True)


# ---------------------------------------------------------------------------
# the benchmark prefill workloads (cfg1-cfg5)
# ---------------------------------------------------------------------------
def _sample_rows(t: int, n: int, seed: int) -> torch.Tensor:
    g = torch.Generator().manual_seed(seed)
    mid = torch.randint(0, t, (n,), generator=g)
    return torch.unique(torch.cat([torch.tensor([0, 1, 63, 64, t // 2, t - 2, t - 1]), mid]))


def _check_prefill_workload(w: wl.Prefill, rows_per_seq: int, seqs: list[int] | None = None, row_chunk: int = 128):
    """Every sequence (or `seqs`): the first and last row of every 32-row
    block (the rows one prefill wave owns; each workgroup's query tile is one
    or two such blocks) plus rows_per_seq sampled rows, against the oracle
    computed in chunks of row_chunk rows."""
    inp = wl.prefill_inputs(w, DEV)
    kw = {}
    if "rope_cos" in inp:
        kw.update(rope_cos=inp["rope_cos"], rope_sin=inp["rope_sin"], rope_q=True, rope_k=True)
    if "alibi_slopes" in inp:
        kw["alibi_slopes"] = inp["alibi_slopes"]
    if w.lengths is not None:
        kw.update(
            cu_seqlens_q=inp["cu_seqlens"],
            cu_seqlens_k=inp["cu_seqlens"],
            max_seqlen_q=inp["max_seqlen"],
            max_seqlen_k=inp["max_seqlen"],
        )
    o, lse = ops.attention_prefill(inp["q"], inp["k"], inp["v"], causal=w.causal, return_lse=True, **kw)
    torch.cuda.synchronize()
    tol = TOL[w.dtype]
    slopes = inp.get("alibi_slopes")
    slopes = slopes.cpu() if slopes is not None else None
    worst = 0.0
    nseq = w.batch
    for b in seqs if seqs is not None else range(nseq):
        if w.lengths is not None:
            s, e = int(inp["cu_seqlens"][b]), int(inp["cu_seqlens"][b + 1])
            qb, kb, vb = inp["q"][s:e][None], inp["k"][s:e][None], inp["v"][s:e][None]
            ob = o[s:e][None]
            lb = lse[:, s:e][None]
        else:
            qb, kb, vb = inp["q"][b : b + 1], inp["k"][b : b + 1], inp["v"][b : b + 1]
            ob, lb = o[b : b + 1], lse[b : b + 1]
        t = qb.shape[1]
        rows = torch.unique(torch.cat([wave_block_rows(t), _sample_rows(t, rows_per_seq, w.seed + b)]))
        qc, kc = qb.cpu().float(), kb.cpu().float()
        if "rope_cos" in inp:
            qc = rope_oracle(qb, inp["rope_cos"], inp["rope_sin"], torch.arange(t))
            kc = rope_oracle(kb, inp["rope_cos"], inp["rope_sin"], torch.arange(t))
        e_o = e_l = 0.0
        for c0 in range(0, len(rows), row_chunk):
            rc = rows[c0 : c0 + row_chunk]
            o_ref, lse_ref = ref.attention_rows(qc, kc, vb.cpu().float(), rc, causal=w.causal, alibi_slopes=slopes)
            e_o = max(e_o, max_err(ob[:, rc], o_ref))
            e_l = max(e_l, lse_err(lb[:, :, rc], lse_ref))
        l_bound = 5e-2 if w.dtype != torch.float32 else 1e-4
        report(w.name, "o", e_o, tol, seq=b, rows=len(rows))
        report(w.name, "lse", e_l, l_bound, seq=b, rows=len(rows))
        worst = max(worst, e_o)
        assert e_o <= tol, f"{w.name} seq {b}: o err {e_o}"
        assert e_l <= l_bound, f"{w.name} seq {b}: lse err {e_l}"
    return worst


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("d", [64, 128])
@pytest.mark.parametrize("form", ["row_pad", "base_offset"])
@pytest.mark.parametrize("causal", [True, False])
def test_prefill_v_not_16b_aligned(dtype, d, form, causal):
    """V rows that are only 8-byte aligned (a padded row stride, or a base 4
    elements into its buffer; the pre-pass reads them with 16-byte loads):
    same result, bit for bit, as an aligned V, and the oracle's."""
    b, t, hq, hkv = 2, 200, 8, 2
    q = _rand((b, t, hq, d), dtype, 31)
    k = _rand((b, t, hkv, d), dtype, 32)
    v = _rand((b, t, hkv, d), dtype, 33)
    qg, kg, vg = q.to(DEV), k.to(DEV), v.to(DEV)
    if form == "row_pad":
        buf = torch.zeros(b, t, hkv * d + 4, dtype=dtype, device=DEV)
        buf[..., : hkv * d] = vg.reshape(b, t, hkv * d)
        vu = buf[..., : hkv * d].unflatten(-1, (hkv, d))
    else:
        buf = torch.zeros(b * t * hkv * d + 4, dtype=dtype, device=DEV)
        buf[4:] = vg.reshape(-1)
        vu = buf[4:].view(b, t, hkv, d)
    assert vu.stride(-1) == 1 and (vu.data_ptr() % 16 != 0 or (vu.stride(1) * vu.element_size()) % 16 != 0)
    o_al = ops.attention_prefill(qg, kg, vg, causal=causal)
    o_un = ops.attention_prefill(qg, kg, vu, causal=causal)
    torch.cuda.synchronize()
    assert torch.equal(o_al, o_un)
    o_ref, _ = ref.attention_rows(q.float(), k.float(), v.float(), torch.arange(t), causal=causal)
    assert max_err(o_un, o_ref) <= TOL[dtype]


def test_cfg1_d12_fp32_full():
    """cfg1 at full size against the oracle's SDPA path (all rows)."""
    w = wl.CFG1
    inp = wl.prefill_inputs(w, DEV)
    o = ops.attention_prefill(
        inp["q"], inp["k"], inp["v"], causal=True, rope_cos=inp["rope_cos"], rope_sin=inp["rope_sin"], rope_q=True, rope_k=True
    )
    t = w.seqlen
    qr = rope_oracle(inp["q"], inp["rope_cos"], inp["rope_sin"], torch.arange(t))
    kr = rope_oracle(inp["k"], inp["rope_cos"], inp["rope_sin"], torch.arange(t))
    o_ref = ref.attention(qr, kr, inp["v"].cpu(), causal=True)
    assert max_err(o, o_ref) <= 1e-4


def test_cfg2_gqa_prefill_block_rows():
    _check_prefill_workload(wl.CFG2, rows_per_seq=24)


def test_cfg3_mqa_alibi_block_rows():
    _check_prefill_workload(wl.CFG3, rows_per_seq=24)


def test_cfg5_varlen_prefill_block_rows():
    _check_prefill_workload(wl.CFG5.prefill, rows_per_seq=16)


@pytest.mark.parametrize("d", [64, 128, 256])
@pytest.mark.parametrize("b,tq,tk,hq,hkv,causal,window", [
    (1, 1, 1, 1, 1, True, -1),  # one row, one key
    (1, 31, 97, 3, 1, True, -1),  # a partial query tile over a partial fourth key tile
    (2, 33, 33, 6, 2, True, -1),  # two query tiles, idle rows
    (1, 160, 160, 5, 5, True, 32),  # windowed: two key tiles a query tile
    (1, 70, 200, 4, 1, False, -1),
    (1, 96, 40, 2, 1, True, -1),  # rows without a key
    (2, 2081, 2081, 24, 8, True, -1),  # more than 3072 items: the LDS ring at D <= 128
])
def test_prefill_fp32_streamed(d, b, tq, tk, hq, hkv, causal, window):
    """fp32 on streamed operands: the edges of its 32-row tiles, each way of
    splitting an item's keys over a workgroup's waves, and both sides of the
    rule that chooses it."""
    rope = tq <= tk
    if tq > 2048:
        _run_rows(b, tq, tk, hq, hkv, d, causal)
    else:
        _run_case(b, tq, tk, hq, hkv, d, torch.float32, causal, seed=d + tq, window=window, rope=rope)


def _run_rows(b, tq, tk, hq, hkv, d, causal):
    """fp32 parity on the first and last row of every query tile."""
    q, k, v = _rand((b, tq, hq, d), torch.float32, 1), _rand((b, tk, hkv, d), torch.float32, 2), _rand((b, tk, hkv, d), torch.float32, 3)
    o = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), causal=causal)
    rows = wave_block_rows(tq)
    o_ref, _ = ref.attention_rows(q, k, v, rows, causal=causal)
    assert max_err(o[:, rows.to(DEV)], o_ref) <= TOL[torch.float32]


@pytest.mark.parametrize("d,b,tq,tk,hq,hkv", [
    (64, 1, 1024, 1024, 64, 16),  # full attention in one whole round of the ring's workgroups
    (128, 1, 1024, 1024, 64, 16),
    (128, 1, 1000, 1050, 56, 14),  # one that is not whole: streamed
    (256, 128, 40, 70, 4, 4),  # few rows of heads with keys of their own, a whole round: the vector ALUs
    (256, 8, 64, 900, 64, 64),
    (256, 8, 65, 200, 64, 64),  # more rows, a longer walk, a round that is not whole: streamed
    (256, 8, 64, 1024, 64, 64),
    (256, 5, 40, 70, 64, 64),
    (256, 128, 20, 70, 4, 4),  # 512 tiles of rows: walks shared by the waves
])
def test_prefill_fp32_rounds_of_equal_work(d, b, tq, tk, hq, hkv):
    """Both sides of the rules for calls that fill the GPU in whole rounds; a
    workspace is asked for unless the vector ALUs take the call."""
    _run_rows(b, tq, tk, hq, hkv, d, False)
    q, k = torch.empty(b, tq, hq, d, device=DEV), torch.empty(b, tk, hkv, d, device=DEV)
    size = ops.plan_prefill(q, k, k, causal=False).args.workspace_bytes
    vector = d == 256 and 32 < tq <= 64 and tk < 1024 and b * hq == 512
    assert (size == 0) == vector


@pytest.mark.parametrize("tk", [64, 65, 200])
def test_prefill_fp32_wide_without_workspace(tk):
    """fp32 at head_dim 256: a call without a workspace gives the same result
    (on the vector ALUs) as one with the workspace that the query asks for."""
    q, k, v = _rand((2, tk, 4, 256), torch.float32, 1).to(DEV), _rand((2, tk, 2, 256), torch.float32, 2).to(DEV), _rand((2, tk, 2, 256), torch.float32, 3).to(DEV)
    plan = ops.plan_prefill(q, k, v, causal=True)
    want = plan().clone()
    plan.args.workspace, plan.args.workspace_bytes = None, 0
    plan.result.zero_()
    got = plan()
    torch.cuda.synchronize()
    assert (_lib.load().goda_attn_prefill_workspace_size(ctypes.byref(plan.args)) > 0) == (tk > 64)
    assert max_err(got, want) <= 1e-5


@pytest.mark.parametrize("tk", [64, 96, 2048])
def test_prefill_fp32_wide_large_values(tk):
    """fp32 at head_dim 256: values of 1e30 under scores that grow by up to 40
    (58 log2 units) along the keys stay finite, whichever kernel runs: no
    probability passes 1, so that an output is at most the largest value. Two
    roundings of a score of 58 log2 units change a probability by 2 * 58 * 2^-24
    * ln 2 = 4.8e-6 of itself, the bound is twice that."""
    d = 256
    q, v = torch.zeros(1, 4, 2, d), _rand((1, tk, 2, d), torch.float32, 3) * 1e30
    k = torch.zeros(1, tk, 2, d)
    q[..., 0] = 1.0
    k[..., 0] = torch.linspace(0.0, 40.0, tk)[None, :, None]
    o = ops.attention_prefill(q.to(DEV), k.to(DEV), v.to(DEV), causal=False, softmax_scale=1.0)
    want = ref.attention(q.double(), k.double(), v.double(), causal=False, scale=1.0, dtype=torch.float64)
    assert (o.cpu().double() - want).abs().max().item() <= 1e-5 * v.abs().max().item()


@pytest.mark.parametrize("dtype,d", [(torch.bfloat16, 64), (torch.bfloat16, 128), (torch.float16, 256)])
@pytest.mark.parametrize("b,tq,tk,hq,hkv,causal,window,alibi", [
    (1, 1500, 1500, 4, 2, True, -1, False),  # few items of unequal length
    (2, 70, 2100, 8, 2, True, -1, True),  # a chunk behind a prefix, ALiBi's downward walk
    (1, 1, 3000, 2, 1, True, 1700, False),  # one row, a window over several pieces
    (1, 40, 1337, 3, 1, False, -1, False),
    (1, 300, 1100, 6, 6, True, 40, False),  # windowed: too short to cut
])
def test_prefill_split_keys(dtype, d, b, tq, tk, hq, hkv, causal, window, alibi):
    """Batches of few items, whose keys are cut into pieces added up by a second
    launch; the workspace has room for them."""
    q, k = torch.empty(b, tq, hq, d, dtype=dtype, device=DEV), torch.empty(b, tk, hkv, d, dtype=dtype, device=DEV)
    plan = ops.plan_prefill(q, k, k, causal=causal, window_left=window)
    tile = 64 if d <= 128 else 32
    images = 2 * b * (-(-tk // tile) * tile) * hkv * d * 2
    assert (plan.args.workspace_bytes > images) == (window != 40)
    _run_case(b, tq, tk, hq, hkv, d, dtype, causal, seed=tq, window=window, alibi=alibi, rope=not alibi)


@pytest.mark.parametrize("dtype,d,hq,hkv", [(torch.bfloat16, 128, 8, 2), (torch.float16, 64, 4, 4), (torch.bfloat16, 256, 8, 1)])
@pytest.mark.parametrize("lens", [[1500, 3, 700, 0, 1499], [2000], [40, 40, 40], [1025] + [17] * 69])
def test_prefill_split_keys_lengths_on_the_device(dtype, d, hq, hkv, lens):
    """Key counts read on the device: sequences cut into several pieces, one, or
    none, and an empty one; rows with no key give 0. 70 sequences are too many
    items to cut, whatever their lengths."""
    b, tq, tk = len(lens), 33, 2048
    q, k, v = _rand((b, tq, hq, d), dtype, 1), _rand((b, tk, hkv, d), dtype, 2), _rand((b, tk, hkv, d), dtype, 3)
    used = torch.tensor(lens, dtype=torch.int32)
    plan = ops.plan_prefill(q.to(DEV), k.to(DEV), v.to(DEV), causal=True, seqused_k=used.to(DEV), return_lse=True)
    images = 2 * b * tk * hkv * d * 2
    assert (plan.args.workspace_bytes > images) == (b <= 5)  # (cut, where a length asks for it)
    o, lse = plan()
    for i, n in enumerate(lens):
        first = max(0, tq - n)  # bottom-right: these rows see no key
        assert torch.count_nonzero(o[i, :first]) == 0 and bool(torch.isneginf(lse[i, :, :first]).all())
        if n == 0:
            continue
        rows = torch.arange(first, tq)
        o_ref, lse_ref = ref.attention_rows(q[i : i + 1].float(), k[i : i + 1, :n].float(), v[i : i + 1, :n].float(), rows, causal=True)
        assert max_err(o[i : i + 1, first:], o_ref) <= TOL[dtype]
        assert lse_err(lse[i : i + 1, :, first:], lse_ref) <= 5e-3


@pytest.mark.parametrize("d", [64, 128, 256])
def test_prefill_split_keys_with_room_for_the_images_alone(d):
    """A workspace without room for the pieces' sums: the items are not cut, and
    the call gives the same result. One that is too small for the tile images
    stays refused."""
    q, k, v = (_rand((1, t, h, d), torch.bfloat16, s).to(DEV) for t, h, s in ((40, 8, 1), (4096, 2, 2), (4096, 2, 3)))
    plan = ops.plan_prefill(q, k, v, causal=True)
    want = plan().clone()
    images = 2 * 4096 * 2 * d * 2
    assert plan.args.workspace_bytes > images  # (cut)
    plan.args.workspace_bytes = images
    plan.result.zero_()
    got = plan()
    torch.cuda.synchronize()
    assert max_err(got, want) <= TOL[torch.bfloat16]
    plan.args.workspace_bytes = images - 1
    with pytest.raises(Exception, match="workspace"):
        plan()


@pytest.mark.parametrize("dtype,d,hq,hkv", [(torch.float16, 64, 4, 4), (torch.bfloat16, 128, 8, 2), (torch.bfloat16, 256, 8, 1)])
@pytest.mark.parametrize("tiles", [1, 2, 3, 4, 8, 9, 16, 17])  # query tiles of the longest sequence
@pytest.mark.parametrize("batch", [1, 5, 8, 65, 72])  # over 64: no ranks; 8, 72: pairs for grids of 1, 2 and 4 tiles
def test_packed_short_sequences_cover_every_tile(dtype, d, hq, hkv, tiles, batch):
    """Packed launches whose query tiles are turned over the XCDs (up to 16 a
    sequence), grids of 1, 2 and 4 tiles a pair among them, and the next size:
    every row of every sequence against a launch of that sequence alone (the
    same sums in the same order, or cut along the keys: one rounding of the
    output apart)."""
    group = hq // hkv
    rows = 8 // min(group, 8) * 32
    longest = rows * (tiles - 1) + 1
    lens = [longest] + [(7 * i * i + 3) % longest + (0 if i % 4 == 3 else 1) for i in range(1, batch)]
    n = sum(lens)
    q, k, v = _rand((n, hq, d), dtype, 1).to(DEV), _rand((n, hkv, d), dtype, 2).to(DEV), _rand((n, hkv, d), dtype, 3).to(DEV)
    starts = [sum(lens[:i]) for i in range(batch + 1)]
    cu = torch.tensor(starts, dtype=torch.int32, device=DEV)
    o = ops.attention_prefill(q, k, v, causal=True, cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=longest, max_seqlen_k=longest)
    for i in range(batch):
        if lens[i] == 0:
            continue
        s = slice(starts[i], starts[i + 1])
        alone = ops.attention_prefill(q[None, s], k[None, s], v[None, s], causal=True)[0]
        assert max_err(o[s], alone) <= TOL[dtype]
