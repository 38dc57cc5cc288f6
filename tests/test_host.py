"""CPU tests of the host-side logic of the drop-in layer and the workload
definitions (no GPU work)."""

from __future__ import annotations

import math

import pytest
import torch

from goda_amd import autograd, ops
from goda_amd import workloads as wl
from goda_amd.mint.kvcache import KVCache
from goda_amd.mint.nn import FlashAttention, GroupedQueryAttention, LinearScaledRoPE, RoPE, alibi_slopes
from goda_amd.mint.nn.flashattn import _bool_base_mask, _segments
from oracle import attention as ref


def test_alibi_slopes_match_oracle():
    for n in (1, 2, 3, 6, 8, 12, 16, 32):
        assert alibi_slopes(n) == ref.alibi_slopes(n) == wl.alibi_slopes(n)


def test_rope_tables_match_oracle():
    r = RoPE(seq_len=300, head_dim=128, rope_base_theta=10000)
    cos, sin = ref.rope_tables(300, 128, 10000.0)
    assert torch.equal(r.cos, cos) and torch.equal(r.sin, sin)
    c2, s2 = wl.rope_tables(300, 128, 10000.0)
    assert torch.equal(c2, cos) and torch.equal(s2, sin)
    rl = LinearScaledRoPE(seq_len=64, head_dim=64, scale_factor=4.0, rope_base_theta=10000)
    cl, sl = ref.rope_tables(64, 64, 10000.0, scale_factor=4.0)
    assert torch.equal(rl.cos, cl) and torch.equal(rl.sin, sl)


def test_rope_forward_matches_oracle():
    r = RoPE(seq_len=64, head_dim=32, rope_base_theta=10000)
    g = torch.Generator().manual_seed(0)
    q = torch.randn(2, 10, 3, 32, generator=g)
    k = torch.randn(2, 10, 1, 32, generator=g)
    q2, k2, bias = r(q, k, start_pos=7)
    pos = torch.arange(7, 17)
    assert bias is None
    assert torch.allclose(q2, ref.apply_rope(q, r.cos, r.sin, pos), atol=1e-6)
    assert torch.allclose(k2, ref.apply_rope(k, r.cos, r.sin, pos), atol=1e-6)


def test_segments_match_oracle():
    doc = torch.tensor([[0, 0, 1, 1, 1, 2], [7, 7, 7, 7, 8, 8], [3, 3, 3, 3, 3, 3]])
    cu, mx, one_run = _segments(doc)
    assert cu.tolist() == ref.doc_ids_to_cu_seqlens(doc).tolist() == [0, 2, 5, 6, 10, 12, 18]
    assert mx == 6 and one_run


def test_segments_flag_ids_that_recur_in_a_row():
    """An id in two separate runs of one row (goda masks by id equality over
    the whole row) is flagged, so the dispatcher takes the dense mask; the
    same id in two different rows is not a recurrence."""
    _, _, one_run = _segments(torch.tensor([[0, 0, 1, 1, 0, 0], [2, 2, 2, 3, 3, 3]]))
    assert not one_run
    _, _, one_run = _segments(torch.tensor([[5, 5, 6, 6, 6, 6], [5, 5, 5, 6, 6, 6]]))
    assert one_run


def test_float_base_mask_follows_the_reference():
    """mint/nn/flashattn.py:236-255: a float (additive) mask reaches SDPA only
    without causal and doc_ids; with either the reference's '&' raises."""
    m = torch.tensor([[0.0, float("-inf")], [0.0, 0.0]])
    out = _bool_base_mask(m, causal=False, doc_ids=None)
    assert out.dtype == torch.bool and out.tolist() == [[True, False], [True, True]]
    with pytest.raises(TypeError):
        _bool_base_mask(m, causal=True, doc_ids=None)
    with pytest.raises(TypeError):
        _bool_base_mask(m, causal=False, doc_ids=torch.zeros(1, 2, dtype=torch.long))
    with pytest.raises(ValueError):
        _bool_base_mask(torch.tensor([[0.0, -1.5]]), causal=False, doc_ids=None)
    b = torch.tensor([[True, False]])
    assert _bool_base_mask(b, causal=True, doc_ids=None) is b


def test_pack_mask_key_size_rule():
    """The key dimension is Lk or 1 (SDPA's broadcast rule); a shorter one is
    only for KV-cache launches sized past the keys the mask names, where the
    missing keys are hidden."""
    m = torch.ones(1, 1, 3, 5, dtype=torch.bool)
    with pytest.raises(ValueError):
        ops.pack_mask(m, 1, 2, 3, 7, "cpu")
    pm = ops.pack_mask(m, 1, 2, 3, 7, "cpu", allow_short_keys=True)
    assert int(pm.bits.view(torch.uint8)[0, 0, 0, 0]) == 0b11111  # keys 5, 6 hidden
    pm1 = ops.pack_mask(torch.ones(1, 1, 3, 1, dtype=torch.bool), 1, 2, 3, 7, "cpu")
    assert int(pm1.bits.view(torch.uint8)[0, 0, 0, 0]) == 0b1111111


def test_flop_and_byte_counts_closed_form():
    w = wl.CFG2
    assert wl.prefill_flops(w) == 4 * 128 * 32 * 4 * 8192 * 8193 / 2
    lens = torch.tensor([1024, 2048], dtype=torch.int32)
    w4 = wl.Decode("t", torch.bfloat16, 2, 32, 8, 128, 4096, (1, 1))
    assert wl.decode_bytes(w4, lens) == (1024 + 2048) * 8 * 128 * 2 * 2 + 2 * 32 * 128 * 2 * 2
    nc = wl.Prefill("nc", torch.bfloat16, 2, 10, 4, 1, 64, causal=False)
    assert wl.prefill_flops(nc) == 4 * 64 * 4 * 2 * 100


def test_workload_seeds_are_deterministic():
    a = wl.prefill_inputs(wl.Prefill("t", torch.bfloat16, 1, 16, 2, 1, 64, seed=3), "cpu")
    b = wl.prefill_inputs(wl.Prefill("t", torch.bfloat16, 1, 16, 2, 1, 64, seed=3), "cpu")
    assert torch.equal(a["q"], b["q"]) and torch.equal(a["v"], b["v"])
    lens = wl.seq_lengths(1024, 32768, 64, 405)
    assert lens.min() >= 1024 and lens.max() <= 32768 and lens.dtype == torch.int32


def test_flashattention_refuses_cpu_tensors():
    """No CPU path: a base mask and a right window are accepted (the right
    window ignored, as in the reference's SDPA branch) and still reach the
    GPU-only kernels, which refuse CPU tensors."""
    fa = FlashAttention()
    q = torch.zeros(1, 4, 2, 64)
    with pytest.raises(ValueError, match="GPU tensor"):
        fa(q, q, q, causal=True)
    with pytest.raises(ValueError, match="GPU tensor"):
        fa(q, q, q, causal=True, base_attn_mask=torch.ones(1, 1, 4, 4, dtype=torch.bool))
    with pytest.raises(ValueError, match="GPU tensor"):
        fa(q, q, q, causal=True, window_size=(2, 2))


@pytest.mark.parametrize("shape", [(3, 1, 1, 70), (3, 1, 5, 70), (3, 4, 5, 70), (5, 70), (3, 1, 5, 1), (70,)])
def test_pack_mask_bits_match_the_boolean_mask(shape):
    """ops.pack_mask (torch ops, runs on the CPU too): bit j % 32 of word
    j // 32 of row (b, h, i) is the mask at key j; broadcast dimensions get a
    zero stride; with allow_short_keys (KV-cache launches) keys past the
    mask's own key count read as hidden."""
    b, hq, tq, tk = 3, 4, 5, 70
    g = torch.Generator().manual_seed(1)
    m = torch.rand(shape, generator=g) < 0.5
    pm = ops.pack_mask(m, b, hq, tq, tk + 10, "cpu", allow_short_keys=True)
    assert pm.bits.dtype == torch.int32 and pm.bits.shape[-1] == 2 * ((tk + 10 + 63) // 64)
    full = m
    while full.dim() < 4:
        full = full.unsqueeze(0)
    full = full.expand(b, hq, tq, full.shape[-1] if full.shape[-1] != 1 else tk + 10)
    words = pm.bits.reshape(-1).to(torch.int64) & 0xFFFFFFFF
    for bb in range(b):
        for h in range(hq):
            for i in range(tq):
                base = bb * pm.stride_b + h * pm.stride_h + i * pm.stride_q
                for j in range(tk + 10):
                    bit = bool((int(words[base + j // 32]) >> (j % 32)) & 1)
                    want = bool(full[bb, h, i, j]) if j < full.shape[-1] else False
                    assert bit == want, (bb, h, i, j)


def test_pack_mask_rejects_non_boolean_and_bad_shapes():
    with pytest.raises(ValueError, match="boolean"):
        ops.pack_mask(torch.zeros(1, 1, 4, 4), 1, 2, 4, 4, "cpu")
    with pytest.raises(ValueError, match="broadcast"):
        ops.pack_mask(torch.ones(2, 1, 4, 4, dtype=torch.bool), 3, 2, 4, 4, "cpu")
    with pytest.raises(ValueError, match="keys"):
        ops.pack_mask(torch.ones(1, 1, 4, 9, dtype=torch.bool), 1, 2, 4, 8, "cpu")


def test_kvcache_host_bound_rejects_overflow_before_any_launch():
    """An append past max_seq_len fails on the host while the lengths are
    known there (as the reference's slice assignment fails,
    mint/kvcache/base.py:40-43), before any kernel is called."""
    kv = KVCache(max_batch_size=2, max_seq_len=8, n_kv_heads=1, head_dim=64, dtype=torch.bfloat16, device="cpu")
    k = torch.zeros(2, 9, 1, 64, dtype=torch.bfloat16)
    with pytest.raises(ValueError, match="max_seq_len"):
        kv.append(k, k)
    assert kv.len_bound == 0
    kv.get_cache_tensors()  # the caller could now change the lengths
    assert kv.len_bound is None
    kv.reset()
    assert kv.len_bound == 0


def test_head_dim_padding_helpers():
    """goda_amd.headdim: the padded size, zero padding, and the torch RoPE
    used for head dims without kernels (against the oracle's rotation)."""
    from goda_amd import headdim

    assert [headdim.padded(d) for d in (8, 32, 64, 80, 96, 128, 160, 256)] == [64, 64, 64, 128, 128, 128, 256, 256]
    with pytest.raises(ValueError):
        headdim.padded(320)
    x = torch.randn(2, 5, 3, 96)
    xp = headdim.pad(x, 128)
    assert xp.shape[-1] == 128 and torch.equal(xp[..., :96], x) and torch.all(xp[..., 96:] == 0)
    cos, sin = ref.rope_tables(40, 96, 10000.0)
    pos = torch.arange(7, 12)
    assert torch.allclose(headdim.rotate(x, cos, sin, pos), ref.apply_rope(x, cos, sin, pos), atol=1e-6)
    # per-sequence positions [B, T]
    pb = torch.stack([pos, pos + 3])
    r = headdim.rotate(x, cos, sin, pb)
    assert torch.allclose(r[1], ref.apply_rope(x[1:2], cos, sin, pos + 3)[0], atol=1e-6)


def test_packed_row_rope_at_a_padded_head_dim(monkeypatch):
    """rope_packed_rows at a head dim without kernels: q and k rotate at their
    packed row index modulo the table length (not at the document's position)
    before the padding, and no RoPE option goes on to the kernels."""
    seen = {}

    def capture(q, k, v, **kw):
        seen.update(kw, q=q, k=k)
        return torch.zeros_like(q)

    monkeypatch.setattr(ops, "attention_prefill", capture)
    d, n, row = 96, 140, 70
    g = torch.Generator().manual_seed(5)
    q, k, v = torch.randn(n, 4, d, generator=g), torch.randn(n, 2, d, generator=g), torch.randn(n, 2, d, generator=g)
    cos, sin = ref.rope_tables(row, d, 10000.0)
    cu = torch.tensor([0, 33, 70, 140], dtype=torch.int32)
    kw = dict(causal=True, rope_cos=cos, rope_sin=sin, rope_q=True, rope_k=True, rope_packed_rows=True)
    autograd.attention_prefill(q, k, v, cu_seqlens_q=cu, cu_seqlens_k=cu, max_seqlen_q=70, max_seqlen_k=70, **kw)
    pos = torch.arange(n) % row
    assert torch.allclose(seen["q"][..., :d], ref.apply_rope(q[None], cos, sin, pos)[0], atol=1e-6)
    assert torch.allclose(seen["k"][..., :d], ref.apply_rope(k[None], cos, sin, pos)[0], atol=1e-6)
    assert not any(name.startswith("rope") for name in seen)
    with pytest.raises(ValueError, match="packed rows"):
        autograd.attention_prefill(q[None], k[None], v[None], **kw)


def test_documents_rope_tables_that_receive_gradients(monkeypatch):
    """Packed documents under RoPE tables that require grad: the rotation is a
    torch op (after the QK-norm), so that the tables get their gradients; one
    position for every row is broadcast; other calls leave both to the kernels."""
    seen = {}

    def capture(q, k, v, **kw):
        seen.clear()
        seen.update(kw)
        return q

    monkeypatch.setattr(autograd, "attention_prefill", capture)
    b, t, h, d = 2, 70, 2, 64
    g = torch.Generator().manual_seed(3)
    q = torch.randn(b, t, h, d, generator=g)
    w = torch.randn(d, generator=g) * 0.1
    docs = (torch.arange(t) // 30).expand(b, t)
    cos, sin = (x.requires_grad_(True) for x in ref.rope_tables(t, d, 10000.0))
    fa = FlashAttention()
    o = fa(q, q, q, causal=True, doc_ids=docs, rope=(cos, sin), qk_norm=(w, w, 1e-6))
    assert "rope_cos" not in seen and "q_norm_weight" not in seen
    n = ref.rms_norm(q, w)
    assert torch.allclose(o, ref.apply_rope(n, cos, sin, torch.arange(t)), atol=1e-5)
    o.sum().backward()
    # d/dcos of x1 cos - x2 sin and x1 sin + x2 cos, summed: x1 + x2
    assert torch.allclose(cos.grad, (n[..., : d // 2] + n[..., d // 2 :]).sum((0, 2)), atol=1e-4)
    assert sin.grad is not None
    with torch.no_grad():
        fa(q, q, q, causal=True, doc_ids=docs, rope=(cos, sin), qk_norm=(w, w, 1e-6))
        assert seen["rope_packed_rows"] and "q_norm_weight" in seen
        one = fa(q, q, q, causal=True, doc_ids=docs, rope=(cos[:1], sin[:1]))
    assert "rope_cos" not in seen and torch.equal(one, q)  # (position 0: the identity)


def test_documents_call_hooked_norm_modules():
    """Packed documents under grad: q_norm / k_norm modules that carry hooks are
    called; without hooks the norm is left to the kernels."""
    t, d = 12, 64
    layer = GroupedQueryAttention(2, 1, d, 32, RoPE(seq_len=t, head_dim=d, rope_base_theta=10000), torch.float32)
    seen = {}

    class Stub(torch.nn.Module):
        def forward(self, q, k, v, **kw):
            seen.clear()
            seen.update(kw)
            return q

    layer.attention = Stub()
    x = torch.randn(1, t, 32)
    docs = torch.zeros(1, t, dtype=torch.long)
    layer(x, doc_ids=docs)
    assert "qk_norm" in seen
    calls = []
    layer.k_norm.register_forward_hook(lambda *a: calls.append("fwd"))
    layer.q_norm.register_full_backward_hook(lambda *a: calls.append("bwd"))
    layer(x, doc_ids=docs).sum().backward()
    assert "qk_norm" not in seen and sorted(calls) == ["bwd", "fwd"]
