"""Chunked causal GQA attention (decode split-K, prefill MFMA, generic) vs the oracle."""
import ctypes as C
from pathlib import Path

import numpy as np
import pytest
import torch

from oracle import attention as att
from oracle import rope
from oracle.bf16 import round_bf16
from tests.gpu_util import bf16_dev, rel_err, to_np_f32

pytestmark = pytest.mark.gpu
ROOT = Path(__file__).resolve().parent.parent
TOL_F32 = 1e-3
TOL_BF16 = 2e-2


def _t(a, dev):
    return torch.from_numpy(np.ascontiguousarray(a)).to(dev)


# ---- the reference's own cases (tests/test_mlx_attention.py:53-137), generic kernel (D=6/4)
def test_reference_cases(dev):
    from lokahi_amd import ops
    rng = np.random.default_rng(0)
    q = rng.standard_normal((1, 4, 7, 6), dtype=np.float32)
    k = rng.standard_normal((1, 2, 9, 6), dtype=np.float32)
    v = rng.standard_normal((1, 2, 9, 6), dtype=np.float32)
    out = ops.attention_no_mask(_t(q, dev), _t(k, dev), _t(v, dev), q_block_size=3, k_block_size=4)
    assert np.allclose(att.naive_gqa(q, k, v), out.cpu().numpy(), atol=1e-5, rtol=1e-5)
    q = rng.standard_normal((2, 4, 7, 6), dtype=np.float32)
    k = rng.standard_normal((2, 2, 7, 6), dtype=np.float32)
    v = rng.standard_normal((2, 2, 7, 6), dtype=np.float32)
    pos = np.broadcast_to(np.arange(7), (2, 7))
    out = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev), query_positions=_t(pos, dev),
                        q_block_size=3, k_block_size=2)
    assert np.allclose(att.naive_gqa(q, k, v, pos), out.cpu().numpy(), atol=1e-5, rtol=1e-5)
    q = rng.standard_normal((1, 4, 1, 6), dtype=np.float32)
    k = rng.standard_normal((1, 2, 6, 6), dtype=np.float32)
    v = rng.standard_normal((1, 2, 6, 6), dtype=np.float32)
    out = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev), query_positions=[[5]])
    assert np.allclose(att.naive_gqa(q, k, v, np.array([[5]])), out.cpu().numpy(), atol=1e-5)
    q = rng.standard_normal((1, 2, 5, 4), dtype=np.float32)
    k = rng.standard_normal((1, 1, 5, 4), dtype=np.float32)
    v = rng.standard_normal((1, 1, 5, 4), dtype=np.float32)
    v2 = v.copy()
    v2[:, :, 3:] += 1000.0
    a = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev), k_block_size=2).cpu().numpy()
    b = ops.attention(_t(q, dev), _t(k, dev), _t(v2, dev), k_block_size=2).cpu().numpy()
    assert np.allclose(a[:, :, :3], b[:, :, :3]) and not np.allclose(a[:, :, 3:], b[:, :, 3:])
    with pytest.raises(ValueError, match="divisible"):
        ops.attention(torch.ones((1, 3, 2, 4), device=dev), torch.ones((1, 2, 2, 4), device=dev),
                      torch.ones((1, 2, 2, 4), device=dev))
    with pytest.raises(ValueError, match="key length >= query length"):
        ops.attention(torch.ones((1, 2, 3, 4), device=dev), torch.ones((1, 2, 2, 4), device=dev),
                      torch.ones((1, 2, 2, 4), device=dev))


def test_config1_chunked_gqa_rope_fp32_prefill_then_decode(dev):
    """B1, Hq8/Hkv2, D64, L512, chunks 128, theta 1e4, fp32."""
    from lokahi_amd import ops
    rng = np.random.default_rng(2024)
    B, Hq, Hkv, D, L = 1, 8, 2, 64, 512
    q = rng.normal(size=(B, Hq, L + 1, D)).astype(np.float32)
    k = rng.normal(size=(B, Hkv, L + 1, D)).astype(np.float32)
    v = rng.normal(size=(B, Hkv, L + 1, D)).astype(np.float32)
    pos = np.arange(L + 1)[None]
    c, s = rope.cos_sin(pos, D, 10000.0)
    qr, kr = rope.apply(q, c, s), rope.apply(k, c, s)
    tq, tk = _t(q, dev), _t(k, dev)
    ops.rope(tq, tk, _t(pos, dev), 10000.0)
    assert np.array_equal(tq.cpu().numpy(), qr) and np.array_equal(tk.cpu().numpy(), kr)
    tv = _t(v, dev)
    pre = ops.attention(tq[:, :, :L].contiguous(), tk[:, :, :L].contiguous(), tv[:, :, :L].contiguous(),
                        query_positions=_t(pos[:, :L], dev), q_block_size=128, k_block_size=128)
    ref = att.chunked_gqa(qr[:, :, :L], kr[:, :, :L], v[:, :, :L], pos[:, :L], True, 128, 128)
    assert rel_err(pre.cpu().numpy(), ref) < TOL_F32
    np.testing.assert_allclose(ref, att.naive_gqa(qr[:, :, :L], kr[:, :, :L], v[:, :, :L], pos[:, :L]),
                               atol=1e-4)
    dec = ops.attention(tq[:, :, L:].contiguous(), tk, tv, query_positions=[[L]])
    ref_d = att.chunked_gqa(qr[:, :, L:], kr, v, np.array([[L]]), True, 128, 128)
    assert rel_err(dec.cpu().numpy(), ref_d) < TOL_F32


def _c_decode(q, k, v):
    lib = C.CDLL(str(ROOT / "oracle" / "libstrata_oracle.so"))
    B, Hq, _, D = q.shape
    _, Hkv, L, _ = k.shape
    out = np.zeros((B, Hq, D), np.float32)
    P = C.c_void_p
    qf = np.ascontiguousarray(q.reshape(B, Hq, D), np.float32)
    lib.oracle_decode_attn(qf.ctypes.data_as(P), k.ctypes.data_as(P), v.ctypes.data_as(P), B, Hq,
                           Hkv, L, D, out.ctypes.data_as(P))
    return out.reshape(B, Hq, 1, D)


@pytest.mark.parametrize("B,L", [(1, 1024), (1, 8192), (16, 1024), (1, 32768), (16, 8192),
                                 (16, 32768)])
def test_config3_cached_decode_bf16(dev, B, L):
    """Hq32/Hkv8, D128, bf16 KV cache; append one token, then attend."""
    from types import SimpleNamespace
    from lokahi_amd import ops
    from lokahi_amd.kvcache import HipKVCache
    Hq, Hkv, D = 32, 8, 128
    g = torch.Generator(device=dev).manual_seed(B * 100000 + L)
    cfg = SimpleNamespace(num_hidden_layers=1, num_key_value_heads=Hkv, num_attention_heads=Hq,
                          hidden_size=Hq * D)
    cache = HipKVCache(cfg, batch_size=B, max_length=L + 1, dtype=torch.bfloat16)
    ctx_k = torch.randn((B, Hkv, L, D), generator=g, device=dev).to(torch.bfloat16)
    ctx_v = torch.randn((B, Hkv, L, D), generator=g, device=dev).to(torch.bfloat16)
    cache.update(ctx_k, ctx_v, 0)
    qn = torch.randn((B, 1, Hq * D), generator=g, device=dev).to(torch.bfloat16)
    kn = torch.randn((B, 1, Hkv * D), generator=g, device=dev).to(torch.bfloat16)
    vn = torch.randn((B, 1, Hkv * D), generator=g, device=dev).to(torch.bfloat16)
    qo = torch.empty((B, Hq, 1, D), dtype=torch.bfloat16, device=dev)
    cache.rope_append(0, qn, kn, vn, Hq, 1, 500000.0, qo)
    K, V = cache.views(0)
    out = ops.attention(qo, K, V, kv_strides=cache.kv_strides)
    assert cache.get_seq_length(0) == L + 1
    kb = K.contiguous().cpu().view(torch.int16).numpy().view(np.uint16)
    vb = V.contiguous().cpu().view(torch.int16).numpy().view(np.uint16)
    ref = _c_decode(to_np_f32(qo), kb, vb)
    assert rel_err(to_np_f32(out), ref) < TOL_BF16
    assert np.abs(to_np_f32(out) - ref).max() < 2e-2


@pytest.mark.parametrize("L,chunk", [(256, 64), (1000, 512), (2048, 512)])
def test_config5_prefill_bf16_mfma(dev, L, chunk):
    """BASELINE config 5 geometry (Hq32/Hkv8, D128, bf16, causal, chunk 512) at test sizes."""
    from lokahi_amd import ops
    rng = np.random.default_rng(L)
    B, Hq, Hkv, D = 1, 32, 8, 128
    q = round_bf16(rng.normal(size=(B, Hq, L, D)).astype(np.float32))
    k = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
    v = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
    out = ops.attention(bf16_dev(q, dev), bf16_dev(k, dev), bf16_dev(v, dev),
                        q_block_size=chunk, k_block_size=chunk)
    ref = att.chunked_gqa(q, k, v, None, True, chunk, chunk)
    assert rel_err(to_np_f32(out), ref) < TOL_BF16


@pytest.mark.parametrize("D,Hq,Hkv", [(64, 8, 2), (128, 12, 4), (64, 24, 8)])
def test_prefill_bf16_mfma32_ragged_positions_and_non_causal(dev, D, Hq, Hkv):
    """The bf16 32x32x16 prefill kernel off the bench geometry: head dims 64
    and 128, groups 4 and 3, batch 2, queries at explicit positions over a
    longer key range (32-key tiles with a tail, rows past Lq in the last
    128-row tile), and the non-causal form, against the float64 oracle."""
    from lokahi_amd import ops
    rng = np.random.default_rng(D * 100 + Hq)
    B, Lq, Lk = 2, 70, 150
    q = round_bf16(rng.normal(size=(B, Hq, Lq, D)).astype(np.float32))
    k = round_bf16(rng.normal(size=(B, Hkv, Lk, D)).astype(np.float32))
    v = round_bf16(rng.normal(size=(B, Hkv, Lk, D)).astype(np.float32))
    pos = np.stack([np.arange(Lk - Lq, Lk), np.sort(rng.integers(0, Lk, Lq))])
    tq, tk, tv = bf16_dev(q, dev), bf16_dev(k, dev), bf16_dev(v, dev)
    out = ops.attention(tq, tk, tv, query_positions=_t(pos, dev))
    assert rel_err(to_np_f32(out), att.naive_gqa(q, k, v, pos)) < TOL_BF16
    nm = ops.attention(tq, tk, tv, causal=False)
    assert rel_err(to_np_f32(nm), att.naive_gqa(q, k, v)) < TOL_BF16
    # bottom-right causal over Lq = Lk = 300 (several tiles, a partial last one)
    L = 300
    q2 = round_bf16(rng.normal(size=(1, Hq, L, D)).astype(np.float32))
    k2 = round_bf16(rng.normal(size=(1, Hkv, L, D)).astype(np.float32))
    v2 = round_bf16(rng.normal(size=(1, Hkv, L, D)).astype(np.float32))
    o2 = ops.attention(bf16_dev(q2, dev), bf16_dev(k2, dev), bf16_dev(v2, dev))
    ref2 = att.naive_gqa(q2, k2, v2, np.arange(L)[None])  # positions: causal
    assert rel_err(to_np_f32(o2), ref2) < TOL_BF16


def test_prefill_fp32_mfma_ragged_and_positions(dev):
    from lokahi_amd import ops
    rng = np.random.default_rng(77)
    B, Hq, Hkv, D = 2, 4, 1, 128
    Lq, Lk = 70, 150
    q = rng.normal(size=(B, Hq, Lq, D)).astype(np.float32)
    k = rng.normal(size=(B, Hkv, Lk, D)).astype(np.float32)
    v = rng.normal(size=(B, Hkv, Lk, D)).astype(np.float32)
    pos = np.stack([np.arange(Lk - Lq, Lk), np.sort(rng.integers(0, Lk, Lq))])
    out = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev), query_positions=_t(pos, dev))
    ref = att.naive_gqa(q, k, v, pos)
    assert rel_err(out.cpu().numpy(), ref) < TOL_F32
    nm = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev), causal=False)
    assert rel_err(nm.cpu().numpy(), att.naive_gqa(q, k, v)) < TOL_F32


def test_decode_equals_last_row_of_prefill_and_chunk_independence(dev):
    from lokahi_amd import ops
    rng = np.random.default_rng(5)
    B, Hq, Hkv, D, L = 1, 16, 4, 64, 300
    q = rng.normal(size=(B, Hq, L, D)).astype(np.float32)
    k = rng.normal(size=(B, Hkv, L, D)).astype(np.float32)
    v = rng.normal(size=(B, Hkv, L, D)).astype(np.float32)
    full = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev)).cpu().numpy()
    last = ops.attention(_t(q[:, :, -1:], dev), _t(k, dev), _t(v, dev)).cpu().numpy()
    np.testing.assert_allclose(full[:, :, -1:], last, atol=1e-4, rtol=1e-4)
    other = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev), q_block_size=7, k_block_size=3)
    np.testing.assert_allclose(full, other.cpu().numpy(), atol=1e-6)


@pytest.mark.parametrize("Hq,dtype", [(24, "bf16"), (48, "bf16"), (24, "f32")])
def test_decode_group_sizes_3_and_6(dev, Hq, dtype):
    """GQA groups of 3 (Llama-3.2-3B: 24 query / 8 KV heads) and 6 on the split-K decode kernel."""
    from lokahi_amd import ops
    rng = np.random.default_rng(Hq)
    B, Hkv, D, L = 2, 8, 128, 700
    q = round_bf16(rng.normal(size=(B, Hq, 1, D)).astype(np.float32))
    k = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
    v = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
    if dtype == "bf16":
        out = to_np_f32(ops.attention(bf16_dev(q, dev), bf16_dev(k, dev), bf16_dev(v, dev)))
        tol = TOL_BF16
    else:
        out = ops.attention(_t(q, dev), _t(k, dev), _t(v, dev)).cpu().numpy()
        tol = TOL_F32
    ref = att.chunked_gqa(q, k, v, None, True, 32768, 1024)
    assert rel_err(out, ref) < tol


@pytest.mark.parametrize("B,Hq,Hkv,D,L", [(16, 24, 8, 128, 300), (32, 8, 2, 64, 257),
                                          (8, 64, 8, 128, 97)])
def test_decode_batched_heads_mfma(dev, B, Hq, Hkv, D, L):
    """B * Hkv >= 64 runs the MFMA decode kernel (the G query heads of a KV head
    are the MFMA columns; G = 3, 4 and 8 here).  Per-row query positions cut
    each row's visible keys at a different point, including inside a 32-key
    tile and at the first key; the reference is float64 attention."""
    from lokahi_amd import ops
    rng = np.random.default_rng(B * 1000 + L)
    q = round_bf16(rng.normal(size=(B, Hq, 1, D)).astype(np.float32))
    k = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
    v = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
    pos = rng.integers(0, L, size=(B, 1))
    pos[0, 0], pos[-1, 0] = 0, L - 1
    out = to_np_f32(ops.attention(bf16_dev(q, dev), bf16_dev(k, dev), bf16_dev(v, dev),
                                  query_positions=torch.from_numpy(pos.astype(np.int32))))
    ref = att.naive_gqa(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64), pos)
    assert rel_err(out, ref) < TOL_BF16
    assert np.abs(out - ref).max() < 2e-2


def test_decode_split_k_back_to_back_and_graph_replays(dev):
    """Split-K decode calls of different geometry in a row (the partials of
    one call in the scratch arena the next call reuses), then graph replays of
    one call with eager calls of another geometry in between: every output
    must match the float64 attention."""
    from lokahi_amd import ops
    rng = np.random.default_rng(2048)
    cases = [(1, 32, 8, 128, 2049), (1, 24, 8, 128, 777), (2, 8, 8, 64, 300),
             (1, 32, 8, 128, 4100), (1, 8, 1, 128, 1500), (1, 32, 8, 128, 65)]
    data = []
    for B, Hq, Hkv, D, L in cases:
        q = round_bf16(rng.normal(size=(B, Hq, 1, D)).astype(np.float32))
        k = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
        v = round_bf16(rng.normal(size=(B, Hkv, L, D)).astype(np.float32))
        ref = att.naive_gqa(q.astype(np.float64), k.astype(np.float64), v.astype(np.float64))
        data.append(([bf16_dev(a, dev) for a in (q, k, v)], ref))
    for rep in range(2):
        for (tq, tk, tv), ref in data:
            out = to_np_f32(ops.attention(tq, tk, tv))
            assert rel_err(out, ref) < TOL_BF16 and np.abs(out - ref).max() < 2e-2, rep
    (tq, tk, tv), ref = data[0]
    out = torch.empty_like(tq)
    ops.attention(tq, tk, tv, out=out)  # eager first: sizes the scratch arena
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        ops.attention(tq, tk, tv, out=out)
    (eq, ek, ev), eref = data[1]
    for _ in range(3):
        out.zero_()
        g.replay()
        torch.cuda.synchronize()
        got = to_np_f32(out)
        assert rel_err(got, ref) < TOL_BF16 and np.abs(got - ref).max() < 2e-2
        e = to_np_f32(ops.attention(eq, ek, ev))
        assert rel_err(e, eref) < TOL_BF16


@pytest.mark.parametrize("dtype,B,Hq,Hkv,D,Lq,Lk,causal,given", [
    ("bf16", 1, 8, 2, 128, 2, 1000, True, False),    # 8 packed rows: one wave per tile
    ("bf16", 2, 6, 2, 64, 17, 1500, True, True),     # group 3, two waves, ragged rows and keys
    ("bf16", 1, 8, 2, 128, 100, 4100, True, False),  # four waves, an uneven last split
    ("bf16", 1, 6, 2, 128, 333, 1333, False, False), # not causal
    ("bf16", 1, 6, 2, 128, 1400, 1400, True, False), # a prompt: tiles that end in the first split
    ("f32", 1, 8, 2, 64, 512, 512, True, False), ("f32", 2, 6, 2, 128, 37, 437, True, True),
    ("f32", 1, 4, 4, 64, 70, 300, False, False)])
def test_prefill_key_splits(dev, dtype, B, Hq, Hkv, D, Lq, Lk, causal, given):
    """Prefill whose keys are split over workgroups (with the workspace ops
    passes) against float64, and against the call without a workspace.  Given
    positions include rows that see no key (0, as keys masked for every row
    give), rows that end in the first split and repeats.  The merge weighs each
    split's sums by one fp32 exp2 (2^-23 each), so the split result stays within
    the unsplit one's own distance from float64 (bf16: weights and outputs
    rounded at 2^-9; fp32: 2^-24 per sum term)."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk)
    q = torch.randn((B, Hq, Lq, D), generator=gen, device=dev).to(dt)
    k = torch.randn((B, Hkv, Lk, D), generator=gen, device=dev).to(dt)
    v = torch.randn((B, Hkv, Lk, D), generator=gen, device=dev).to(dt)
    need = C.c_int64()
    _abi.check(_abi.load().strata_attn_workspace(ops._ctx(0), ops._code(q), ops._code(k), ops._code(v),
                                                 B, Hq, Hkv, Lq, Lk, D, int(causal), C.byref(need)))
    assert need.value > 0  # the call is split
    pos = torch.arange(Lk - Lq, Lk, device=dev, dtype=torch.int32).expand(B, Lq)
    if given:
        pos = torch.randint(0, Lk, (B, Lq), generator=gen, device=dev, dtype=torch.int32)
        pos[0, 3], pos[0, 5], pos[-1, 7] = -1, 0, pos[-1, 6]
    row = pos[:, None, :, None] if causal else torch.full((B, 1, Lq, 1), Lk, device=dev)
    mask = torch.arange(Lk, device=dev) <= row
    sc = torch.matmul(q.double(), k.double().repeat_interleave(Hq // Hkv, 1).transpose(2, 3).contiguous())
    w = torch.exp(sc / D**0.5 - sc.amax(-1, keepdim=True) / D**0.5) * mask
    ref = torch.matmul(w, v.double().repeat_interleave(Hq // Hkv, 1)) / w.sum(-1, keepdim=True).clamp_min(1e-12)
    got = ops.attention(q, k, v, query_positions=pos if given else None, causal=causal)
    one = torch.empty_like(q)
    p32 = pos.contiguous()
    _abi.check(_abi.load().strata_attn_gqa(
        ops._ctx(0), q.data_ptr(), ops._code(q), k.data_ptr(), ops._code(k), v.data_ptr(), ops._code(v),
        Hkv * Lk * D, Lk * D, p32.data_ptr() if given else None, B, Hq, Hkv, Lq, Lk, D, int(causal),
        32768, 1024, C.c_float(1e-12), one.data_ptr(), ops._stream(0)))
    err, err1 = (float((o.double() - ref).norm() / ref.norm()) for o in (got, one))
    assert err1 < (5e-3 if dtype == "bf16" else 2e-6) and err < 1.2 * err1 + 1e-7, (err, err1)
    # a NaN key reaches the rows that see it, and no other
    k[0, 0, Lk // 3] = float("nan")
    got = ops.attention(q, k, v, query_positions=pos if given else None, causal=causal)
    sees = (mask[0, 0, :, Lk // 3] if causal else torch.ones(Lq, dtype=torch.bool, device=dev))
    assert bool(got[0, :Hq // Hkv, sees].isnan().all()) and bool(got[0, Hq // Hkv:].isfinite().all())


@pytest.mark.parametrize("dtype,B,Hq,Hkv,D,Lq,Lk,given", [
    ("bf16", 1, 8, 2, 128, 4, 230, False), ("bf16", 2, 6, 2, 64, 20, 234, True),
    ("bf16", 1, 8, 8, 128, 7, 90, False),
    ("f32", 1, 8, 2, 64, 100, 100, False), ("f32", 2, 6, 2, 64, 7, 70, True),
    ("f32", 1, 4, 4, 128, 33, 33, False), ("f32", 40, 8, 2, 64, 21, 40, False)])
def test_prefill_few_rows_without_split(dev, dtype, B, Hq, Hkv, D, Lq, Lk, given):
    """Short unsplit prefill against float64: bf16 tiles of 32 or 64 rows that
    four or eight waves load, fp32 tiles of 16 and 32 rows (16 * 40 * 2 tiles
    fill the CUs: 64).  Given positions include rows that see no key (0) and
    rows that see them all.  bf16 rounds weights and outputs at 2^-9, fp32 each
    sum term at 2^-24."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk)
    q, k, v = (torch.randn((B, h, l, D), generator=gen, device=dev).to(dt)
               for h, l in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    need = C.c_int64()
    _abi.check(_abi.load().strata_attn_workspace(ops._ctx(0), ops._code(q), ops._code(k), ops._code(v),
                                                 B, Hq, Hkv, Lq, Lk, D, 1, C.byref(need)))
    assert need.value == 0  # the call is not split
    pos = torch.arange(Lk - Lq, Lk, device=dev, dtype=torch.int32).expand(B, Lq)
    if given:
        pos = torch.randint(0, Lk, (B, Lq), generator=gen, device=dev, dtype=torch.int32)
        pos[0, 3], pos[0, 5], pos[-1, 6] = -1, 0, Lk - 1
    mask = torch.arange(Lk, device=dev) <= pos[:, None, :, None]
    sc = torch.matmul(q.double(), k.double().repeat_interleave(Hq // Hkv, 1).transpose(2, 3).contiguous())
    w = torch.exp((sc - sc.amax(-1, keepdim=True)) / D**0.5) * mask
    ref = torch.matmul(w, v.double().repeat_interleave(Hq // Hkv, 1)) / w.sum(-1, keepdim=True).clamp_min(1e-12)
    got = ops.attention(q, k, v, query_positions=pos if given else None)
    assert float((got.double() - ref).norm() / ref.norm()) < (5e-3 if dtype == "bf16" else 2e-6)
    if given:
        assert bool((got[0, :, 3] == 0).all())


@pytest.mark.parametrize("Hq,Hkv,D,Lq,Lk", [(24, 8, 128, 200, 200), (6, 2, 64, 193, 211),
                                            (32, 8, 128, 700, 707), (8, 8, 128, 130, 1000),
                                            (32, 8, 128, 1100, 1100), (32, 8, 128, 3000, 3000)])
def test_prefill_without_split(dev, Hq, Hkv, D, Lq, Lk):
    """Unsplit bf16 prefill (no workspace), the shapes of a small batch: key tiles
    shared by two wave groups of a workgroup (an odd and an even number of
    tiles, a last tile for one group only) and, for the last shape, 64-key
    tiles, against float64 rows; and each row's bits whatever the other rows
    of its tile hold."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    gen = torch.Generator(device=dev).manual_seed(Lq + D)
    q, k, v = (torch.randn((1, h, l, D), generator=gen, device=dev).bfloat16()
               for h, l in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))

    def call(q):
        out = torch.empty_like(q)
        _abi.check(_abi.load().strata_attn_gqa(
            ops._ctx(0), q.data_ptr(), ops._code(q), k.data_ptr(), ops._code(k), v.data_ptr(),
            ops._code(v), Hkv * Lk * D, Lk * D, None, 1, Hq, Hkv, q.shape[2], Lk, D, 1, 32768, 1024,
            C.c_float(1e-12), out.data_ptr(), ops._stream(0)))
        return out

    got = call(q)
    rows = torch.tensor(sorted({0, 1, 31, 32, Lq // 2, Lq - 2, Lq - 1}), device=dev)
    sc = torch.matmul(q[:, :, rows].double(),
                      k.double().repeat_interleave(Hq // Hkv, 1).transpose(2, 3).contiguous()) / D**0.5
    sc.masked_fill_(torch.arange(Lk, device=dev) > (rows + Lk - Lq)[:, None], float("-inf"))
    ref = torch.matmul(torch.softmax(sc, -1), v.double().repeat_interleave(Hq // Hkv, 1))
    assert float((got[:, :, rows].double() - ref).norm() / ref.norm()) < 5e-3
    assert bool(got.isfinite().all())
    keep = torch.arange(Lq, device=dev) % 3 != 1
    other = torch.where(keep[:, None], q, 3 * torch.randn(q.shape, generator=gen, device=dev).bfloat16())
    again = call(other)
    assert torch.equal(again[:, :, keep], got[:, :, keep])
    assert not torch.equal(again[:, :, ~keep], got[:, :, ~keep])


@pytest.mark.parametrize("kernel,D", [("one wave", 128), ("one wave", 64), ("two waves", 64), ("two waves", 128),
                                      ("short", 64), ("short", 128), ("plain", 128), ("plain", 64),
                                      ("64 keys", 64), ("64 keys", 128), ("three rounds", 128)])
@pytest.mark.parametrize("mask", ["causal", "given", "none"])
def test_prefill_unsplit_kernels_of_a_full_gpu(dev, kernel, D, mask):
    """The unsplit bf16 kernels for more tiles than CUs, the batch sized from the
    CU count: tiles of one and of two waves (up to 32 and 64 packed rows), of one
    wave for three key steps, the plain four-wave kernel (few steps, or tiles of
    one length in three rounds) and 64-key tiles (in two), causal, with given
    positions (rows that see no key, or all) and without a mask.  The first, a
    middle and the last batch row against float64
    (bf16 weights and outputs: 2^-9 each); rows keep their bits whatever the
    other rows of their tile hold."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    cus, Hq, Hkv = torch.cuda.get_device_properties(0).multi_processor_count, 12, 4
    Lq, Lk, tiles, per_cu = {"one wave": (10, 101, 1, 1), "two waves": (21, 201, 1, 1),
                             "short": (30, 70, 3, 1), "plain": (100, 164, 3, 6), "64 keys": (100, 260, 3, 1),
                             "three rounds": (100, 260, 3, 2)}[kernel]
    B = per_cu * cus // (tiles * Hkv) + 1
    gen = torch.Generator(device=dev).manual_seed(D + Lq)
    q, k, v = (torch.randn((B, h, l, D), generator=gen, device=dev).bfloat16()
               for h, l in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    pos = torch.arange(Lk - Lq, Lk, device=dev, dtype=torch.int32).repeat(B, 1)
    if mask == "given":
        pos = torch.randint(0, Lk, (B, Lq), generator=gen, device=dev, dtype=torch.int32)
        pos[:, 3], pos[:, 6] = -1, Lk - 1

    def call(q):
        out = torch.empty_like(q)
        _abi.check(_abi.load().strata_attn_gqa(
            ops._ctx(0), q.data_ptr(), ops._code(q), k.data_ptr(), ops._code(k), v.data_ptr(),
            ops._code(v), Hkv * Lk * D, Lk * D, pos.data_ptr() if mask == "given" else None, B, Hq, Hkv, Lq,
            Lk, D, int(mask != "none"), 32768, 1024, C.c_float(1e-12), out.data_ptr(), ops._stream(0)))
        return out

    got = call(q)
    rows = torch.tensor([0, B // 2, B - 1], device=dev)
    sc = torch.matmul(q[rows].double(),
                      k[rows].double().repeat_interleave(Hq // Hkv, 1).transpose(2, 3).contiguous()) / D**0.5
    w = torch.exp(sc - sc.amax(-1, keepdim=True))
    if mask != "none":
        w = w * (torch.arange(Lk, device=dev) <= pos[rows][:, None, :, None])
    ref = torch.matmul(w, v[rows].double().repeat_interleave(Hq // Hkv, 1)) / w.sum(-1, keepdim=True).clamp_min(1e-12)
    assert float((got[rows].double() - ref).norm() / ref.norm()) < 5e-3
    assert bool(got.isfinite().all())
    keep = torch.arange(Lq, device=dev) % 3 != 1
    again = call(torch.where(keep[:, None], q, 3 * torch.randn(q.shape, generator=gen, device=dev).bfloat16()))
    assert torch.equal(again[:, :, keep], got[:, :, keep])


@pytest.mark.parametrize("B,Hq,Hkv,D,Lq,Lk,causal", [(2, 8, 4, 64, 130, 130, False), (1, 16, 8, 128, 37, 200, True),
                                                     (8, 2, 1, 64, 33, 1000, True), (3, 24, 8, 128, 20, 300, False),
                                                     (3, 6, 3, 64, 70, 150, False)])
def test_prefill_f32_tiles_of_one_length(dev, B, Hq, Hkv, D, Lq, Lk, causal):
    """fp32 prefill without a mask or after a history, whose tiles run head by
    head where B x KV heads is a multiple of 8 (all shapes but the last), with
    and without a split of the keys, against float64 (2^-24 per sum term)."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk)
    q, k, v = (torch.randn((B, h, l, D), generator=gen, device=dev) for h, l in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    sc = torch.matmul(q.double(), k.double().repeat_interleave(Hq // Hkv, 1).transpose(2, 3).contiguous()) / D**0.5
    if causal:
        seen = torch.arange(Lk, device=dev) <= torch.arange(Lk - Lq, Lk, device=dev)[:, None]
        sc = sc.masked_fill(~seen, float("-inf"))
    ref = torch.matmul(torch.softmax(sc, -1), v.double().repeat_interleave(Hq // Hkv, 1))
    got = ops.attention(q, k, v, causal=causal)
    one = torch.empty_like(q)
    _abi.check(_abi.load().strata_attn_gqa(
        ops._ctx(0), q.data_ptr(), ops._code(q), k.data_ptr(), ops._code(k), v.data_ptr(), ops._code(v),
        Hkv * Lk * D, Lk * D, None, B, Hq, Hkv, Lq, Lk, D, int(causal), 32768, 1024, C.c_float(1e-12),
        one.data_ptr(), ops._stream(0)))
    for y in (got, one):
        assert float((y - ref).norm() / ref.norm()) < 1e-5


@pytest.mark.parametrize("dtype,B,Hq,Hkv,D,Lq,Lk", [("bf16", 1, 32, 8, 128, 100, 4100), ("bf16", 3, 6, 2, 64, 30, 1500),
                                                    ("f32", 1, 8, 2, 64, 200, 712), ("f32", 2, 6, 2, 128, 37, 437)])
def test_prefill_key_splits_over_cache_views(dev, dtype, B, Hq, Hkv, D, Lq, Lk):
    """Split prefill over K and V that are views into a longer cache, whose slots
    past the keys hold NaN: the bits of the call on contiguous copies."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk)
    lmax = Lk + 177
    q = torch.randn((B, Hq, Lq, D), generator=gen, device=dev).to(dt)
    kc, vc = (torch.full((B, Hkv, lmax, D), float("nan"), device=dev, dtype=dt) for _ in range(2))
    k, v = kc[:, :, :Lk], vc[:, :, :Lk]
    for t in (k, v):
        t.copy_(torch.randn((B, Hkv, Lk, D), generator=gen, device=dev))
    need = C.c_int64()
    _abi.check(_abi.load().strata_attn_workspace(ops._ctx(0), ops._code(q), ops._code(k), ops._code(v),
                                                 B, Hq, Hkv, Lq, Lk, D, 1, C.byref(need)))
    assert need.value > 0  # the call is split
    pos = torch.arange(Lk - Lq, Lk, device=dev, dtype=torch.int32)
    got = ops.attention(q, k, v, query_positions=pos, kv_strides=(Hkv * lmax * D, lmax * D))
    ref = ops.attention(q, k.contiguous(), v.contiguous(), query_positions=pos)
    assert torch.equal(got, ref) and bool(got.isfinite().all())


@pytest.mark.parametrize("dtype,B,Hq,Hkv,D,Lq,Lk,split", [
    ("bf16", 1, 32, 8, 128, 8, 100, False),     # 32 packed rows, four waves load
    ("bf16", 40, 32, 8, 64, 8, 97, False),      # one-wave tiles
    ("bf16", 40, 32, 8, 128, 16, 97, False),    # two-wave tiles
    ("bf16", 1, 24, 8, 128, 200, 289, False),   # two wave groups, Lk % 64 == 33
    ("bf16", 4, 24, 8, 64, 500, 544, False),    # 64-key tiles, Lk % 64 == 32
    ("bf16", 40, 32, 8, 128, 100, 132, False),  # the plain kernel
    ("bf16", 1, 32, 8, 128, 100, 2017, True), ("bf16", 2, 6, 2, 64, 17, 1508, True),
    ("bf16", 1, 8, 2, 128, 8, 1313, True),
    ("f32", 1, 8, 2, 64, 4, 100, False), ("f32", 1, 8, 2, 128, 60, 65, False),
    ("f32", 1, 8, 2, 64, 300, 545, True), ("f32", 2, 8, 2, 128, 5, 740, True)])
def test_prefill_positions_past_the_keys(dev, dtype, B, Hq, Hkv, D, Lq, Lk, split):
    """Given positions at or past the last key (absolute positions over a
    trimmed cache): such a row sees every key, and no more than those, whatever
    part of a tile the last keys fill.  Against float64 over the rule key <=
    position; bf16 rounds weights and outputs at 2^-9, fp32 each sum term at
    2^-24."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    dt = torch.bfloat16 if dtype == "bf16" else torch.float32
    gen = torch.Generator(device=dev).manual_seed(Lq + Lk)
    q, k, v = (torch.randn((B, h, l, D), generator=gen, device=dev).to(dt)
               for h, l in ((Hq, Lq), (Hkv, Lk), (Hkv, Lk)))
    need = C.c_int64()
    _abi.check(_abi.load().strata_attn_workspace(ops._ctx(0), ops._code(q), ops._code(k), ops._code(v),
                                                 B, Hq, Hkv, Lq, Lk, D, 1, C.byref(need)))
    assert (need.value > 0) == split
    past = torch.randint(Lk, 2 * Lk + 200, (B, Lq), generator=gen, device=dev, dtype=torch.int32)
    some = past.clone()  # a tile with both kinds of rows
    some[:, ::3] = torch.randint(0, Lk, (B, (Lq + 2) // 3), generator=gen, device=dev, dtype=torch.int32)
    sc = torch.matmul(q.double(), k.double().repeat_interleave(Hq // Hkv, 1).transpose(2, 3).contiguous())
    sc = torch.exp((sc - sc.amax(-1, keepdim=True)) / D**0.5)
    for pos in (past, some, past.clamp_min(2**31 - 1)):
        w = sc * (torch.arange(Lk, device=dev) <= pos[:, None, :, None])
        ref = torch.matmul(w, v.double().repeat_interleave(Hq // Hkv, 1)) / w.sum(-1, keepdim=True)
        got = ops.attention(q, k, v, query_positions=pos)
        err = float((got.double() - ref).norm() / ref.norm())
        assert err < (5e-3 if dtype == "bf16" else 2e-6), (int(pos.min()), err)


def test_attention_option_types(dev):
    """Block sizes and eps of any type that converts to an int and a float."""
    from lokahi_amd import ops
    q, k, v = (torch.randn((1, h, 5, 64), device=dev) for h in (4, 2, 2))
    ref = ops.attention(q, k, v)
    for qb, kb, eps in ((512.0, np.float64(256), np.float32(1e-12)), (float("inf"), 2**40, torch.tensor(1e-12)),
                        (np.int64(8), torch.tensor(4), 0)):
        out = ops.attention(q, k, v, q_block_size=qb, k_block_size=kb, eps=eps)
        assert torch.equal(out, ref)  # every weight sum is 1 - 2^-22 or more, above each eps
    with pytest.raises(ValueError, match="block sizes"):
        ops.attention(q, k, v, k_block_size=0.5)


@pytest.mark.parametrize("dtype,D", [("bf16", 128), ("bf16", 64), ("f32", 128), ("f32", 64)])
def test_workspace_bound_covers_every_call(dev, dtype, D):
    """strata_attn_workspace_max (what the decoder engine keeps) against the
    need of calls within its lengths: the lengths where the need peaks (24
    heads: 2771 tokens after 2336, 3000 after 8000), and random ones, causal or
    not; and it stays within a few times the largest of them."""
    import ctypes as C
    import random
    from lokahi_amd import _abi, ops
    lib, h, code = _abi.load(), ops._ctx(0), (_abi.BF16 if dtype == "bf16" else _abi.F32)
    n = C.c_int64()

    def need(B, Hq, Hkv, lq, lk, causal=1):
        _abi.check(lib.strata_attn_workspace(h, code, code, code, B, Hq, Hkv, lq, lk, D, causal, C.byref(n)))
        return n.value

    rng = random.Random(D)
    for B, Hq, Hkv in ((1, 24, 8), (2, 32, 8), (8, 32, 8), (1, 8, 2), (1, 64, 8), (3, 6, 6)):
        for most in (100, 260, 2048, 16384):
            _abi.check(lib.strata_attn_workspace_max(h, code, code, code, B, Hq, Hkv, most // B, most, D, C.byref(n)))
            bound, peak = n.value, 0
            pairs = [(lq, lk) for lq, lk in ((2771, 5107), (3000, 11000), (1000, 9000), (10, 458))
                     if lq <= most // B and lk <= most]
            for _ in range(3000):
                lq = min(most // B, int(2 * (most / 2 / B) ** rng.random()))
                pairs.append((lq, rng.randint(lq, most)))
            for lq, lk in pairs:
                got = need(B, Hq, Hkv, lq, lk, int(rng.random() < 0.8))
                assert got <= bound, (B, Hq, Hkv, most, lq, lk, got, bound)
                peak = max(peak, got)
            assert most < 2048 or bound < 8 * peak
