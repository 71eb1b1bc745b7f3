"""q4 linear (GEMV / MFMA GEMM), bf16 linear and the quantizer vs the oracle."""
import numpy as np
import pytest
import torch

from oracle import q4
from oracle.bf16 import bf16_bits_to_f32, f32_to_bf16_bits, round_bf16
from tests.gpu_util import bf16_dev, rel_err, to_dev, to_np_f32

pytestmark = pytest.mark.gpu

# Llama-3-8B decode linears (north_star config 2): (N, K)
SHAPES_8B = [(4096, 4096), (1024, 4096), (14336, 4096), (4096, 14336)]
TOL_BF16 = 2e-2   # rel-err bound for bf16 outputs
TOL_F32 = 1e-3    # rel-err bound for fp32 outputs


def _problem(rng, N, K, M=1):
    w, s, b = q4.quantize(rng.normal(0, 0.02, (N, K)).astype(np.float32), 64)
    x = f32_to_bf16_bits(rng.normal(0, 1, (M, K)).astype(np.float32))
    return w, s, b, x


@pytest.mark.parametrize("N,K", SHAPES_8B)
def test_gemv_decode_shapes_match_oracle(dev, N, K):
    from lokahi_amd import ops
    rng = np.random.default_rng(N + K)
    w, s, b, x = _problem(rng, N, K)
    ref = q4.quantized_matmul(bf16_bits_to_f32(x), w, s, b)
    tw, ts, tb, tx = (to_dev(a, dev) for a in (w, s, b, x))
    y32 = to_np_f32(ops.linear(tx, tw, ts, tb, out_dtype=torch.float32))
    assert rel_err(y32, ref) < TOL_F32
    y16 = to_np_f32(ops.linear(tx, tw, ts, tb))
    assert rel_err(y16, ref) < TOL_BF16
    # bf16 output is the RNE rounding of (nearly) the fp32 result
    assert np.mean(f32_to_bf16_bits(y32) == f32_to_bf16_bits(y16)) > 0.999


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 8])
def test_gemv_small_batches_and_fp32_activations(dev, M):
    from lokahi_amd import ops
    rng = np.random.default_rng(M)
    N, K = 384, 1024
    w, s, b, x = _problem(rng, N, K, M)
    ref = q4.quantized_matmul(bf16_bits_to_f32(x), w, s, b)
    tw, ts, tb = (to_dev(a, dev) for a in (w, s, b))
    y = to_np_f32(ops.linear(to_dev(x, dev), tw, ts, tb, out_dtype=torch.float32))
    assert rel_err(y, ref) < TOL_F32
    xf = rng.normal(0, 1, (M, K)).astype(np.float32)  # reference dtype flow: fp32 activations
    y = to_np_f32(ops.linear(torch.from_numpy(xf).to(dev), tw, ts, tb))
    assert rel_err(y, q4.quantized_matmul(xf, w, s, b)) < TOL_F32


def test_gemv_multi_problem_one_launch(dev):
    from lokahi_amd import ops
    rng = np.random.default_rng(9)
    K = 2048
    probs = [_problem(rng, n, K)[:3] for n in (512, 128, 128)]  # q / k / v-like
    x = f32_to_bf16_bits(rng.normal(0, 1, (1, K)).astype(np.float32))
    outs = ops.linear_multi(to_dev(x, dev), [tuple(to_dev(a, dev) for a in p) for p in probs],
                            out_dtype=torch.float32)
    for (w, s, b), y in zip(probs, outs):
        assert rel_err(to_np_f32(y), q4.quantized_matmul(bf16_bits_to_f32(x), w, s, b)) < TOL_F32


def test_gemv_edge_shapes(dev):
    from lokahi_amd import ops
    rng = np.random.default_rng(10)
    for N, K in [(1, 64), (3, 64), (17, 192), (1000, 320)]:
        w, s, b, x = _problem(rng, N, K)
        y = to_np_f32(ops.linear(to_dev(x, dev), *(to_dev(a, dev) for a in (w, s, b)),
                                 out_dtype=torch.float32))
        assert rel_err(y, q4.quantized_matmul(bf16_bits_to_f32(x), w, s, b)) < TOL_F32, (N, K)
    # all-zero codes: closed form y = sum_g b_g * sum x_g
    K = 256
    zw = np.zeros((4, K // 8), np.uint32)
    s = f32_to_bf16_bits(np.full((4, K // 64), 0.5, np.float32))
    bb = f32_to_bf16_bits(rng.normal(0, 1, (4, K // 64)).astype(np.float32))
    x = f32_to_bf16_bits(rng.normal(0, 1, (1, K)).astype(np.float32))
    y = to_np_f32(ops.linear(to_dev(x, dev), to_dev(zw, dev), to_dev(s, dev), to_dev(bb, dev),
                             out_dtype=torch.float32))
    expect = bf16_bits_to_f32(x).reshape(K // 64, 64).sum(1).astype(np.float64) @ bf16_bits_to_f32(bb).T
    np.testing.assert_allclose(y[0], expect, rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("M,N,K", [(64, 256, 512), (200, 1000, 1024), (1000, 384, 4096),
                                   (9, 128, 64), (2048, 4096, 4096)])
def test_gemm_prefill_matches_oracle(dev, M, N, K):
    from lokahi_amd import ops
    rng = np.random.default_rng(M * 7 + N)
    w, s, b, x = _problem(rng, N, K, M)
    y = to_np_f32(ops.linear(to_dev(x, dev), *(to_dev(a, dev) for a in (w, s, b)),
                             out_dtype=torch.float32))
    ref = q4.quantized_matmul(bf16_bits_to_f32(x), w, s, b)
    # weights are dequantized to bf16 in LDS (as MLX's qmm does): bf16 tolerance
    # against the exact product, fp32 tolerance against x @ bf16(dequant(W)).T
    assert rel_err(y, ref) < TOL_BF16
    wq = round_bf16(q4.dequantize(w, s, b, 64).astype(np.float32)).astype(np.float64)
    ref_b = bf16_bits_to_f32(x).astype(np.float64) @ wq.T
    assert rel_err(y, ref_b) < TOL_F32


@pytest.mark.parametrize("M,N,K", [(300, 1000, 1024), (512, 4096, 4096), (257, 96, 64)])
def test_gemm_prefill_rows_match_oracle(dev, M, N, K):
    """Prefill rows run the fused-dequant kernels (MFMA, or the 128 x 128 tile
    kernel for N not a multiple of 256): the bf16-staged product within fp32
    tolerance, the exact product within bf16 tolerance."""
    from lokahi_amd import ops
    rng = np.random.default_rng(M + N + K)
    w, s, b, x = _problem(rng, N, K, M)
    tw, ts, tb = (to_dev(a, dev) for a in (w, s, b))
    ref = q4.quantized_matmul(bf16_bits_to_f32(x), w, s, b)
    wq = round_bf16(q4.dequantize(w, s, b, 64).astype(np.float32)).astype(np.float64)
    ref_b = bf16_bits_to_f32(x).astype(np.float64) @ wq.T
    y32 = to_np_f32(ops.linear(to_dev(x, dev), tw, ts, tb, out_dtype=torch.float32))
    y16 = to_np_f32(ops.linear(to_dev(x, dev), tw, ts, tb))
    assert rel_err(y32, ref_b) < TOL_F32
    assert rel_err(y16, ref) < TOL_BF16


def test_linear_rejects_bad_parameters(dev):
    from lokahi_amd import ops
    w = torch.zeros((4, 8), dtype=torch.uint32, device=dev)
    s = torch.zeros((4, 1), dtype=torch.bfloat16, device=dev)
    x = torch.zeros((1, 64), dtype=torch.bfloat16, device=dev)
    with pytest.raises(ValueError):
        ops.linear(x, w, s, s, bits=8)
    with pytest.raises(ValueError):
        ops.linear(torch.zeros((1, 96), dtype=torch.bfloat16, device=dev), w, s, s)


def test_bf16_dense_linear(dev):
    from lokahi_amd import ops
    rng = np.random.default_rng(12)
    # K = 4096 takes the x-ahead-of-weights kernels (batch tiles 1, 2, 4;
    # M = 5 leaves three zeroed rows in its second tile)
    for M, N, K in [(1, 1000, 512), (3, 333, 256), (1, 777, 4096), (2, 500, 4096),
                    (4, 300, 4096), (5, 130, 4096)]:
        W = f32_to_bf16_bits(rng.normal(0, 0.02, (N, K)).astype(np.float32))
        x = f32_to_bf16_bits(rng.normal(0, 1, (M, K)).astype(np.float32))
        y = to_np_f32(ops.linear(to_dev(x, dev), to_dev(W, dev), None, None, out_dtype=torch.float32))
        ref = bf16_bits_to_f32(x).astype(np.float64) @ bf16_bits_to_f32(W).T.astype(np.float64)
        assert rel_err(y, ref) < TOL_F32


def test_quantizer_is_bit_exact_with_oracle(dev):
    from lokahi_amd import ops
    rng = np.random.default_rng(13)
    wf = rng.normal(0, 0.02, (300, 512)).astype(np.float32)
    pw, sc, bi = ops.quantize(torch.from_numpy(wf).to(dev))
    ew, es, eb = q4.quantize(wf, 64)
    assert np.array_equal(pw.cpu().view(torch.int32).numpy().view(np.uint32), ew)
    assert np.array_equal(sc.cpu().view(torch.int16).numpy().view(np.uint16), es)
    assert np.array_equal(bi.cpu().view(torch.int16).numpy().view(np.uint16), eb)


def test_gemm_many_prompt_lengths(dev):
    """Prefill M is the prompt length: a run of distinct lengths through the
    per-call re-layout and split-K routing stays correct."""
    from lokahi_amd import ops
    rng = np.random.default_rng(260)
    N, K = 256, 128
    w, s, b, x = _problem(rng, N, K, 600)
    tw, ts, tb, tx = (to_dev(a, dev) for a in (w, s, b, x))
    wq = round_bf16(q4.dequantize(w, s, b, 64).astype(np.float32)).astype(np.float64)
    for M in range(300, 560, 7):
        y = ops.linear(tx[:M], tw, ts, tb, out_dtype=torch.float32)
        ref = bf16_bits_to_f32(x[:M]).astype(np.float64) @ wq.T
        assert rel_err(to_np_f32(y), ref) < TOL_F32, M


@pytest.mark.parametrize("M,K", [(9, 1024), (16, 3584), (17, 1024), (40, 2048), (64, 1024),
                                 (65, 1024), (150, 512), (300, 1024)])
def test_gemm_few_rows_skinny_kernel(dev, M, K):
    """Up to 39 rows the skinny kernel runs: 16 or 64 output columns per
    workgroup, the K quarters of each column block summed in LDS (from 40
    rows, linears whose N is a multiple of 256 take the MFMA kernel, whose
    own test follows).  q/k/v-like linears in one launch, bf16 and fp32
    outputs, against x @ bf16(dequant(W)).T in float64, and bit-identical to
    separate launches of each linear."""
    from lokahi_amd import ops
    rng = np.random.default_rng(M * 7 + K)
    ns = (1024, 256, 256) if M != 16 else (16384, 16, 48)  # 64- and 16-column blocks
    probs = [_problem(rng, n, K)[:3] for n in ns]
    x = f32_to_bf16_bits(rng.normal(0, 1, (M, K)).astype(np.float32))
    dprobs = [tuple(to_dev(a, dev) for a in p) for p in probs]
    xd = to_dev(x, dev)
    y32 = ops.linear_multi(xd, dprobs, out_dtype=torch.float32)
    y16 = ops.linear_multi(xd, dprobs)
    for (w, s, b), a32, a16, dp in zip(probs, y32, y16, dprobs):
        wq = round_bf16(q4.dequantize(w, s, b, 64).astype(np.float32)).astype(np.float64)
        ref_b = bf16_bits_to_f32(x).astype(np.float64) @ wq.T
        assert rel_err(to_np_f32(a32), ref_b) < TOL_F32
        assert rel_err(to_np_f32(a16), q4.quantized_matmul(bf16_bits_to_f32(x), w, s, b)) < TOL_BF16
        alone = ops.linear(xd, *dp, out_dtype=torch.float32)
        assert torch.equal(alone, a32)


@pytest.mark.parametrize("M,K,ns", [(65, 4096, (4096, 1024, 1024)), (100, 1024, (1024, 256, 256)),
                                    (128, 4096, (14336,)), (200, 14336, (4096,)),
                                    (255, 2048, (512, 1536)), (300, 1024, (1024, 256, 256)),
                                    (777, 4096, (4096,)), (128, 4096, (14336, 4096)),
                                    (40, 512, (256,)), (1000, 64, (256, 512))])
def test_gemm_mid_rows_split_k(dev, M, K, ns):
    """40 rows and up, N a multiple of 256: the 256-column MFMA
    kernel over all rows (a partial last row tile), each linear whose tiles
    leave CUs idle split over K slices whose fp32 partial sums are added in
    slice order.  Against x @ bf16(dequant(W)).T in float64 and the oracle's
    q4 matmul; a linear gives the same bits in a fused launch as alone (the
    split depends on its own M, K and N only).  Includes a call whose
    linears get different slice counts (two launches), K = 64 (one group,
    no split) and exactly 40 rows at a short K."""
    from lokahi_amd import ops
    rng = np.random.default_rng(M * 11 + K)
    probs = [_problem(rng, n, K)[:3] for n in ns]
    x = f32_to_bf16_bits(rng.normal(0, 1, (M, K)).astype(np.float32))
    dprobs = [tuple(to_dev(a, dev) for a in p) for p in probs]
    xd = to_dev(x, dev)
    y32 = ops.linear_multi(xd, dprobs, out_dtype=torch.float32)
    y16 = ops.linear_multi(xd, dprobs)
    xf = bf16_bits_to_f32(x)
    for (w, s, b), a32, a16, dp in zip(probs, y32, y16, dprobs):
        wq = round_bf16(q4.dequantize(w, s, b, 64).astype(np.float32)).astype(np.float64)
        ref_b = xf.astype(np.float64) @ wq.T
        assert rel_err(to_np_f32(a32), ref_b) < TOL_F32
        assert rel_err(to_np_f32(a16), q4.quantized_matmul(xf, w, s, b)) < TOL_BF16
        assert torch.equal(ops.linear(xd, *dp, out_dtype=torch.float32), a32)
        assert torch.equal(ops.linear(xd, *dp), a16)


@pytest.mark.parametrize("M,N,K", [(3, 24576, 64), (9, 8200, 192), (32, 4097, 1024), (33, 8192, 320),
                                   (64, 2049, 4096), (161, 1000, 128), (700, 513, 256), (13, 6144, 72)])
def test_bf16_dense_linear_rows(dev, M, N, K):
    """Several rows of the dense linear: the MFMA kernel's row tiles (32-160
    rows, partial last ones), W tiles cut by N, an odd N (scalar stores), K
    below one accumulation chain and not a multiple of it, and K % 64 != 0
    (the GEMV).  fp32 sums of exact bf16 products: K terms of relative error
    2^-24 each stay under K * 2^-24 of the sum of magnitudes, here far below
    1e-5 of the result; bf16 outputs are the rounded fp32 ones."""
    from lokahi_amd import ops
    gen = torch.Generator(device=dev).manual_seed(M + N)
    W = (torch.randn((N, K), generator=gen, device=dev) * 0.02).bfloat16()
    x = torch.randn((M, K), generator=gen, device=dev).bfloat16()
    ref = x.double() @ W.double().T
    y = ops.linear(x, W, None, None, out_dtype=torch.float32)
    assert float((y - ref).norm() / ref.norm()) < 1e-5
    assert float((y - ref).abs().max() / ref.square().mean().sqrt()) < 1e-4
    assert torch.equal(ops.linear(x, W, None, None), y.bfloat16())
    if K % 64:
        return  # the GEMV multiplies the last x chunk by zero weights past K
    # an infinite or NaN activation reaches its own row only, as in a plain sum
    W.abs_()
    x[0, 0], x[1, K - 1], x[2, K // 2] = float("inf"), float("-inf"), float("nan")
    y = ops.linear(x, W, None, None, out_dtype=torch.float32)
    ref = x.float() @ W.float().T
    assert torch.equal(y[:3].isnan(), ref[:3].isnan())
    assert torch.equal(torch.where(y[:2].isinf(), y[:2], 0.), torch.where(ref[:2].isinf(), ref[:2], 0.))
    assert bool(y[3:].isfinite().all())


@pytest.mark.parametrize("M,K,ns", [(9, 512, (16, 48)), (16, 3072, (16384, 64)), (17, 1024, (1040,)),
                                    (32, 4096, (8192, 8192)), (33, 1536, (8192, 1024, 80)),
                                    (49, 2048, (256, 8192)), (64, 512, (768, 16)),
                                    (65, 1024, (256, 8192)), (129, 192, (512,)), (130, 128, (256,))])
def test_gemm_rows_at_kernel_borders(dev, M, K, ns):
    """Row counts where a linear's kernel changes (32 / 33 by width, 64 / 65),
    16-row blocks of the skinny kernel, linears of one call on different
    kernels, and K % 128 != 0 (the MFMA kernel's per-call re-layout).  fp32
    sums of exact bf16 products against float64: K terms at 2^-24 each."""
    from lokahi_amd import ops
    rng = np.random.default_rng(M * 13 + K)
    probs = [_problem(rng, n, K)[:3] for n in ns]
    x = f32_to_bf16_bits(rng.normal(0, 1, (M, K)).astype(np.float32))
    dprobs = [tuple(to_dev(a, dev) for a in p) for p in probs]
    xd = to_dev(x, dev)
    ys = ops.linear_multi(xd, dprobs, out_dtype=torch.float32)
    for (w, s, b), y, dp in zip(probs, ys, dprobs):
        wq = round_bf16(q4.dequantize(w, s, b, 64).astype(np.float32)).astype(np.float64)
        ref = bf16_bits_to_f32(x).astype(np.float64) @ wq.T
        assert rel_err(to_np_f32(y), ref) < 1e-5
        assert torch.equal(ops.linear(xd, *dp, out_dtype=torch.float32), y)


def test_gemm_layouts_agree(dev):
    """The MFMA kernel on the linear's own tensors (up to 512 rows) and on its
    re-laid-out copy (more rows) gives the same bits for the same rows."""
    from lokahi_amd import ops
    gen = torch.Generator(device=dev).manual_seed(4)
    w = ops.quantize(torch.randn((14336, 512), generator=gen, device=dev) * 0.02)
    x = torch.randn((513, 512), generator=gen, device=dev).bfloat16()
    assert torch.equal(ops.linear(x, *w)[:512], ops.linear(x[:512], *w))


@pytest.mark.parametrize("M,K,ns", [(3, 512, (16,)), (4, 1024, (1024, 48)), (5, 4096, (4096, 1024)),
                                    (7, 3072, (16384, 64)), (8, 14336, (64,)), (4, 4096, (256,)),
                                    (8, 448, (100,))])
def test_few_rows_keep_fp32_weights(dev, M, K, ns):
    """3-8 rows on the matrix cores (K % 512 == 0, N % 16 == 0) and the GEMV's
    shapes beside them: the weights' fp32 values, not their bf16 rounding.
    Codes enter as 128 + q, so sums of 32 terms carry 2^-24 of about 128 / 8
    times the result's size: below 1e-5 of the largest output, which bf16
    weights (2^-9 each) miss a hundredfold."""
    from lokahi_amd import ops
    rng = np.random.default_rng(M * 17 + K)
    probs = [_problem(rng, n, K)[:3] for n in ns]
    x = f32_to_bf16_bits(rng.normal(0, 1, (M, K)).astype(np.float32))
    dprobs = [tuple(to_dev(a, dev) for a in p) for p in probs]
    xd = to_dev(x, dev)
    for (w, s, b), y, dp in zip(probs, ops.linear_multi(xd, dprobs, out_dtype=torch.float32), dprobs):
        ref = bf16_bits_to_f32(x).astype(np.float64) @ q4.dequantize(w, s, b, 64).astype(np.float64).T
        assert rel_err(to_np_f32(y), ref) < 1e-5
        assert torch.equal(ops.linear(xd, *dp, out_dtype=torch.float32), y)


@pytest.mark.parametrize("M,K,ns", [(33, 512, (8192,)), (39, 4096, (14336, 14336)), (34, 1024, (8192, 48)),
                                    (36, 192, (256,)), (38, 320, (512, 256))])
def test_short_prefill_needs_no_scratch(dev, M, K, ns):
    """33-39 rows under capture with a context whose scratch arena cannot grow:
    the call runs as it does for fewer rows (on K slices or a re-layout it has
    no scratch for, it goes without), on every replay.  fp32 sums of exact
    bf16 products against float64: K terms at 2^-24 each."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    gen = torch.Generator(device=dev).manual_seed(M + K)
    ws = [ops.quantize(torch.randn((n, K), generator=gen, device=dev) * 0.02) for n in ns]
    x = torch.randn((M, K), generator=gen, device=dev).bfloat16()
    warm = ops.linear_multi(x, ws, out_dtype=torch.float32)
    ctx = _abi.Context(0)
    ys = [torch.empty_like(y) for y in warm]
    arr = (_abi.Q4Weight * len(ns))(*[_abi.Q4Weight(w.data_ptr(), s.data_ptr(), b.data_ptr(), n, y.data_ptr())
                                      for (w, s, b), n, y in zip(ws, ns, ys)])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rc = _abi.load().strata_linear_q4_multi(ctx.handle, x.data_ptr(), _abi.BF16, M, K, arr, len(ns), 64, 4,
                                                _abi.F32, ops._raw_stream(0))
    _abi.check(rc)
    for scale in (1.0, -2.0):
        x.mul_(scale)
        graph.replay()
        torch.cuda.synchronize()
        for (w, s, b), y, yw in zip(ws, ys, warm):
            ref = x.double() @ ops.dequantize(w, s, b).double().T
            assert float((y - ref).norm() / ref.norm()) < 1e-5
            if scale == 1.0:
                assert float((y - yw).norm() / yw.norm()) < 1e-5


@pytest.mark.parametrize("M,K,ns", [(5, 1536, (320, 48)), (9, 512, (16384, 48)), (33, 4096, (14336, 14336)), (39, 8192, (8192,)),
                                    (34, 1024, (8192, 8192, 256)), (36, 192, (8192,)), (39, 640, (256, 512))])
@pytest.mark.parametrize("offset", [0, 1])
def test_short_prefill_shares_no_memory(dev, M, K, ns, offset):
    """Up to 39 rows a call keeps nothing in memory that calls on other streams
    use: the same bits with a context that has no scratch and cannot get any (a
    captured call), and from two streams at once; also with scales and biases
    that start 2 bytes past a 4-byte boundary."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    gen = torch.Generator(device=dev).manual_seed(M + K)
    ws = [ops.quantize(torch.randn((n, K), generator=gen, device=dev) * 0.02) for n in ns]

    def moved(t):
        buf = torch.empty(t.numel() + offset, dtype=t.dtype, device=dev)
        buf[offset:] = t.flatten()
        return buf[offset:].view(t.shape)

    ws = [(w, moved(s), moved(b)) for w, s, b in ws]
    xs = torch.randn((2, M, K), generator=gen, device=dev).bfloat16()
    refs = [ops.linear_multi(x, ws, out_dtype=torch.float32) for x in xs]
    ctx = _abi.Context(0)
    ys = [torch.empty_like(y) for y in refs[0]]
    arr = (_abi.Q4Weight * len(ns))(*[_abi.Q4Weight(w.data_ptr(), s.data_ptr(), b.data_ptr(), n, y.data_ptr())
                                      for (w, s, b), n, y in zip(ws, ns, ys)])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        rc = _abi.load().strata_linear_q4_multi(ctx.handle, xs.data_ptr(), _abi.BF16, M, K, arr, len(ns), 64, 4,
                                                _abi.F32, ops._raw_stream(0))
    _abi.check(rc)
    graph.replay()
    torch.cuda.synchronize()
    assert all(torch.equal(y, r) for y, r in zip(ys, refs[0]))
    streams = [torch.cuda.Stream() for _ in range(2)]
    outs = [[], []]
    for _ in range(20):
        for i, stream in enumerate(streams):
            with torch.cuda.stream(stream):
                outs[i].append(ops.linear_multi(xs[i], ws, out_dtype=torch.float32))
    torch.cuda.synchronize()
    for got, ref in zip(outs, refs):
        assert all(torch.equal(y, r) for g in got for y, r in zip(g, ref))


def test_few_rows_beyond_32_bit_offsets(dev):
    """x of 4 GiB (64 rows): byte offsets that 32 bits do not hold.  x is zero
    but for a few columns, so the reference needs only those."""
    from lokahi_amd import ops
    M, K, N = 64, 1 << 25, 16
    gen = torch.Generator(device=dev).manual_seed(5)
    w = torch.randint(-2**31, 2**31 - 1, (N, K // 8), generator=gen, device=dev, dtype=torch.int32)
    s, b = (torch.rand((N, K // 64), generator=gen, device=dev).bfloat16() for _ in range(2))
    cols = torch.tensor([0, 1, 65, K // 4 + 7, K // 2, K - 70, K - 1], device=dev)
    xc = torch.randn((M, len(cols)), generator=gen, device=dev).bfloat16()
    x = torch.zeros((M, K), device=dev, dtype=torch.bfloat16)
    x[:, cols] = xc
    y = ops.linear(x, w, s, b, out_dtype=torch.float32)
    codes = (w[:, cols // 8] >> (4 * (cols % 8))) & 15
    wq = (codes * s[:, cols // 64].float() + b[:, cols // 64].float()).bfloat16()
    ref = xc.double() @ wq.double().T
    assert float((y - ref).norm() / ref.norm()) < 1e-5


@pytest.mark.parametrize("M,K,ns", [(9, 512, (48,)), (24, 8192, (3072,)), (32, 1024, (16384, 64)),
                                    (64, 1536, (80, 1024)), (40, 512, (8192, 256))])
def test_scales_at_odd_addresses(dev, M, K, ns):
    """Scales and biases that start 2 bytes past a 4-byte boundary (views into a
    larger buffer) take the same kernels as aligned ones: the same bits, also on
    every replay of a captured call; with a scratch arena that cannot grow, fp32
    sums in another order (K terms at 2^-24 each)."""
    import ctypes as C
    from lokahi_amd import _abi, ops
    gen = torch.Generator(device=dev).manual_seed(M + K)
    ws = [ops.quantize(torch.randn((n, K), generator=gen, device=dev) * 0.02) for n in ns]
    x = torch.randn((M, K), generator=gen, device=dev).bfloat16()

    def odd(t):
        buf = torch.empty(t.numel() + 1, dtype=t.dtype, device=dev)
        buf[1:] = t.flatten()
        return buf[1:].view(t.shape)

    wo = [(w, odd(s), odd(b)) for w, s, b in ws]
    assert all(t.data_ptr() % 4 == 2 for _, s, b in wo for t in (s, b))
    ref = ops.linear_multi(x, ws, out_dtype=torch.float32)
    for y, r in zip(ops.linear_multi(x, wo, out_dtype=torch.float32), ref):
        assert torch.equal(y, r)
    ys = [torch.empty_like(y) for y in ref]
    arr = (_abi.Q4Weight * len(ns))(*[_abi.Q4Weight(w.data_ptr(), s.data_ptr(), b.data_ptr(), n, y.data_ptr())
                                      for (w, s, b), n, y in zip(wo, ns, ys)])
    fresh = _abi.Context(0)
    for handle, bound in ((ops._ctx(0), 0.0), (fresh.handle, 1e-5)):
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            rc = _abi.load().strata_linear_q4_multi(handle, x.data_ptr(), _abi.BF16, M, K, arr, len(ns), 64, 4,
                                                    _abi.F32, ops._raw_stream(0))
        _abi.check(rc)
        for _ in range(3):
            for y in ys:
                y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            for y, r in zip(ys, ref):
                assert float((y - r).norm() / r.norm()) <= bound


@pytest.mark.parametrize("M,K,ns", [(4, 4096, (4096, 1024)), (3, 8192, (1024, 48)), (5, 8192, (1024, 48)),
                                    (4, 4608, (256,)), (3, 12288, (64,)), (6, 1024, (320, 100, 64)),
                                    (8, 512, (36, 16)), (4, 3584, (16384, 320))])
def test_few_rows_either_kernel(dev, M, K, ns):
    """3-8 rows on both sides of the choice between the GEMV (K that fills its
    steps, up to 4 rows) and the MFMA kernel, and linears of one call on either
    (N % 16 != 0: the GEMV): the weights' fp32 values against float64, and each
    linear's bits as alone."""
    from lokahi_amd import ops
    gen = torch.Generator(device=dev).manual_seed(M * K)
    x = torch.randn((M, K), generator=gen, device=dev).bfloat16()
    ws = [ops.quantize(torch.randn((n, K), generator=gen, device=dev) * 0.02) for n in ns]
    ys = ops.linear_multi(x, ws, out_dtype=torch.float32)
    for (w, s, b), n, y in zip(ws, ns, ys):
        codes = torch.stack([(w.view(torch.int32) >> (4 * i)) & 15 for i in range(8)], -1).view(n, K // 64, 64)
        wd = (codes * s.double()[..., None] + b.double()[..., None]).view(n, K)
        ref = x.double() @ wd.T
        assert float((y - ref).norm() / ref.norm()) < 1e-5
        assert torch.equal(ops.linear(x, w, s, b, out_dtype=torch.float32), y)


@pytest.mark.parametrize("M,N,K", [(64, 2559, 4096), (64, 2561, 4096), (12, 8192, 4096), (14, 10240, 4096),
                                   (4, 65536, 1024), (4, 65535, 1024), (4, 65536, 4096), (3, 12288, 2048),
                                   (16, 8192, 8192), (15, 8191, 8192), (8, 20480, 5120), (8, 20478, 5120),
                                   (2, 100, 16384), (5, 100, 8256)])
def test_bf16_dense_linear_either_kernel(dev, M, N, K):
    """Both sides of the dense linear's choice between the GEMV and the MFMA
    kernel (passes x columns by K, 4 rows, and K whose rows the GEMV's LDS does
    not hold).  fp32 sums of exact bf16 products against float64: K terms at
    2^-24 each."""
    from lokahi_amd import ops
    gen = torch.Generator(device=dev).manual_seed(M + N)
    W = (torch.randn((N, K), generator=gen, device=dev) * 0.02).bfloat16()
    x = torch.randn((M, K), generator=gen, device=dev).bfloat16()
    ref = torch.cat([x.double() @ w.double().T for w in W.split(16384)], 1)
    y = ops.linear(x, W, None, None, out_dtype=torch.float32)
    assert float((y - ref).norm() / ref.norm()) < 1e-5
    assert torch.equal(ops.linear(x, W, None, None), y.bfloat16())
