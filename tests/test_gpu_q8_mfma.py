"""GPU parity of the int8 MFMA decode matvecs (nine tokens and more on Q4_K, GGUF and tiled): against the float64 product
of the Q8_1 activations, at edges of the token blocks (9, 16, 17, 32, 33), ragged rows, and fewer super-blocks than waves.
Products are exact and sums 32-bit: rel-L2 1e-6 (measured 0.7 - 1.3e-7); pair rows equal the one-matrix call's bit for
bit. And bit for bit (make_kernel_tests.py:264-268): every token of a call equals its one-token call, in each summation
order (items up to and past one super-block a lane, K slices of two and four super-blocks, one to three tiled slices a
wave), rows quantized in the kernel equal the planar buffer, and the tiled layout equals the GGUF blocks at K = 4096."""
import numpy as np
import pytest

from helpers import assert_bits_equal, assert_close_rel_l2, dev_bf16, dev_f32, dev_u8, host
from oracle import formats as of
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,N,K", [(9, 4096, 256), (16, 2056, 1280), (17, 4104, 4096), (32, 1040, 2560), (33, 1005, 8192),
                                   (63, 528, 12288)])
@pytest.mark.parametrize("fmt", ["q4_k", "q4_kt"])
@pytest.mark.parametrize("mode", ["store", "acc", "swiglu"])
def test_mv_q8_mfma(dev, fmt, mode, M, N, K):
    import qmm.ops as ops
    from qmm import synth
    if fmt == "q4_kt":
        N, K = -(-N // 16) * 16, -(-K // 512) * 512
    rng = np.random.default_rng(M + N + K)
    w = [synth.q4_k_weights(rng, N, K) for _ in range(2)]
    xb = synth.to_bf16_bits(rng.standard_normal((M, K)).astype(np.float32))
    xt, xq = dev_bf16(xb, dev), ref.q8_1(synth.bf16_bits_to_f32(xb))
    p = [ref.gemv(xq, of.dequant_q4_k(v, N, K)) for v in w]
    wt = [dev_u8(v, dev) for v in w]
    if fmt == "q4_kt":
        wt = [ops.tile_q4k(t, N, K) for t in wt]
    y0 = rng.standard_normal((M, N)).astype(np.float32)
    if mode == "swiglu":
        y = ops.linear(fmt, xt, wt[0], N, K, mode="swiglu", w2=wt[1])
        want = ref.silu_mul(*p)
    else:
        y = ops.linear(fmt, xt, wt[0], N, K, mode=mode, y=dev_f32(y0, dev) if mode == "acc" else None)
        want = p[0] + (y0 if mode == "acc" else 0)
    assert_close_rel_l2(host(y), want, 1e-6, f"{fmt} {mode} {M}x{N}x{K}")
    if mode == "store":
        a, b = ops.mv_pair_q8(fmt, wt[0], wt[1], xt, N, K)
        assert_bits_equal(host(a), host(y), "pair y")
        assert_bits_equal(host(b), host(ops.mv_q8(fmt, wt[1], xt, N, K)), "pair y2")


def _same(got, want, what):
    """Equal bit for bit; a NaN equals any NaN."""
    nan = np.isnan(want)
    np.testing.assert_array_equal(np.isnan(got), nan, err_msg=what)
    assert_bits_equal(np.where(nan, 0, got).astype(np.float32), np.where(nan, 0, want).astype(np.float32), what)


def _call(fmt, mode, xt, w, N, K, y0=None):
    import qmm.ops as ops
    if mode == "pair":
        return [host(v) for v in ops.mv_pair_q8(fmt, *w, xt, N, K)]
    if mode == "swiglu":
        return [host(ops.mv_swiglu_q8(fmt, *w, xt, N, K))]
    y = None if y0 is None else dev_f32(y0, xt.device)
    return [host(ops.mv_q8(fmt, w[0], xt, N, K, y=y, accumulate=y is not None))]


@pytest.mark.parametrize("fmt,M,N,K", [
    ("q4_k", 9, 3700, 256), ("q4_k", 33, 1005, 1280), ("q4_k", 16, 2056, 2560),     # up to one super-block an item lane
    ("q4_k", 24, 1400, 4352), ("q4_k", 11, 3001, 12288),                             # several
    ("q4_k", 17, 2050, 4096), ("q4_k", 63, 528, 4096), ("q4_k", 12, 2800, 8192),     # K slices (swiglu: items)
    ("q4_kt", 9, 3712, 1024), ("q4_kt", 20, 1648, 2560), ("q4_kt", 33, 1008, 4096),   # one tiled slice a wave
    ("q4_kt", 16, 2048, 5120), ("q4_kt", 40, 832, 12288)])                           # two, three
@pytest.mark.parametrize("mode", ["store", "acc", "swiglu", "pair"])
def test_multi_token_equals_one_token(dev, fmt, mode, M, N, K):
    """Token 3 holds a group whose f16 scale is infinite: its outputs are those of the one-token call too."""
    import qmm.ops as ops
    from qmm import synth
    rng = np.random.default_rng(M + N + K)
    w = [dev_u8(synth.q4_k_weights(rng, N, K), dev) for _ in range(2)]
    if fmt == "q4_kt":
        w = [ops.tile_q4k(t, N, K) for t in w]
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[3, 32:64] *= 1e8
    xt = dev_bf16(synth.to_bf16_bits(x), dev)
    y0 = rng.standard_normal((M, N)).astype(np.float32) if mode == "acc" else None
    got = _call(fmt, mode, xt, w, N, K, y0)
    assert not np.isfinite(got[0][3]).any() and np.isfinite(got[0][4:]).all()
    for t in (0, 1, 3, M // 2, M - 1):
        one = _call(fmt, mode, xt[t:t + 1].contiguous(), w, N, K, None if y0 is None else y0[t:t + 1])
        for a, b in zip(got, one):
            _same(a[t], b[0], f"{fmt} {mode} {M}x{N}x{K} token {t}")


@pytest.mark.parametrize("K", [4096, 8192])
def test_rows_planar_and_layouts_agree(dev, K):
    """Q4_K through the C ABI with bf16 rows (quantized in the kernel) against the planar buffer, and the tiled layout
    against the GGUF blocks (K = 4096), at 12 and 33 tokens."""
    import torch
    import qmm.ops as ops
    from qmm import _lib, synth
    rng = np.random.default_rng(K)
    N = 2800
    w = dev_u8(synth.q4_k_weights(rng, N, K), dev)
    for M in (12, 33):
        xt = dev_bf16(synth.to_bf16_bits(rng.standard_normal((M, K)).astype(np.float32)), dev)
        xq = ops.quant_q8(xt)
        planar = host(ops.mv_q8("q4_k", w, xq, N, K, tokens=M))
        y = torch.empty((M, N), dtype=torch.float32, device=dev)
        _lib.call("qmm_mv_q8", 1, K, N, M, 0, xt.data_ptr(), 2, w.data_ptr(), y.data_ptr(),
                  torch.cuda.current_stream().cuda_stream)
        assert_bits_equal(host(y), planar, f"rows against planar, {M} tokens")
        if K == 4096:
            tiled = ops.mv_q8("q4_kt", ops.tile_q4k(w, N, K), xq, N, K, tokens=M)
            assert_bits_equal(host(tiled), planar, f"tiled against GGUF, {M} tokens")


@pytest.mark.parametrize("M,K", [(1, 4096), (3, 8192), (4, 2048)])
def test_pair_rows_equal_one_matrix_few_tokens(dev, M, K):
    """GGUF Q4_K pairs below nine tokens: the one-matrix call's bits, also where that is the K-sliced kernel's."""
    import qmm.ops as ops
    from qmm import synth
    rng = np.random.default_rng(M + K)
    N = 1003
    w = [dev_u8(synth.q4_k_weights(rng, N, K), dev) for _ in range(2)]
    xt = dev_bf16(synth.to_bf16_bits(rng.standard_normal((M, K)).astype(np.float32)), dev)
    got = ops.mv_pair_q8("q4_k", *w, xt, N, K)
    for g, v in zip(got, w):
        assert_bits_equal(host(g), host(ops.mv_q8("q4_k", v, xt, N, K)), f"pair M={M} K={K}")
