"""GPU parity of the int8 MFMA decode matvecs (nine tokens and more on Q4_K, GGUF and tiled): against the float64 product
of the Q8_1 activations, at edges of the token blocks (9, 16, 17, 32, 33), ragged rows, and fewer super-blocks than waves.
Products are exact and sums 32-bit: rel-L2 1e-6 (measured 0.7 - 1.3e-7); pair rows equal the one-matrix call's bit for
bit."""
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
