"""GPU parity of the tile GEMM's workgroup shapes (qmm_gemm picks one by the tile count): every format and mode at sizes
that take each shape (Q4_K store / acc: the first four the kernel of gemm_dense.hip), with partial row and column tiles,
K-parts of unequal and zero length, and 64-row runs of padding rows inside a 128-row tile. Oracle: the float64 product of the f16 operand and the exactly dequantized weights, rel-L2
1e-3 (f16 weights round at 2^-11: 2.8e-4 rms, 4e-4 for the product of two such sums)."""
import numpy as np
import pytest

from helpers import assert_close_rel_l2, dev_f32, dev_u8, host
from oracle import formats as of
from oracle import ref

pytestmark = pytest.mark.gpu

SIZES = [(64, 128, 256),       # 64 x 128 tiles, four K-parts of which two are empty
         (77, 145, 768),       # the same, parts of one and two steps
         (200, 129, 1280),     # a last row tile of eight rows (one 32-row block)
         (300, 4097, 256),     # 64 x 256 tiles as gate / up
         (300, 8190, 256),     # 64 x 256 tiles; as gate / up 128 x 256 tiles, two K-parts of one step each
         (1100, 4001, 512),    # 128 x 256 tiles, two K-parts; as gate / up 64 x 256
         (4090, 3327, 256)]    # 128 x 256 tiles, one K-part


@pytest.mark.parametrize("M,N,K", SIZES)
@pytest.mark.parametrize("fmt", ["q4_k", "q4_kt", "q6_k", "q4_0"])
@pytest.mark.parametrize("mode", ["store", "acc", "swiglu"])
def test_tile_gemm_shapes(dev, fmt, mode, M, N, K):
    import torch
    import qmm.ops as ops
    from qmm import synth
    if fmt == "q4_kt":
        N, K = N // 16 * 16, -(-K // 512) * 512
    rng = np.random.default_rng(M + N + K)
    base = "q4_k" if fmt == "q4_kt" else fmt
    w = [synth.weights(base, rng, N, K) for _ in range(2 if mode == "swiglu" else 1)]
    x = rng.standard_normal((M, K)).astype(np.float16)
    sc = np.exp2(rng.integers(-2, 3, (M, 1))).astype(np.float32)
    scales = np.concatenate([1 / sc, sc], 1)
    y0 = rng.standard_normal((M, N)).astype(np.float32) if mode == "acc" else np.full((M, N), 7.0, np.float32)
    if M > 1000:                                   # padding rows 64 .. 127: nothing is computed or written
        scales[64:128] = 0
    prods = [ref.gemv(x.astype(np.float32), of.dequantize(base, v, N, K)) * sc for v in w]
    want = prods[0] + y0 if mode == "acc" else prods[0]
    if mode == "swiglu":
        want = ref.silu_mul(prods[0], prods[1])
    wt = [dev_u8(v, dev) for v in w]
    if fmt == "q4_kt":
        wt = [ops.tile_q4k(t, N, K) for t in wt]
    y = dev_f32(y0, dev)
    ops.gemm(fmt, mode, torch.from_numpy(x).to(dev), wt[0], N, K, w2=wt[1] if mode == "swiglu" else None,
             scales=dev_f32(scales, dev), y=y)
    got = host(y)
    live = np.ones(M, bool)
    if M > 1000:
        live[64:128] = False
        np.testing.assert_array_equal(got[64:128], y0[64:128])
    assert_close_rel_l2(got[live], want[live], 1e-3, f"{fmt} {mode} {M}x{N}x{K}")
