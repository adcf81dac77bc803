"""GPU parity of the row scale's workgroup-a-row kernel (rows past 8192 values) and of the router matvec's tilings (1 x 1
to 8 x 8 rows x tokens a wave). The row scale is exact against the oracle's operand; a router logit does not depend on
the tiling, so a batch's logits equal one-token calls' bit for bit (and the float64 product within 1e-5: 32-bit sums of
up to 2880 products)."""
import numpy as np
import pytest

from helpers import assert_bits_equal, assert_close_rel_l2, dev_bf16, dev_f32, host
from oracle import ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("K", [8200, 12288, 12296, 16384, 16392, 32768, 32776])   # the last: the scalar kernel
@pytest.mark.parametrize("dtype", ["f32", "bf16"])
def test_row_scale_long_rows(dev, dtype, K):
    import qmm.ops as ops
    from qmm import synth
    rng = np.random.default_rng(K)
    x = (rng.standard_normal((5, K)) * np.exp2(rng.integers(-10, 24, (5, 1)))).astype(np.float32)
    x[3] = 0
    x[4, -1] = 3.1e7                                   # the maximum in the row's last value
    if dtype == "bf16":
        xb = synth.to_bf16_bits(x)
        x, xt = synth.bf16_bits_to_f32(xb), dev_bf16(xb, dev)
    else:
        xt = dev_f32(x, dev)
    x16, sc = ops.row_scale_f16(xt)
    e = np.asarray(ref.row_scale_exponent(x)).reshape(-1)
    np.testing.assert_array_equal(host(sc), np.stack([2.0 ** -e, 2.0 ** e], 1).astype(np.float32))
    want = (x * (2.0 ** -e)[:, None].astype(np.float32)).astype(np.float16)
    np.testing.assert_array_equal(host(x16).view(np.uint16), want.view(np.uint16))


@pytest.mark.parametrize("T,E,H", [(3, 128, 2048), (13, 128, 2048), (70, 128, 2048), (515, 128, 2048), (300, 37, 2880),
                                   (9000, 9, 260), (5, 1, 768)])
@pytest.mark.parametrize("xdt,wdt", [("bf16", "f32"), ("f32", "bf16")])
def test_router_tilings(dev, T, E, H, xdt, wdt):
    import qmm.ops as ops
    from qmm import synth
    rng = np.random.default_rng(T + E + H)
    vals, dts = [], (xdt, wdt)
    for shape, dt in zip(((T, H), (E, H)), dts):
        v = rng.standard_normal(shape).astype(np.float32)
        b = synth.to_bf16_bits(v)
        vals.append((synth.bf16_bits_to_f32(b), dev_bf16(b, dev)) if dt == "bf16" else (v, dev_f32(v, dev)))
    (x, xt), (w, wt) = vals
    _, _, logits = ops.moe_route(xt, wt, 1, 1, True)
    got = host(logits)
    assert_close_rel_l2(got, x.astype(np.float64) @ w.astype(np.float64).T, 1e-5, "logits")
    for t in (0, T // 2, T - 1):
        _, _, one = ops.moe_route(xt[t:t + 1].contiguous(), wt, 1, 1, True)
        assert_bits_equal(host(one)[0], got[t], f"token {t}")
