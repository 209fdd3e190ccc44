"""The matrix cores' f32 sums at the ends of f32's range, against the oracle, bit
for bit: v_mfma_f32's steps are fused multiply-adds rounded one by one with
subnormals kept, which the float-math products, the row attention and the integer
products' scale products rest on. Inputs, products and sums that are subnormal, and
exponents spread over the whole range; rows an infinity makes infinite or NaN."""

import numpy as np
import pytest

from oracle import oracle as O
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


def same_or_both_nan(a, b):
    a, b = np.asarray(a, np.float32), np.asarray(b, np.float32)
    return np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(a[~np.isnan(a)].view(np.uint32),
                                                                       b[~np.isnan(b)].view(np.uint32))


def spread(seed, shape, low, high):
    """Values of either sign with exponents uniform in [low, high)."""
    e = low + (high - low) * synth.uniform(seed, shape)
    sign = np.where(synth.uniform(seed ^ 0x55, shape) < 0.5, -1.0, 1.0)
    with np.errstate(under="ignore"):
        return (sign * np.exp2(e)).astype(np.float32)


# Exponents of x and of the weights.
RANGES = [((-80, -60), (-80, -60)), ((-149, -126), (-3, 3)), ((-100, 40), (-60, 40)), ((-140, 0), (-20, 60))]


@pytest.mark.parametrize("xs,ws", RANGES)
def test_float_rows(gpu, xs, ws):
    print(f"case float rows of exponents {xs} by {ws}", flush=True)
    n, k, m = 96, 544, 40
    x, w = spread(201, (m, k), *xs), spread(202, (n, k), *ws)
    want = O.matmul_f32(x, w)
    assert (np.abs(want) < 2.0**-126).any() == (RANGES.index((xs, ws)) < 2)  # subnormal outputs among them
    layer = hip.Dense.f32(w)
    assert same_or_both_nan(layer.forward(x), want)
    layer.free()


@pytest.mark.parametrize("hd", [64, 128])
@pytest.mark.parametrize("scores,values", [((-75, -65), (-149, -130)), ((-20, 4), (-149, -100)), ((-70, 2), (-149, 60))])
def test_attention_rows(gpu, hd, scores, values):
    print(f"case attention rows hd={hd} exponents {scores} {values}", flush=True)
    tq, tk, heads = 20, 150, 2
    q, k = spread(203, (tq, heads * hd), *scores), spread(204, (tk, heads * hd), *scores)
    v = spread(205, (tk, heads * hd), *values)
    got = hip.attention(q, k, v, heads, heads, hd, False, hip.EXACT)
    assert same_or_both_nan(got, O.attention(q, k, v, heads, heads, hd, causal=False))


@pytest.mark.parametrize("kind,k", [("int8", 512), ("ternary", 512), ("q8_0", 512), ("q8_0", 480)])
@pytest.mark.parametrize("rows", [5, 40])
def test_scale_products(gpu, kind, k, rows):
    """Group scales whose products are subnormal; a zero group; a row with an infinity."""
    print(f"case scale products {kind} k={k} rows={rows}", flush=True)
    n = 96
    x = spread(206, (rows, k), -70, -40)
    x[1, 128:256] = 0.0
    x[2] = spread(207, (k,), -149, -120)
    x[3, 7] = np.inf
    if kind == "q8_0":
        # (f16 scales: the x scales are rounded through f16 too.)
        x[4] = spread(209, (k,), -14, -2)
        codes, sbits = synth.q8_0_matrix(synth.seed_for(208, 1), n, k)
        sbits = np.where(synth.uniform(208, sbits.shape) < 0.5, 1, sbits).astype(np.uint16)  # f16's least
        layer = hip.Dense.q8_0(n, k, synth.q8_0_blocks(codes, sbits))
        want = O.Int8(codes, sbits.view(np.float16).astype(np.float32), 32, True)(x)
    else:
        scales = np.abs(spread(208, (n, k // 128), -110, -70))
        if kind == "int8":
            codes = synth.ints(209, (n, k), -127, 127).astype(np.int8)
            layer, want = hip.Dense.int8(codes, scales), O.Int8(codes, scales, 128, False)(x)
        else:
            codes = synth.ints(209, (n, k), 0, 2).astype(np.uint8)
            layer, want = hip.Dense.ternary(codes, scales), O.Ternary(codes, scales)(x)
    assert same_or_both_nan(layer.forward(x), want)
    layer.free()
