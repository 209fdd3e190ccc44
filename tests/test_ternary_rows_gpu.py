"""Ternary products of more than 8 rows (the matrix cores) against the oracle,
bit for bit: the edges of the 32 x 32 and 32 x 64 tiles and 64-row blocks, one
group and more than the loads in flight; relu; the 8-row launches' bits; and
passes of fewer rows than the product has when the scratch does not hold all."""

import numpy as np
import pytest

from oracle import oracle as O
from tests.device_memory import Device
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def inputs(n, k, m):
    codes = synth.ints(31 + n, (n, k), 0, 2).astype(np.uint8)
    scales = (0.01 + 0.04 * synth.uniform(32, (n, k // 128))).astype(np.float32)
    return codes, scales, synth.activations(33 + m, m, k)


@pytest.mark.parametrize("n,k,m", [(32, 128, 9), (33, 256, 31), (64, 384, 32), (65, 512, 33), (31, 640, 64),
                                   (200, 1024, 65), (4096, 256, 512), (4100, 384, 530), (1024, 4096, 40)])
def test_ternary_rows(gpu, n, k, m):
    print(f"case ternary rows n={n} k={k} m={m}", flush=True)
    codes, scales, x = inputs(n, k, m)
    layer = hip.Dense.ternary(codes, scales)
    got = layer.forward(x)
    assert bits_equal(got, O.Ternary(codes, scales)(x))
    assert bits_equal(got[8:16], layer.forward(x[8:16]))  # launches of up to 8 rows
    assert bits_equal(layer.forward(x, relu=True), np.maximum(got, 0))
    layer.free()


def test_passes_of_the_scratch(gpu):
    """8192 inputs: 448 rows fill the no-allocation array, so 1000 rows take three passes."""
    n, k, m = 48, 8192, 1000
    print(f"case ternary rows in passes n={n} k={k} m={m}", flush=True)
    codes, scales, x = inputs(n, k, m)
    layer = hip.Dense.ternary(codes, scales)
    D = Device()
    try:
        y = D.empty(m * n * 4)
        hip.check(hip.lib().trit_hip_layer_forward_device_noalloc(layer.h, D.upload(x), m, 0, y, None))
        assert bits_equal(D.download(y, (m, n)), O.Ternary(codes, scales)(x))
    finally:
        D.free()
        layer.free()
