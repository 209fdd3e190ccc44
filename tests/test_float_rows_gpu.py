"""Float-math products of more than 8 rows (the f32 matrix cores) against the
oracle's 16-lane order, bit for bit: every weight kind at the edges of its
tiles (16 rows and columns, 32 x 16 and 32 x 64 blocks), of its 256-input
operand blocks and of the chains' four-step loads; bias and relu; and passes of
fewer rows than the product has when the scratch does not hold them all."""

import numpy as np
import pytest

from oracle import oracle as O
from tests.device_memory import Device
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu

SHAPES = [(16, 160, 9), (17, 256, 16), (63, 288, 17), (64, 512, 33), (65, 1056, 31), (96, 4352, 40),
          (2049, 320, 230), (640, 192, 811)]


def bits_equal(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def layer_and_weights(kind, n, k, bias=None):
    if kind == "f16":
        bits = synth.f16_bits(synth.activations(81 + n, n, k) * 0.02).reshape(n, k)
        return hip.Dense.f16(bits, bias), bits.view(np.float16).astype(np.float32)
    if kind == "f32":
        w = synth.activations(82 + n, n, k) * np.float32(0.05)
        return hip.Dense.f32(w, bias), w
    codes = synth.ints(83 + n, (n, k), -127, 127).astype(np.int8)
    scales = (np.abs(synth.activations(84 + n, n, k // 32)) * np.float32(0.01)).astype(np.float32)
    return hip.Dense.q8(codes, scales, bias), codes.astype(np.float32) * np.repeat(scales, 32, axis=1)


@pytest.mark.parametrize("kind", ["f16", "f32", "q8"])
@pytest.mark.parametrize("n,k,m", SHAPES)
def test_many_rows(gpu, kind, n, k, m):
    print(f"case {kind} rows n={n} k={k} m={m}", flush=True)
    layer, w = layer_and_weights(kind, n, k)
    x = synth.activations(85 + m, m, k)
    assert bits_equal(layer.forward(x), O.matmul_f32(x, w))
    layer.free()


@pytest.mark.parametrize("kind,k", [("f16", 240), ("f16", 333), ("f32", 135), ("f32", 1001), ("f16", 4097)])
def test_odd_inputs(gpu, kind, k):
    """Chains whose steps are no multiple of four, and a padded last step."""
    n, m = 50, 37
    print(f"case {kind} rows n={n} k={k} m={m} bias relu", flush=True)
    bias = synth.activations(86, 1, n)[0]
    layer, w = layer_and_weights(kind, n, k, bias)
    x = synth.activations(87, m, k)
    assert bits_equal(layer.forward(x, relu=True), np.maximum(O.matmul_f32(x, w) + bias, 0))
    layer.free()


def test_passes_of_the_scratch(gpu):
    """8192 inputs: 128 rows fill the no-allocation array, so 300 rows take three passes."""
    n, k, m = 40, 8192, 300
    print(f"case f16 rows in passes n={n} k={k} m={m}", flush=True)
    layer, w = layer_and_weights("f16", n, k)
    x = synth.activations(88, m, k)
    D = Device()
    try:
        y = D.empty(m * n * 4)
        hip.check(hip.lib().trit_hip_layer_forward_device_noalloc(layer.h, D.upload(x), m, 0, y, None))
        assert bits_equal(D.download(y, (m, n)), O.matmul_f32(x, w))
    finally:
        D.free()
        layer.free()
