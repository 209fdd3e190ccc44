"""Products of 9 to 17 rows on both sides of the rules that choose between two
launches of up to 8 rows and the matrix cores, against the oracle, bit for bit;
rows that start at any 4-byte boundary among them."""

import numpy as np
import pytest

from oracle import oracle as O
from tests.device_memory import Device
from tests.test_float_rows_gpu import bits_equal, layer_and_weights
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,n,k", [
    ("f16", 512, 512), ("f16", 513, 512), ("f16", 1024, 4096), ("f16", 1025, 512), ("f16", 40, 8192), ("f16", 64, 1024),
    ("f32", 512, 1024), ("f32", 513, 2048), ("f32", 64, 2112), ("q8", 1024, 512), ("q8", 1025, 1024), ("q8", 513, 2304)])
def test_float_rows(gpu, kind, n, k):
    print(f"case few rows {kind} n={n} k={k}", flush=True)
    layer, w = layer_and_weights(kind, n, k)
    x = synth.activations(71, 17, k)
    want = O.matmul_f32(x, w)
    D = Device()
    try:
        y, dx = D.empty(17 * n * 4), D.upload(x)
        odd = D.upload(np.concatenate([x.reshape(-1)[:1], x.reshape(-1)]))
        for rows in (9, 12, 13, 16, 17):
            for at in (dx, odd.value + 4):
                hip.check(hip.lib().trit_hip_layer_forward_device(layer.h, at, rows, 0, y, None))
                assert bits_equal(D.download(y, (rows, n)), want[:rows]), (rows, at)
    finally:
        D.free()
        layer.free()


@pytest.mark.parametrize("n,k", [(1024, 3584), (2048, 4096), (1024, 4096), (1028, 4096), (1024, 5120), (31, 5120),
                                 (64, 6144), (64, 6784), (64, 6912)])
def test_ternary_rows(gpu, n, k):
    print(f"case few rows ternary n={n} k={k}", flush=True)
    codes, scales = synth.ternary_matrix(synth.seed_for(72, n), n, k)
    layer = hip.Dense.ternary(codes, scales)
    x = synth.activations(73, 17, k)
    want = O.Ternary(codes, scales)(x)
    D = Device()
    try:
        y, dx = D.empty(17 * n * 4), D.upload(x)
        for rows in (9, 10, 12, 13, 16, 17):
            hip.check(hip.lib().trit_hip_layer_forward_device(layer.h, dx, rows, 0, y, None))
            assert bits_equal(D.download(y, (rows, n)), want[:rows]), rows
            hip.check(hip.lib().trit_hip_layer_forward_device_noalloc(layer.h, dx, rows, 0, y, None))
            assert bits_equal(D.download(y, (rows, n)), want[:rows]), rows
    finally:
        D.free()
        layer.free()


# The tiles' rules: 32 x 64 outputs a block from 512 blocks (or a round of 224 to
# 256 with long rows), 32 x 16 before; steps that are and are not a multiple of four.
@pytest.mark.parametrize("kind,n,k,m", [
    ("f16", 2049, 320, 500), ("f16", 1984, 320, 512), ("f16", 2048, 333, 510), ("f16", 512, 1040, 897),
    ("f16", 450, 1024, 1030), ("f32", 640, 192, 1650), ("f32", 1100, 1001, 930), ("f32", 512, 1024, 1000),
    ("q8", 2100, 288, 512), ("q8", 470, 1056, 1020)])
def test_float_tiles(gpu, kind, n, k, m):
    print(f"case tiles {kind} n={n} k={k} m={m}", flush=True)
    layer, w = layer_and_weights(kind, n, k)
    x = synth.activations(74 + m, m, k)
    assert bits_equal(layer.forward(x), O.matmul_f32(x, w, O.isa_best()))
    layer.free()


@pytest.mark.parametrize("n,k,m", [(4096, 256, 320), (4096, 256, 321), (4090, 384, 340), (1500, 256, 1000)])
def test_ternary_tiles(gpu, n, k, m):
    print(f"case tiles ternary n={n} k={k} m={m}", flush=True)
    codes, scales = synth.ternary_matrix(synth.seed_for(75, n), n, k)
    layer = hip.Dense.ternary(codes, scales)
    x = synth.activations(76 + m, m, k)
    assert bits_equal(layer.forward(x), O.Ternary(codes, scales)(x))
    layer.free()
