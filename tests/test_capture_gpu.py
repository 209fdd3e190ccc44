"""trit_hip_layer_forward_device under stream capture, and beside graphs
captured from it, bit for bit: a graph of an integer product keeps its scratch
while float-math and ternary products of many rows grow memory of their own on
the same thread, and those products, captured themselves, run in launches of 8
rows. Every replay is checked, with eager work and waits in between."""

import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O
from tests.device_memory import Device
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


def bits_equal(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


class Graph:
    """What `body(stream)` queues, captured."""

    def __init__(self, body):
        self.L, self.stream, self.exec = C.CDLL("libamdhip64.so"), C.c_void_p(), C.c_void_p()
        graph = C.c_void_p()
        assert self.L.hipStreamCreate(C.byref(self.stream)) == 0
        assert self.L.hipStreamBeginCapture(self.stream, 1) == 0  # thread-local
        body(self.stream)
        assert self.L.hipStreamEndCapture(self.stream, C.byref(graph)) == 0
        assert self.L.hipGraphInstantiate(C.byref(self.exec), graph, None, None, C.c_size_t(0)) == 0
        assert self.L.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.L.hipGraphLaunch(self.exec, self.stream) == 0
        assert self.L.hipStreamSynchronize(self.stream) == 0

    def free(self):
        assert self.L.hipGraphExecDestroy(self.exec) == 0
        assert self.L.hipStreamDestroy(self.stream) == 0


def forward(layer, x, m, y, stream=None):
    hip.check(hip.lib().trit_hip_layer_forward_device(layer.h, x, m, 0, y, stream))


def test_growing_products_leave_a_captured_scratch(gpu):
    print("case a captured q8_0 product beside growing f16 and ternary products", flush=True)
    n, k = 512, 1024
    codes, sbits = synth.q8_0_matrix(synth.seed_for(3, 1), n, k)
    q8 = hip.Dense.q8_0(n, k, synth.q8_0_blocks(codes, sbits))
    half = hip.Dense.f16(synth.f16_bits(synth.activations(61, 96, 4096) * 0.02).reshape(96, 4096))
    tern = hip.Dense.ternary(*synth.ternary_matrix(synth.seed_for(3, 2), 128, 4096))
    D = Device()
    try:
        x8, x = synth.activations(62, 8, k), synth.activations(63, 3000, 4096)
        want = O.Int8(codes, sbits.view(np.float16).astype(np.float32), 32, True)(x8)
        dx8, dx = D.upload(x8), D.upload(x)
        y8, yf, yt = D.empty(8 * n * 4), D.empty(3000 * 96 * 4), D.empty(3000 * 128 * 4)
        forward(q8, dx8, 8, y8)  # the scratch is there before the capture
        D.download(y8, (8, n))
        graph = Graph(lambda s: forward(q8, dx8, 8, y8, s))
        for rows in (40, 600, 3000):  # growth in steps, past the scratch's size
            forward(half, dx, rows, yf)
            forward(tern, dx, rows, yt)
            D.download(yf, (rows, 96))
            graph.replay()
            assert bits_equal(D.download(y8, (8, n)), want), rows
        graph.free()
    finally:
        D.free()


@pytest.mark.parametrize("kind", ["f16", "ternary"])
def test_captured_many_rows(gpu, kind):
    print(f"case captured {kind} rows", flush=True)
    n, k, m = 128, 512, 43
    x = synth.activations(64, m, k)
    if kind == "f16":
        bits = synth.f16_bits(synth.activations(65, n, k) * 0.02).reshape(n, k)
        layer, want = hip.Dense.f16(bits), O.matmul_f32(x, bits.view(np.float16).astype(np.float32))
    else:
        codes, scales = synth.ternary_matrix(synth.seed_for(3, 3), n, k)
        layer, want = hip.Dense.ternary(codes, scales), O.Ternary(codes, scales)(x)
    D = Device()
    try:
        dx, y = D.upload(x), D.empty(m * n * 4)
        forward(layer, dx, 8, y)  # the 8-row launches' scratch
        D.download(y, (m, n))
        graph = Graph(lambda s: forward(layer, dx, m, y, s))
        for _ in range(3):
            forward(layer, dx, 5, y)
            D.download(y, (m, n))
            graph.replay()
            assert bits_equal(D.download(y, (m, n)), want)
        graph.free()
    finally:
        D.free()
