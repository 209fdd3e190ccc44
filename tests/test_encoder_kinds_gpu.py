"""Audio encoders of one layer, against the oracle, bit for bit: the layer norm's
kernels at the edges of their row lengths (registers for 16, 24, 32, 40 and 64
values a lane, rows of fewer than 32 values or more than 2079, tails past the
last whole 32), and the weight kinds whose products add the GELU and the residual
in their store: ternary, int8 and f32 layers of few and of many rows, int8
convolutions quantized from their maps."""

import numpy as np
import pytest

from oracle import oracle as O
from trit_amd import hip, synth

pytestmark = pytest.mark.gpu


class Layers:
    """Device layers and the oracle's products for the same weights."""

    def __init__(self, seed):
        self.seed, self.t = seed, 0

    def next(self):
        self.t += 1
        return synth.seed_for(self.seed, self.t)

    def vec(self, n, base=0.0, spread=0.2):
        return (base + spread * (2 * synth.uniform(self.next(), n) - 1)).astype(np.float32)

    def make(self, kind, n, k):
        isa = O.isa_best()
        if kind == "f32":
            w, bias = (synth.normal(self.next(), (n, k)) / np.sqrt(k)).astype(np.float32), self.vec(n)
            return hip.Dense.f32(w, bias), lambda x: (O.matmul_f32(x, w, isa) + bias).astype(np.float32)
        if kind == "ternary":
            codes, scales = synth.ternary_matrix(self.next(), n, k)
            lay = O.Ternary(codes, scales)
            return hip.Dense.ternary(codes, scales), lambda x: lay(np.ascontiguousarray(x, np.float32))
        codes, bias = synth.ints(self.next(), (n, k), -127, 127).astype(np.int8), self.vec(n)
        scales = ((0.5 + synth.uniform(self.next(), (n, k // 128))) / (73 * np.sqrt(k))).astype(np.float32)
        lay = O.Int8(codes, scales, 128, False, isa)
        return hip.Dense.int8(codes, scales, bias), lambda x: (lay(np.ascontiguousarray(x, np.float32)) + bias).astype(
            np.float32)


def same_bits(a, b):
    return np.array_equal(np.asarray(a, np.float32).view(np.uint32), np.asarray(b, np.float32).view(np.uint32))


def check_encoder(kind, d, heads, ffn, mels, positions):
    print(f"case encoder {kind} d={d} heads={heads} ffn={ffn} positions={positions}", flush=True)
    L = Layers(190 + d)
    cfg = dict(d=d, layers=1, heads=heads, ffn=ffn, mels=mels, positions=positions)
    shapes = [(d, 3 * mels), (d, 3 * d), (3 * d, d), (d, d), (ffn, d), (d, ffn)]
    made = [L.make(kind, n, k) for n, k in shapes]
    norms = [v for _ in range(2) for v in (L.vec(d, 1.0), L.vec(d))] + [L.vec(d, 1.0), L.vec(d)]
    pos = L.vec(positions * d, 0.0, 0.5).reshape(positions, d)
    enc = hip.Encoder(cfg, made[0][0], made[1][0], pos, [m[0] for m in made[2:]], norms)
    ref = O.Encoder(cfg, [m[1] for m in made], pos, norms)
    mel = synth.activations(191, 2 * positions, mels)
    want = ref.encode(mel)
    assert same_bits(enc.encode(mel), want)
    assert same_bits(enc.encode(mel), want)  # the second call's buffers are the first's


@pytest.mark.parametrize("d,heads", [(24, 1), (32, 1), (40, 1), (536, 67), (544, 17), (792, 9), (800, 10), (1048, 131),
                                     (1056, 33), (1304, 163), (1312, 41), (2072, 37), (2080, 65)])
def test_layer_norm_lengths(gpu, d, heads):
    check_encoder("f32", d, heads, 32, 8, 7)


@pytest.mark.parametrize("kind", ["ternary", "int8", "f32"])
@pytest.mark.parametrize("positions", [4, 20, 70])
def test_kinds(gpu, kind, positions):
    check_encoder(kind, 128, 2, 256, 128, positions)


@pytest.mark.parametrize("frames", [8, 70, 200])
def test_int8_convolutions(gpu, frames):
    print(f"case asr int8 convolutions frames={frames}", flush=True)
    L = Layers(195)
    cfg = dict(d=128, layers=1, heads=2, ffn=256, mels=16, channels=128, chunk=40, window_chunks=2, out=128,
               max_positions=40)
    shapes = [(128, 9), (128, 1152), (128, 1152), (128, 256), (384, 128), (128, 128), (256, 128), (128, 256), (128, 128),
              (128, 128)]
    made = [L.make("f32" if i == 0 else "int8", n, k) for i, (n, k) in enumerate(shapes)]
    norms = [v for _ in range(2) for v in (L.vec(128, 1.0), L.vec(128))] + [L.vec(128, 1.0), L.vec(128)]
    dev, ref = [m[0] for m in made], [m[1] for m in made]
    enc = hip.AsrEncoder(cfg, dev[:3], dev[3], dev[4:8], norms, dev[8], dev[9])
    mel = synth.activations(196, frames, 16)
    assert same_bits(enc.encode(mel, frames), O.AsrEncoder(cfg, ref, norms, enc.positions()).encode(mel, frames))
