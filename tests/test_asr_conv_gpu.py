"""Convolutions quantized straight from their input maps (Q8_0 convolutions of
an ASR encoder) against the oracle, bit for bit: odd and even map sizes, a last
chunk shorter than the rest, channels whose columns end inside a 128-byte
product stage, and so few rows that the columns are written out instead."""

import numpy as np
import pytest

from tests.test_asr_encoder_gpu import make
from trit_amd import synth

pytestmark = pytest.mark.gpu

BASE = dict(d=64, layers=1, heads=1, ffn=128, window_chunks=2, out=64, max_positions=40)


@pytest.mark.parametrize("mels,channels,chunk,frames", [(16, 32, 32, 70), (15, 32, 29, 100), (33, 96, 31, 64),
                                                        (16, 128, 8, 8), (40, 160, 50, 333)])
def test_conv_from_maps(gpu, mels, channels, chunk, frames):
    print(f"case asr convolutions mels={mels} channels={channels} chunk={chunk} frames={frames}", flush=True)
    enc, ref = make(dict(BASE, mels=mels, channels=channels, chunk=chunk), 180 + frames, False)
    mel = synth.activations(181 + frames, frames, mels)
    got, want = enc.encode(mel, frames), ref.encode(mel, frames)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), float(np.max(np.abs(got - want)))
